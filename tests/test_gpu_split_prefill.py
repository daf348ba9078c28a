"""Prefill calls whose keys are split over workgroups (flash_fwd_r64's split grid and merge_pieces): a few blocks of
query rows over a long cache, causal rows whose last block runs longest, bidirectional rows, prefix-causal rows, at
heads of 128 and 64. Each is checked against the CPU oracle, and against the same call with no workspace, which runs
unsplit; under stream capture the call runs unsplit too, whether or not the library holds a workspace for the stream."""
import numpy as np
import pytest

import oracle as O

torch = pytest.importorskip("torch")
pytestmark = pytest.mark.gpu

import gpu_util as G  # noqa: E402
import mako_attn as M  # noqa: E402

U32 = 0xFFFFFFFF
CASES = [
    # dim, heads, kv, n_q, n_k, q_pos0, block, dtype, out
    (128, 8, 2, 70, 1500, 1430, U32, O.BF16, "same"),    # the diagonal crosses the last piece's first tiles
    (128, 8, 2, 17, 3001, 2984, U32, O.F16, "f32"),      # one part block of rows, many pieces
    (128, 4, 4, 300, 1700, 1400, U32, O.F16, "same"),    # 256 rows an item: the diagonal spans five tiles
    (128, 4, 2, 1600, 1600, 0, U32, O.BF16, "f32"),      # items of one piece beside items of several
    (128, 2, 1, 65, 1999, 0, 0, O.BF16, "same"),         # bidirectional
    (128, 8, 2, 200, 2100, 700, 800, O.F16, "f32"),      # prefix-causal: rows from 800 on see every key
    (64, 4, 4, 100, 1300, 1200, U32, O.BF16, "same"),
    (64, 2, 2, 513, 1537, 0, 0, O.F16, "f32"),
]


def inputs(case):
    dim, heads, kv, n_q, n_k, q_pos0, block, dt, out = case
    rng = np.random.default_rng(n_q + n_k)
    q_pad, k_pad = n_q + 3, n_k + 5
    host = [G.randn_bits(rng, (h, n, dim), dt) for h, n in ((heads, q_pad), (kv, k_pad), (kv, k_pad))]
    args = dict(n_q=n_q, q_pad=q_pad, n_k=n_k, k_pad=k_pad, heads=heads, kv_heads=kv, q_pos0=q_pos0, block=block,
                dim=dim)
    o = torch.full((n_q, heads * dim), float("nan"), dtype=torch.float32 if out == "f32" else G.TORCH[dt],
                   device="cuda")
    return host, args, o, torch.full((heads, n_q), float("nan"), dtype=torch.float32, device="cuda")


@pytest.mark.parametrize("case", CASES, ids=lambda c: "d{}q{}k{}b{}".format(c[0], c[3], c[4], c[6]))
def test_split_prefill(case):
    host, args, o, lse = inputs(case)
    q, k, v = (G.to_dev(b, case[7]) for b in host)
    need = M.attn_fwd_workspace(**args)
    assert need > 0, "the call is not split"
    print(f"split prefill {case}: {need} bytes", flush=True)
    M.attn_fwd(q, k, v, o, lse=lse, workspace=torch.empty(need, dtype=torch.uint8, device="cuda"), **args)
    o1, lse1 = torch.full_like(o, float("nan")), torch.full_like(lse, float("nan"))
    M.attn_fwd(q, k, v, o1, lse=lse1, workspace=None, **args)
    o2 = torch.full_like(o, float("nan"))
    M.attn_fwd(q, k, v, o2, workspace=M.LIBRARY, **args)
    torch.cuda.synchronize()
    want_o, want_l = O.attn_dense(*host, dtype=case[7], **args)
    for what, a, b in (("split", o, lse), ("unsplit", o1, lse1)):
        G.assert_attn_close(G.to_host(a), want_o, what)
        G.assert_rows_l2(G.to_host(a), want_o, what, case[0])
        G.assert_lse_close(b.cpu().numpy(), want_l, what)
    assert torch.equal(o, o2)


def test_split_prefill_under_capture():
    host, args, o, lse = inputs(CASES[0])
    q, k, v = (G.to_dev(b, CASES[0][7]) for b in host)
    want = torch.full_like(o, float("nan"))
    M.attn_fwd(q, k, v, want, workspace=None, **args)
    s = torch.cuda.Stream()
    s.wait_stream(torch.cuda.current_stream())
    M.attn_fwd(q, k, v, o, stream=s.cuda_stream, **args)  # the library holds the workspace; the graph must not keep it
    s.synchronize()
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph, stream=s):
        M.attn_fwd(q, k, v, o, lse=lse, stream=s.cuda_stream, **args)
    for _ in range(3):
        o.fill_(float("nan"))
        graph.replay()
        torch.cuda.synchronize()
        assert torch.equal(o, want)


NONFINITE = [
    # tensor, its first row changed, value; the calls below cut 1500 keys into pieces of at least six 64-key tiles
    ("k", 5, "nan"), ("k", 1001, "nan"), ("k", 5, "inf"), ("k", 1001, "inf"), ("k", 1001, "-inf"),
    ("v", 5, "nan"), ("v", 1001, "inf"), ("q", 0, "nan"), ("q", 69, "inf"),
]


@pytest.mark.parametrize("what,row,value", NONFINITE, ids=lambda x: str(x))
@pytest.mark.parametrize("dim,dt,out", [(128, O.BF16, "same"), (64, O.F16, "f32")], ids=["d128", "d64"])
def test_split_prefill_carries_non_finite_values(dim, dt, out, what, row, value):
    """One value that is not finite, in the first piece's keys, a later one's or a query: the split call's outputs and
    log-sums are not finite where the unsplit call's are not, and agree elsewhere (each side is within the tolerance of
    the exact result, so they differ by twice it at most)."""
    host, args, o, lse = inputs((dim, 8, 2, 70, 1500, 1430, U32, dt, out))
    q, k, v = (G.to_dev(b, dt) for b in host)
    {"q": q, "k": k, "v": v}[what][:, row, 3] = float(value)
    need = M.attn_fwd_workspace(**args)
    assert need > 0, "the call is not split"
    M.attn_fwd(q, k, v, o, lse=lse, workspace=torch.empty(need, dtype=torch.uint8, device="cuda"), **args)
    o1, lse1 = torch.full_like(o, float("nan")), torch.full_like(lse, float("nan"))
    M.attn_fwd(q, k, v, o1, lse=lse1, workspace=None, **args)
    torch.cuda.synchronize()
    for got, want in ((o, o1), (lse, lse1)):
        assert torch.equal(torch.isnan(got), torch.isnan(want))
        inf = torch.isinf(want)
        assert torch.equal(torch.isinf(got), inf) and torch.equal(got[inf], want[inf])
        ok = torch.isfinite(want)
        err = (got[ok].float() - want[ok].float()).abs()
        assert bool((err <= 2 * (G.ATOL + G.RTOL * want[ok].float().abs())).all())
    assert bool((~torch.isfinite(o1)).any())
