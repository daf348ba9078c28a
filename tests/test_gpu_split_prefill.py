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


# Grids of 8 head groups and multiples (a list of pieces an XCD), and more pieces than 256 compute units (the later
# rounds deal in the reverse order): dim, heads, kv, n_q, n_k, q_pos0, block, dtype, out, head groups, pieces
LISTS = [
    (128, 32, 8, 70, 1500, 1430, U32, O.BF16, "same", 8, 64),
    (128, 64, 16, 33, 1200, 1167, U32, O.F16, "f32", 16, 48),     # two head groups an XCD
    (128, 32, 8, 200, 2100, 1700, 1800, O.BF16, "f32", 8, 152),     # prefix-causal rows: pieces of several lengths
    (64, 16, 16, 2048, 2048, 0, U32, O.BF16, "same", 16, 192),    # causal rows from 0, items of one piece and of two
    (64, 32, 8, 700, 4000, 3300, U32, O.F16, "same", 8, 504),     # two rounds of the XCDs' lists
    (64, 48, 12, 500, 6000, 5500, U32, O.BF16, "f32", 12, 480),   # two rounds of one list
]


def pieces_of(args, need):
    """The pieces of a call whose workspace is `need` bytes (o and log-sums of that many pieces)."""
    dim, heads, n_q, n_k = (args[k] for k in ("dim", "heads", "n_q", "n_k"))
    group = heads // args["kv_heads"]
    hq = 4 if group % 4 == 0 else 2 if group % 2 == 0 else 1
    rows, cuts = 256 // hq, need // (n_q * heads * (dim + 1) * 4)
    last = [args["q_pos0"] + min(r + rows, n_q) - 1 for r in range(0, n_q, rows)]
    tiles = [-(-(n_k if p >= args["block"] else min(n_k, p + 1)) // 64) for p in last]
    per = -(-tiles[-1] // cuts)
    return heads // hq, heads // hq * sum(-(-t // per) for t in tiles)


@pytest.mark.parametrize("case", LISTS, ids=lambda c: "d{}h{}q{}k{}b{}".format(c[0], c[1], c[3], c[4], c[6]))
def test_split_prefill_lists(case):
    """Every head against the unsplit call (both are within the tolerance of the exact result), and the first and the
    last kv head's against the oracle."""
    host, args, o, lse = inputs(case[:9])
    dt, kv, heads = case[7], case[2], case[1]
    q, k, v = (G.to_dev(b, dt) for b in host)
    need = M.attn_fwd_workspace(**args)
    assert need > 0, "the call is not split"
    groups, pieces = pieces_of(args, need)
    assert (groups, pieces) == case[9:]
    print(f"split lists {case}: {pieces} pieces", flush=True)
    M.attn_fwd(q, k, v, o, lse=lse, workspace=torch.empty(need, dtype=torch.uint8, device="cuda"), **args)
    o1, lse1 = torch.full_like(o, float("nan")), torch.full_like(lse, float("nan"))
    M.attn_fwd(q, k, v, o1, lse=lse1, workspace=None, **args)
    torch.cuda.synchronize()
    err = (o.float() - o1.float()).abs()
    assert bool((err <= 2 * (G.ATOL + G.RTOL * o1.float().abs())).all())
    assert bool(((lse - lse1).abs() <= 2 * G.LSE_TOL).all())
    g = heads // kv
    for kh in (0, kv - 1):
        hs = slice(kh * g, (kh + 1) * g)
        sub = dict(args, heads=g, kv_heads=1)
        want_o, want_l = O.attn_dense(*(np.ascontiguousarray(x) for x in (host[0][hs], host[1][kh:kh + 1], host[2][kh:kh + 1])),
                                      dtype=dt, **sub)
        cols = slice(kh * g * case[0], (kh + 1) * g * case[0])
        G.assert_attn_close(G.to_host(o[:, cols]), want_o, f"kv head {kh}")
        G.assert_lse_close(lse[hs].cpu().numpy(), want_l, f"kv head {kh}")


@pytest.mark.parametrize("case", [CASES[0], CASES[3], CASES[6]], ids=lambda c: "d{}q{}k{}".format(c[0], c[3], c[4]))
def test_split_prefill_wide_rows_and_short_workspaces(case):
    """Output rows wider than the heads (the other columns stay); a workspace one byte short or off 16 bytes: the bits of
    the unsplit call, nothing written past what was given."""
    host, args, o, lse = inputs(case)
    q, k, v = (G.to_dev(b, case[7]) for b in host)
    need, wid = M.attn_fwd_workspace(**args), o.shape[1]
    buf = torch.zeros(need + 16, dtype=torch.uint8, device="cuda")
    M.attn_fwd(q, k, v, o, lse=lse, workspace=buf[:need], **args)
    wide = torch.full((args["n_q"], wid + 36), 7.0, dtype=o.dtype, device="cuda")
    M.attn_fwd(q, k, v, wide, workspace=buf[:need], width=wid + 36, **args)
    torch.cuda.synchronize()
    assert torch.equal(wide[:, :wid], o) and bool((wide[:, wid:] == 7.0).all())
    assert int(buf[need:].sum()) == 0
    buf.zero_()
    unsplit = torch.empty_like(o)
    M.attn_fwd(q, k, v, unsplit, workspace=None, **args)
    for ws in (buf[:need - 1], buf[8:], buf[:256]):
        got = torch.full_like(o, float("nan"))
        M.attn_fwd(q, k, v, got, workspace=ws, **args)
        torch.cuda.synchronize()
        assert torch.equal(got, unsplit)
    assert int(buf.sum()) == 0


@pytest.mark.parametrize("dim,heads,kv,n_q,n_k", [(128, 32, 8, 70, 1500), (64, 4, 2, 130, 1300)], ids=["d128", "d64"])
def test_split_prefill_from_rows(dim, heads, kv, n_q, n_k):
    """mako_attn_fwd_rows splits as mako_attn_fwd does: the bits of the tiles' producers and that call."""
    rng = np.random.default_rng(n_k)
    xq, xk, xv = (torch.from_numpy(rng.standard_normal((r, h * dim)).astype(np.float32)).to("cuda")
                  for r, h in ((n_q, heads), (n_k, kv), (n_k, kv)))
    call = dict(n_q=n_q, n_k=n_k, heads=heads, kv_heads=kv, q_pos0=n_k - n_q, block=U32)
    tiles = []
    for x, r, h in ((xq, n_q, heads), (xk, n_k, kv), (xv, n_k, kv)):
        y = torch.empty((h, r, dim), dtype=torch.bfloat16, device="cuda")
        M.heads(x, y, rows=r, ld=h * dim, col0=0, stride=dim, dim=dim, heads=h, n_pad=r)
        tiles.append(y)
    args = dict(call, q_pad=n_q, k_pad=n_k, dim=dim)
    assert M.attn_fwd_workspace(**args) > 0, "the call is not split"
    want = torch.empty((n_q, heads * dim), dtype=torch.bfloat16, device="cuda")
    M.attn_fwd(*tiles, want, **args)
    h = lambda n, r: dict(rows=r, ld=n * dim, col0=0, stride=dim, dim=dim, heads=n)  # noqa: E731
    need = M.attn_fwd_rows_workspace(dim=dim, **call)
    for ws in (M.LIBRARY, torch.empty(need, dtype=torch.uint8, device="cuda")):
        got = torch.full_like(want, float("nan"))
        M.attn_fwd_rows(xq, xk, xv, got, h(heads, n_q), h(kv, n_k), h(kv, n_k), in_dtype=M.BF16, workspace=ws, **call)
        torch.cuda.synchronize()
        assert torch.equal(got, want)
