"""The output projection after attention (mako_proj_bf16: Runtime::proj with BF16 weights) on the GPU against the
CPU oracle: bf16 activations as the attention writes them, f32 activations rounded in the GEMM's loads, the bf16
split, tiles cut by t and n, strided x and y rows, and the Qwen3-8B o_proj shape (4096 tokens, 4096 -> 4096); and
the handoff itself: mako_attn_fwd writing bf16 rows [n_q][heads * D] that mako_proj_bf16 reads with no conversion.

Tolerance: bf16 times bf16 is exact in f32, so the only error is the f32 summation over k; every element must be
within 2 k 2^-24 sum|terms| of the oracle's double-precision sum (sum|terms| from the oracle on |x| and |w|; twice
that with the split's second product). Columns past n keep a sentinel.
"""
import numpy as np
import pytest

import oracle as O

torch = pytest.importorskip("torch")
pytestmark = pytest.mark.gpu

import gpu_util as G  # noqa: E402
import mako_attn as M  # noqa: E402

U = 2.0 ** -24
SENTINEL = 1234.5


def abs_bits(b):
    return np.asarray(b, np.uint16) & np.uint16(0x7FFF)


def run_proj(rng, t, k, n, x_dtype, split, ldx=0, ldy=0, scale=1.0, workspace=M.LIBRARY):
    ldx_, ldy_ = ldx or k, ldy or n
    w = O.to_bf16_bits(rng.standard_normal((n, k)) * 0.05)
    xf = (rng.standard_normal((t, ldx_)) * scale).astype(np.float32)
    x = xf if x_dtype == O.F32 else O.to_bf16_bits(xf)
    wd = G.to_dev(w, O.BF16)
    xd = torch.from_numpy(x).to("cuda") if x_dtype == O.F32 else G.to_dev(x, O.BF16)
    y = torch.full((t, ldy_), SENTINEL, dtype=torch.float32, device="cuda")
    print(f"proj t={t} k={k} n={n} x={'f32' if x_dtype == O.F32 else 'bf16'} split={split} ldx={ldx} ldy={ldy}",
          flush=True)
    M.proj_bf16(wd, xd, y, t=t, k=k, n=n, ldx=ldx, ldy=ldy, split=split, workspace=workspace)
    torch.cuda.synchronize()
    got = y.cpu().numpy()
    want = O.proj_bf16(x, w, t=t, k=k, n=n, ldx=ldx, ldy=ldy, x_dtype=x_dtype, split=split,
                       y=np.full((t, ldy_), SENTINEL))
    xa = np.abs(x) if x_dtype == O.F32 else abs_bits(x)
    mag = O.proj_bf16(xa, abs_bits(w), t=t, k=k, n=n, ldx=ldx, ldy=ldy, x_dtype=x_dtype, split=split)
    return got, want, mag


def assert_sum_close(got, want, bound, what):
    err = np.abs(np.asarray(got, np.float64) - want)
    bad = err > bound + 1e-30
    assert not bad.any(), (f"{what}: {int(bad.sum())} of {bad.size} elements beyond the f32 summation bound, worst "
                           f"{err.max():.3e} at {np.unravel_index(np.argmax(err - bound), err.shape)}")


CASES = [
    # t, k, n, x dtype, split, ldx, ldy
    (300, 256, 320, O.BF16, 0, 0, 0),       # part tiles in both dimensions
    (256, 4096, 256, O.F32, 0, 0, 0),       # a long k
    (77, 128, 96, O.F32, 1, 0, 0),          # the split, one part tile
    (513, 1024, 1000, O.BF16, 0, 1032, 1010),  # strided x and y rows
    (1, 64, 1, O.F32, 0, 0, 0),
    (600, 512, 700, O.F32, 1, 520, 0),      # the split over several 128-row tiles
    (1100, 192, 2048, O.F32, 0, 0, 0),      # more tiles than the 8 XCDs take evenly
    # bf16 activations of one, two and three K stages, part tiles
    (200, 64, 130, O.BF16, 0, 0, 0),
    (129, 128, 200, O.BF16, 0, 136, 0),
    (70, 192, 257, O.BF16, 0, 0, 260),
]


@pytest.mark.parametrize("case", CASES, ids=lambda c: "t{}k{}n{}{}{}".format(
    *c[:3], "f32" if c[3] == O.F32 else "bf16", "s" if c[4] else ""))
def test_proj(case):
    t, k, n, xd, split, ldx, ldy = case
    rng = np.random.default_rng(t + k + n)
    got, want, mag = run_proj(rng, t, k, n, xd, split, ldx, ldy, scale=3.0)
    nn = n
    assert_sum_close(got[:, :nn], want[:, :nn], (4 if split else 2) * k * U * mag[:, :nn], "proj")
    assert (got[:, nn:] == SENTINEL).all(), "a column past n was written"


def test_qwen3_8b_o_proj():
    """Qwen3-8B's o_proj after a 4096-token prefill (src/models/qwen_text.cpp:312): 4096 x 4096 bf16 weights over
    bf16 attention rows; 64 sampled rows against the oracle."""
    rng = np.random.default_rng(8)
    t = k = n = 4096
    w = O.to_bf16_bits(rng.standard_normal((n, k)) * 0.02)
    x = O.to_bf16_bits(rng.standard_normal((t, k)))
    y = torch.empty((t, n), dtype=torch.float32, device="cuda")
    print("qwen3-8b o_proj", flush=True)
    M.proj_bf16(G.to_dev(w, O.BF16), G.to_dev(x, O.BF16), y, t=t, k=k, n=n)
    torch.cuda.synchronize()
    rows = np.sort(rng.choice(t, 64, replace=False))
    got = y.cpu().numpy()[rows]
    want = O.proj_bf16(x[rows], w, t=64, k=k, n=n, x_dtype=O.BF16)
    mag = O.proj_bf16(abs_bits(x[rows]), abs_bits(w), t=64, k=k, n=n, x_dtype=O.BF16)
    assert_sum_close(got, want, 2 * k * U * mag, "o_proj")


def test_attention_rows_feed_the_projection():
    """mako_attn_fwd with a bf16 output writes [n_q][heads * D] rows; mako_proj_bf16 reads them as x directly. The
    result equals the oracle's projection of exactly those bf16 rows (the attention itself is checked elsewhere)."""
    rng = np.random.default_rng(12)
    S, H, KV, D = 320, 8, 2, 128
    q = G.randn_bits(rng, (H, S, D), O.BF16)
    kk = G.randn_bits(rng, (KV, S, D), O.BF16)
    v = G.randn_bits(rng, (KV, S, D), O.BF16)
    o = torch.empty((S, H * D), dtype=torch.bfloat16, device="cuda")
    M.attn_fwd(G.to_dev(q, O.BF16), G.to_dev(kk, O.BF16), G.to_dev(v, O.BF16), o, n_q=S, q_pad=S, n_k=S, k_pad=S,
               heads=H, kv_heads=KV, q_pos0=0, block=M.U32_MAX, dim=D)
    n = 512
    w = O.to_bf16_bits(rng.standard_normal((n, H * D)) * 0.05)
    y = torch.empty((S, n), dtype=torch.float32, device="cuda")
    M.proj_bf16(G.to_dev(w, O.BF16), o, y, t=S, k=H * D, n=n)
    torch.cuda.synchronize()
    xb = o.view(torch.int16).cpu().numpy().view(np.uint16)
    want = O.proj_bf16(xb, w, t=S, k=H * D, n=n, x_dtype=O.BF16)
    mag = O.proj_bf16(abs_bits(xb), abs_bits(w), t=S, k=H * D, n=n, x_dtype=O.BF16)
    assert_sum_close(y.cpu().numpy(), want, 2 * H * D * U * mag, "attention -> proj")


@pytest.mark.parametrize("t", [1, 2, 15, 16, 17, 32, 33, 63, 64])
@pytest.mark.parametrize("k,n,ldx,ldy", [(64, 1, 0, 0), (576, 49, 584, 60), (4160, 130, 0, 0)])
@pytest.mark.parametrize("xd,split", [(O.BF16, 0), (O.F32, 0), (O.F32, 1)], ids=["bf16", "f32", "split"])
def test_few_rows(t, k, n, ldx, ldy, xd, split):
    """proj_few: blocks of 16 rows of x (1, 2 and 4 of them, the last one partial), one K chunk, a few more than the
    waves take together, many; part blocks of columns."""
    got, want, mag = run_proj(np.random.default_rng(t + k), t, k, n, xd, split, ldx, ldy)
    assert_sum_close(got[:, :n], want[:, :n], (4 if split else 2) * k * U * mag[:, :n], "proj")
    assert (got[:, n:] == SENTINEL).all(), "a column past n was written"


# Calls by the kernel that takes their bf16 rows (f32 rows after round_rows, but for the next two) on 256 compute units,
# which tests/test_host_paths.py checks: t, k, n, ldx, ldy. Part tiles in both dimensions; K stages (64 values) fewer than the
# ring has, as many and more; for proj_dma one, two and three (its prologue's and tail's waits), and a strided x.
TILES = {
    "proj_ring<64, 64, 8>": [(100, 64, 130, 0, 0), (65, 576, 257, 584, 260)],
    "proj_ring<64, 128, 6>": [(300, 192, 4100, 0, 0), (290, 448, 4090, 456, 0)],
    "proj_ring<128, 128, 4>": [(850, 128, 4100, 0, 0), (1000, 320, 4090, 328, 4092)],
    "proj_ring<128, 256, 3>": [(900, 128, 4100, 0, 0), (2000, 64, 4090, 0, 0), (1990, 320, 4090, 328, 0),
                               (1000, 320, 4100, 328, 0)],
    "proj_dma": [(1990, 256, 4100, 0, 0), (1990, 64, 4100, 0, 0), (1990, 128, 4100, 136, 0), (2500, 192, 4090, 0, 4092),
                 (1990, 1088, 4100, 1096, 0)],
}
# those whose f32 rows proj_tiles takes without the split (K too short to pay for the rounding)
SHORT_K = [(1990, 256, 4100, 0, 0), (1990, 64, 4100, 0, 0), (1990, 128, 4100, 136, 0), (2500, 192, 4090, 0, 4092)]

# those that proj_tiles takes with the split
SPLIT_TILES = [(900, 128, 4100, 0, 0), (2000, 64, 4090, 0, 0), (1990, 320, 4090, 328, 0)]


# A few rows by kernel: x dtype, split, t, k, n. proj_few up to a round or two of its n / 16 workgroups over 256 compute
# units, the tiles for wider weights.
FEW = {
    "proj_few<1, false, false>": [(O.BF16, 0, 1, 4096, 4096), (O.BF16, 0, 16, 14336, 4096), (O.BF16, 0, 1, 1024, 1024)],
    "proj_few<2, false, false>": [(O.BF16, 0, 32, 4096, 4090)],
    "proj_few<1, true, false>": [(O.F32, 0, 1, 4096, 8192)],
    "proj_few<1, true, true>": [(O.F32, 1, 16, 4096, 4096), (O.F32, 1, 1, 4096, 12290)],
    "proj_few<4, true, true>": [(O.F32, 1, 48, 4096, 4096)],
    "proj_ring<64, 64, 8>": [(O.BF16, 0, 1, 1024, 16370), (O.BF16, 0, 32, 576, 16384), (O.F32, 0, 16, 1024, 16380),
                             (O.F32, 1, 33, 4096, 8190)],
    "proj_ring<64, 128, 6>": [(O.BF16, 0, 7, 256, 28670), (O.F32, 0, 24, 256, 28672), (O.F32, 1, 17, 256, 28674)],
    "proj_tiles<128, true, true>": [(O.F32, 1, 33, 128, 65536), (O.F32, 1, 65, 256, 40962)],
}


@pytest.mark.parametrize("case", [c for calls in FEW.values() for c in calls],
                         ids=lambda c: "{}{}t{}k{}n{}".format("f32" if c[0] == O.F32 else "bf16", "s" if c[1] else "", *c[2:]))
def test_few_rows_by_width(case):
    xd, split, t, k, n = case
    got, want, mag = run_proj(np.random.default_rng(n), t, k, n, xd, split)
    assert_sum_close(got, want, (4 if split else 2) * k * U * mag, "proj")


@pytest.mark.parametrize("t,k,n,ldx,ldy", [c for calls in TILES.values() for c in calls])
@pytest.mark.parametrize("xd,split", [(O.BF16, 0), (O.F32, 0), (O.F32, 1)], ids=["bf16", "f32", "split"])
def test_ring_tiles(t, k, n, ldx, ldy, xd, split):
    """The DMA kernels' tiles, and the rounding pass before them for f32 rows; 40 rows (the last one among them) against
    the oracle."""
    rng = np.random.default_rng(t + k)
    ld = ldx or k
    w = O.to_bf16_bits(rng.standard_normal((n, k)) * 0.05)
    xf = rng.standard_normal((t, ld)).astype(np.float32)
    x = xf if xd == O.F32 else O.to_bf16_bits(xf)
    y = torch.full((t, ldy or n), SENTINEL, dtype=torch.float32, device="cuda")
    print(f"proj ring t={t} k={k} n={n} xd={xd} split={split}", flush=True)
    M.proj_bf16(G.to_dev(w, O.BF16), torch.from_numpy(x).to("cuda") if xd == O.F32 else G.to_dev(x, O.BF16), y, t=t, k=k,
                n=n, ldx=ldx, ldy=ldy, split=split)
    torch.cuda.synchronize()
    rows = np.sort(np.append(rng.choice(t - 1, 39, replace=False), t - 1))
    got = y.cpu().numpy()
    assert (got[:, n:] == SENTINEL).all(), "a column past n was written"
    xr = np.ascontiguousarray(x[rows])
    want = O.proj_bf16(xr, w, t=40, k=k, n=n, ldx=ldx, x_dtype=xd, split=split)
    mag = O.proj_bf16(np.abs(xr) if xd == O.F32 else abs_bits(xr), abs_bits(w), t=40, k=k, n=n, ldx=ldx, x_dtype=xd,
                      split=split)
    assert_sum_close(got[rows][:, :n], want[:, :n], (4 if split else 2) * k * U * mag[:, :n], "proj")


# f32 rows of calls that are given no workspace, by kernel: t, k, n, split, ldx, ldy
NO_WORKSPACE = {
    "proj_few<4, true, true>": [(50, 192, 77, 1, 200, 80), (64, 192, 16, 1, 0, 0)],
    "proj_few<4, true, false>": [(33, 576, 49, 0, 584, 60)],
    "proj_tiles<128, true, true>": [(77, 128, 96, 1, 0, 0), (600, 512, 700, 1, 520, 0), (257, 64, 515, 1, 72, 520)],
    "proj_tiles<256, true, false>": [(256, 4096, 256, 0, 0, 0), (300, 320, 330, 0, 328, 340), (1100, 192, 2048, 0, 0, 0),
                                     (65, 64, 1, 0, 0, 0)],
}


@pytest.mark.parametrize("case", [c for calls in NO_WORKSPACE.values() for c in calls],
                         ids=lambda c: "t{}k{}n{}{}".format(*c[:3], "s" if c[3] else ""))
def test_f32_rows_without_a_workspace(case):
    """The kernels that round f32 rows as they load them."""
    t, k, n, split, ldx, ldy = case
    got, want, mag = run_proj(np.random.default_rng(t + k + n), t, k, n, O.F32, split, ldx, ldy, scale=3.0, workspace=None)
    assert_sum_close(got[:, :n], want[:, :n], (4 if split else 2) * k * U * mag[:, :n], "proj")
    assert (got[:, n:] == SENTINEL).all(), "a column past n was written"


@pytest.mark.parametrize("split", [0, 1])
def test_proj_workspace(split):
    """The bytes asked for: the library's own result, under capture too; one byte less or a start off 16 bytes: the call
    without a workspace; nothing written past what was given."""
    t, k, n = 300, 256, 320
    rng = np.random.default_rng(split)
    w = G.to_dev(O.to_bf16_bits(rng.standard_normal((n, k)) * 0.05), O.BF16)
    x = torch.from_numpy(rng.standard_normal((t, k)).astype(np.float32)).to("cuda")
    need = M.proj_bf16_workspace(t=t, k=k, n=n, x_dtype=M.F32, split=split)
    assert need == t * k * 2 * (2 if split else 1)
    buf = torch.zeros(need + 16, dtype=torch.uint8, device="cuda")

    def call(workspace, stream=None, y=None):
        y = torch.full((t, n), SENTINEL, dtype=torch.float32, device="cuda") if y is None else y
        M.proj_bf16(w, x, y, t=t, k=k, n=n, split=split, workspace=workspace, stream=stream)
        return y

    unrounded = call(None)
    for ws in (buf[:need - 1], buf[8:]):
        assert torch.equal(call(ws), unrounded)
    assert int(buf.sum()) == 0
    want = call(M.LIBRARY)
    assert torch.equal(call(buf[:need]), want) and int(buf[need:].sum()) == 0
    y = torch.empty_like(want)
    s = torch.cuda.Stream()
    s.wait_stream(torch.cuda.current_stream())
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph, stream=s):
        call(buf[:need], stream=s.cuda_stream, y=y)
    for _ in range(3):
        y.fill_(SENTINEL)
        graph.replay()
        torch.cuda.synchronize()
        assert torch.equal(y, want)


@pytest.mark.parametrize("t,split", [(60, 1), (300, 0), (300, 1)])
def test_f32_rows_under_capture(t, split):
    """A captured call on a stream the library holds no workspace for rounds in the tiles: each replay gives the bound."""
    k, n = 256, 320
    rng = np.random.default_rng(t)
    w = O.to_bf16_bits(rng.standard_normal((n, k)) * 0.05)
    x = rng.standard_normal((t, k)).astype(np.float32)
    wd, xd = G.to_dev(w, O.BF16), torch.from_numpy(x).to("cuda")
    y = torch.empty((t, n), dtype=torch.float32, device="cuda")
    s = torch.cuda.Stream()
    s.wait_stream(torch.cuda.current_stream())
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph, stream=s):
        M.proj_bf16(wd, xd, y, t=t, k=k, n=n, split=split, stream=s.cuda_stream)
    want = O.proj_bf16(x, w, t=t, k=k, n=n, x_dtype=O.F32, split=split)
    mag = O.proj_bf16(np.abs(x), abs_bits(w), t=t, k=k, n=n, x_dtype=O.F32, split=split)
    for _ in range(3):
        y.fill_(SENTINEL)
        graph.replay()
        torch.cuda.synchronize()
        assert_sum_close(y.cpu().numpy(), want, (4 if split else 2) * k * U * mag, "proj")
