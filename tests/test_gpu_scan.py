"""The gated delta rule (mako_kda_scan, the reference's kda_scan) on the GPU against the CPU oracle: the inputs the
linear-attention layers feed it (q and k L2-normalised per head, v normal, g a log-decay in [-0.5, 0], beta in
(0, 1)), a nonzero starting state, strided rows, the rollback snapshot (after the first token, the last, and at a
boundary of the kernel's 16-token batches), token counts one past and one short of a batch multiple, no tokens,
and the Qwen3.5 shape (32 heads of 128 over 4096 tokens, four heads checked).

Tolerance: the oracle runs in double; the kernel in f32 with a different summation order (8 values a lane, then a
16-lane tree) and the hardware exponential. Every output and state element within 2e-5 + 1e-4 |ref| (the f32
rounding of 128-term sums carried through the recurrence stays well inside it at these lengths).
"""
import numpy as np
import pytest

import oracle as O

torch = pytest.importorskip("torch")
pytestmark = pytest.mark.gpu

import mako_attn as M  # noqa: E402

ATOL, RTOL = 2e-5, 1e-4
D = 128


def inputs(rng, T, H, ld=None, scale_state=0.0):
    ld = ld or H * D
    unit = lambda x: x / np.linalg.norm(x, axis=-1, keepdims=True)

    def rows(x):
        out = np.zeros((T, ld), np.float32)
        out[:, :H * D] = x.reshape(T, H * D)
        return out

    q = rows(unit(rng.standard_normal((T, H, D))))
    k = rows(unit(rng.standard_normal((T, H, D))))
    v = rows(rng.standard_normal((T, H, D)))
    g = rows(rng.uniform(-0.5, 0.0, (T, H, D)))
    beta = rng.uniform(0.05, 0.95, (T, H)).astype(np.float32)
    state = (rng.standard_normal((H, D, D)) * scale_state).astype(np.float32)
    return q, k, v, g, beta, state


def dev(x):
    return torch.from_numpy(np.ascontiguousarray(x)).to("cuda")


def assert_close(got, want, what):
    err = np.abs(np.asarray(got, np.float64) - want)
    bad = err > ATOL + RTOL * np.abs(want)
    assert not bad.any(), (f"{what}: {int(bad.sum())} of {bad.size} beyond tolerance, worst {err.max():.3e} at "
                           f"{np.unravel_index(np.argmax(err), err.shape)} (ref {want.flat[np.argmax(err)]:.4e})")


def run(q, k, v, g, beta, state, *, T, H, ld=None, snap=0):
    ld = ld or H * D
    o = torch.full((max(T, 1), ld), 7.0, dtype=torch.float32, device="cuda")
    st = dev(state)
    snap_d = torch.zeros((H, D, D), dtype=torch.float32, device="cuda") if snap else None
    print(f"kda_scan T={T} H={H} ld={ld} snap={snap}", flush=True)
    M.kda_scan(dev(q), dev(k), dev(v), dev(g), dev(beta), st, o, tokens=T, heads=H, qkv_stride=ld, inner=ld,
               snap=snap, snap_state=snap_d)
    torch.cuda.synchronize()
    return o.cpu().numpy(), st.cpu().numpy(), (snap_d.cpu().numpy() if snap else None)


@pytest.mark.parametrize("T,H,ld,snap", [(200, 4, 0, 0), (37, 2, 320, 20), (1, 1, 0, 1), (16, 3, 0, 16),
                                         (17, 2, 0, 17), (33, 1, 0, 32), (47, 3, 400, 1), (31, 2, 0, 0)],
                         ids=["t200h4", "t37h2_strided_snap20", "t1", "t16h3_snap16", "t17h2_snap_last",
                              "t33h1_snap_batch_edge", "t47h3_strided_snap_first", "t31h2"])
def test_kda_scan(T, H, ld, snap):
    rng = np.random.default_rng(T * 7 + H)
    q, k, v, g, beta, state = inputs(rng, T, H, ld or None, scale_state=0.3)
    o, st, sn = run(q, k, v, g, beta, state, T=T, H=H, ld=ld or None, snap=snap)
    ldx = ld or H * D
    want_o, want_st, want_sn = O.kda_scan(q, k, v, g, beta, state.astype(np.float64), tokens=T, heads=H,
                                          qkv_stride=ldx, inner=ldx, snap=snap, o=np.full((T, ldx), 7.0))
    assert_close(o[:T], want_o, "o")
    assert_close(st, want_st, "state")
    if snap:
        assert_close(sn, want_sn, "snapshot")


def test_strong_decays_and_growth():
    """Batches whose decays leave the kernel's rescaling range run unscaled: a channel decaying by -4 a token for a
    whole batch (-64 over it), single tokens at -50, a channel growing by +3 a token (+48), and weak batches between
    (rescaled); the last batch partial."""
    rng = np.random.default_rng(77)
    T, H = 91, 2
    q, k, v, g, beta, state = inputs(rng, T, H, scale_state=0.3)
    g[16:32, 5] = -4.0                   # batch 1: a channel at -64 over the batch
    g[40, D + 7] = -50.0                 # batch 2: one token, one channel
    g[70, :D] = -50.0                    # batch 4: one token, every channel of head 0
    g[48:64, D + 9] = 3.0                # batch 3: growth, +48 over the batch
    o, st, _ = run(q, k, v, g, beta, state, T=T, H=H)
    want_o, want_st, _ = O.kda_scan(q, k, v, g, beta, state.astype(np.float64), tokens=T, heads=H)
    assert_close(o[:T], want_o, "o")
    assert_close(st, want_st, "state")


def test_no_tokens_leaves_the_state():
    rng = np.random.default_rng(3)
    q, k, v, g, beta, state = inputs(rng, 1, 2, scale_state=1.0)
    _, st, _ = run(q, k, v, g, beta, state, T=0, H=2)
    assert np.array_equal(st, state)


def test_qwen35_linear_attention_shape():
    """32 heads of 128 over 4096 tokens (the linear-attention layers of Qwen3.5's encoder,
    src/models/qwen_text.cpp:374-382: qkv_stride = inner = 32 * 128, state zeroed): four heads against the oracle."""
    rng = np.random.default_rng(35)
    T, H = 4096, 32
    q, k, v, g, beta, state = inputs(rng, T, H)
    o, st, _ = run(q, k, v, g, beta, np.zeros_like(state), T=T, H=H)
    for h in (0, 9, 22, 31):
        sl = slice(h * D, (h + 1) * D)
        want_o, want_st, _ = O.kda_scan(q[:, sl], k[:, sl], v[:, sl], g[:, sl], beta[:, h:h + 1], tokens=T, heads=1)
        assert_close(o[:, sl], want_o, f"o head {h}")
        assert_close(st[h], want_st[0], f"state head {h}")


@pytest.mark.parametrize("T,H,ld,snap", [(96, 2, 0, 0), (97, 1, 0, 97), (111, 2, 320, 1), (128, 3, 0, 16),
                                         (150, 2, 0, 33), (300, 1, 0, 299), (1000, 2, 400, 512)])
def test_chunks(T, H, ld, snap):
    """Runs long enough for the chunks of 16 tokens: whole and part last chunks, a snapshot that ends a chunk after the
    first token, at a chunk's edge, inside one and before the last token."""
    rng = np.random.default_rng(T * 3 + snap)
    q, k, v, g, beta, state = inputs(rng, T, H, ld or None, scale_state=0.3)
    o, st, sn = run(q, k, v, g, beta, state, T=T, H=H, ld=ld or None, snap=snap)
    ldx = ld or H * D
    want_o, want_st, want_sn = O.kda_scan(q, k, v, g, beta, state.astype(np.float64), tokens=T, heads=H,
                                          qkv_stride=ldx, inner=ldx, snap=snap, o=np.full((T, ldx), 7.0))
    assert_close(o[:T], want_o, "o")
    assert_close(st, want_st, "state")
    if snap:
        assert_close(sn, want_sn, "snapshot")


def test_chunks_strong_decays_and_growth():
    """test_strong_decays_and_growth's decays in a run that goes by chunks: factors of e^-64 and e^48 over a chunk, a
    channel and a head cleared by one token, a channel that grows and is cut back inside a chunk. An output is a sum of 128 terms of the state's size, each rounded
    by up to 2^-24 an operation, and the growth leaves states of 1e18 whose terms cancel in some outputs (the recurrence
    itself, token by token in f32, is off by 1e-3 of such an output): 128 2^-24 of the largest output of the head so
    far, which stands for the state's size, is added to the tolerance."""
    rng = np.random.default_rng(78)
    T, H = 187, 2
    q, k, v, g, beta, state = inputs(rng, T, H, scale_state=0.3)
    g[16:32, 5] = -4.0
    g[40, D + 7] = -50.0
    g[70, :D] = -50.0
    g[48:64, D + 9] = 3.0
    g[100:104, 11] = 6.0
    g[104:108, 11] = -6.0
    o, st, _ = run(q, k, v, g, beta, state, T=T, H=H)
    want_o, want_st, _ = O.kda_scan(q, k, v, g, beta, state.astype(np.float64), tokens=T, heads=H)
    for h in range(H):
        got, want = o[:T, h * D:(h + 1) * D], want_o[:, h * D:(h + 1) * D]
        size = np.maximum.accumulate(np.abs(want).max(1))[:, None]
        err = np.abs(got - want)
        assert np.all(err <= ATOL + RTOL * np.abs(want) + 128 * 2.0 ** -24 * size), f"head {h}: worst {err.max():.3e}"
    size = np.abs(want_st).max((1, 2), keepdims=True)
    assert np.all(np.abs(st - want_st) <= ATOL + RTOL * np.abs(want_st) + 128 * 2.0 ** -24 * size), "state"


def test_chunks_under_capture():
    """A captured call on a stream the library holds no workspace for runs token by token; each replay continues the
    state as the eager call does."""
    rng = np.random.default_rng(79)
    T, H = 130, 2
    host = inputs(rng, T, H, scale_state=0.3)
    q, k, v, g, beta, st = (dev(x) for x in host)
    state0, o = st.clone(), torch.empty_like(v)
    s = torch.cuda.Stream()
    s.wait_stream(torch.cuda.current_stream())
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph, stream=s):
        M.kda_scan(q, k, v, g, beta, st, o, tokens=T, heads=H, stream=s.cuda_stream)
    want_o, want_st, _ = O.kda_scan(*host[:5], host[5].astype(np.float64), tokens=T, heads=H)
    for _ in range(3):
        st.copy_(state0)
        o.zero_()
        graph.replay()
        torch.cuda.synchronize()
        assert_close(o.cpu().numpy(), want_o, "o")
        assert_close(st.cpu().numpy(), want_st, "state")


def both_routes(host, *, T, H, snap=0):
    """Outputs, state and snapshot by chunks, and token by token (a call without a workspace)."""
    out = []
    need = M.kda_scan_workspace(tokens=T, heads=H, snap=snap)
    assert need > 0, "the call does not go by chunks"
    for ws in (torch.empty(need, dtype=torch.uint8, device="cuda"), None):
        q, k, v, g, beta, st = (dev(x) for x in host)
        o = torch.full_like(v, 7.0)
        sn = torch.full_like(st, 7.0)
        print(f"kda_scan T={T} H={H} snap={snap} workspace={ws is not None}", flush=True)
        M.kda_scan(q, k, v, g, beta, st, o, tokens=T, heads=H, snap=snap, snap_state=sn, workspace=ws)
        torch.cuda.synchronize()
        out.append([x.cpu().numpy() for x in (o, st, sn)])
    return out


def assert_same_where_finite(by_chunks, by_token):
    """Not finite in the same places, and elsewhere within the tolerance of each other that each has of the oracle."""
    for what, got, want in zip(("o", "state", "snapshot"), by_chunks, by_token):
        fin = np.isfinite(want)
        assert np.array_equal(np.isfinite(got), fin), f"{what}: {int((np.isfinite(got) != fin).sum())} places differ"
        err = np.abs(got[fin].astype(np.float64) - want[fin])
        assert np.all(err <= 2 * (ATOL + RTOL * np.abs(want[fin]))), f"{what}: worst {err.max():.3e}"


@pytest.mark.parametrize("value", ["nan", "inf", "-inf"])
@pytest.mark.parametrize("what,t", [("q", 72), ("k", 72), ("v", 72), ("v", 0), ("v", 129), ("g", 72), ("beta", 72),
                                    ("state", 0)])
def test_a_value_that_is_not_finite_stays_causal(what, t, value):
    """One value of head 1 that is not finite, at a token inside a chunk, at the first or the last (in a part chunk):
    by chunks it reaches the outputs, the state and the snapshot that it reaches token by token, and the outputs before
    its token and the other heads are as without it."""
    T, H, snap = 130, 3, 75
    host = inputs(np.random.default_rng(80), T, H, scale_state=0.3)
    clean = [x.copy() for x in host]
    x = host[("q", "k", "v", "g", "beta", "state").index(what)]
    if what == "state":
        x[1, 4, 9] = float(value)  # column 4 of the state's transpose
    elif what == "beta":
        x[t, 1] = float(value)
    else:
        x[t, D + 9] = float(value)
    by_chunks, by_token = both_routes(host, T=T, H=H, snap=snap)
    assert_same_where_finite(by_chunks, by_token)
    want, _, _ = O.kda_scan(*clean[:5], clean[5].astype(np.float64), tokens=T, heads=H)
    assert_close(by_chunks[0][:t], want[:t], "o before the token")
    for h in (0, 2):
        assert_close(by_chunks[0][:, h * D:(h + 1) * D], want[:, h * D:(h + 1) * D], f"o of head {h}")


def test_growth_past_f32_over_a_state_of_zero():
    """A channel that no key and no state uses grows by e^12 a token: past f32 within a chunk (e^192), never by the
    recurrence, whose state there stays 0."""
    T, H = 130, 3
    host = inputs(np.random.default_rng(81), T, H)
    q, k, v, g, beta, state = host
    g[:, 9] = 12.0
    k[:, 9] = 0.0
    by_chunks, by_token = both_routes(host, T=T, H=H)
    assert_same_where_finite(by_chunks, by_token)
    want_o, want_st, _ = O.kda_scan(q, k, v, g, beta, np.zeros((H, D, D)), tokens=T, heads=H)
    assert_close(by_chunks[0], want_o, "o")
    assert_close(by_chunks[1], want_st, "state")


@pytest.mark.parametrize("snap", [1100, 1104, 1105, 1536])
def test_chunks_in_several_launches(snap):
    """64 heads' images of 16 tokens take 1.75 MiB, so 1600 tokens go in launches of 36 chunks, three of them: a snapshot
    in the second launch (inside a chunk, at its edge, one token past it) and in the third; and a value that is not
    finite in the second, which goes on token by token, with the third after it."""
    T, H = 1600, 64
    host = inputs(np.random.default_rng(snap), T, H, scale_state=0.3)
    q, k, v, g, beta, state = host
    image = 28 * 1024 * H
    assert M.kda_scan_workspace(tokens=T, heads=H, snap=snap) == (64 << 20) // image * image and (64 << 20) // image == 36
    o, st, sn = run(q, k, v, g, beta, state, T=T, H=H, snap=snap)
    for h in (0, 31, 63):
        sl = slice(h * D, (h + 1) * D)
        want_o, want_st, want_sn = O.kda_scan(*(np.ascontiguousarray(x[:, sl]) for x in (q, k, v, g)),
                                              np.ascontiguousarray(beta[:, h:h + 1]), state[h:h + 1].astype(np.float64),
                                              tokens=T, heads=1, snap=snap)
        assert_close(o[:, sl], want_o, f"o head {h}")
        assert_close(st[h], want_st[0], f"state head {h}")
        assert_close(sn[h], want_sn[0], f"snapshot head {h}")
    v[1000, 31 * D + 3] = float("nan")
    assert_same_where_finite(*both_routes(host, T=T, H=H, snap=snap))


@pytest.mark.parametrize("cut", ["exact", "short", "misaligned", "none"])
def test_scan_workspace(cut):
    """The bytes asked for: the library's own result; one less, a start off 16 bytes or none: token by token."""
    T, H, snap = 200, 2, 33
    host = inputs(np.random.default_rng(82), T, H, scale_state=0.3)
    need = M.kda_scan_workspace(tokens=T, heads=H, snap=snap)
    buf = torch.zeros(need + 16, dtype=torch.uint8, device="cuda")
    ws = {"exact": buf[:need], "short": buf[:need - 1], "misaligned": buf[8:], "none": None}[cut]
    res = []
    for w in (M.LIBRARY if cut == "exact" else None, ws):
        q, k, v, g, beta, st = (dev(x) for x in host)
        o, sn = torch.full_like(v, 7.0), torch.full_like(st, 7.0)
        M.kda_scan(q, k, v, g, beta, st, o, tokens=T, heads=H, snap=snap, snap_state=sn, workspace=w)
        torch.cuda.synchronize()
        res.append((o, st, sn))
    assert all(torch.equal(a, b) for a, b in zip(*res))
    assert int(buf[need:].sum()) == 0 and (cut == "exact" or int(buf.sum()) == 0)


def test_chunks_under_capture_with_a_workspace():
    """With the caller's workspace a captured call goes by chunks, and each replay has the eager call's bits."""
    rng = np.random.default_rng(83)
    T, H = 130, 2
    host = inputs(rng, T, H, scale_state=0.3)
    q, k, v, g, beta, st = (dev(x) for x in host)
    state0, o = st.clone(), torch.empty_like(v)
    ws = torch.empty(M.kda_scan_workspace(tokens=T, heads=H), dtype=torch.uint8, device="cuda")
    M.kda_scan(q, k, v, g, beta, st, o, tokens=T, heads=H, workspace=ws)
    torch.cuda.synchronize()
    want_o, want_st = o.clone(), st.clone()
    s = torch.cuda.Stream()
    s.wait_stream(torch.cuda.current_stream())
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph, stream=s):
        M.kda_scan(q, k, v, g, beta, st, o, tokens=T, heads=H, stream=s.cuda_stream, workspace=ws)
    for _ in range(3):
        st.copy_(state0)
        o.zero_()
        graph.replay()
        torch.cuda.synchronize()
        assert torch.equal(o, want_o) and torch.equal(st, want_st)


def test_outputs_in_the_place_of_v():
    """o in v's buffer, and the snapshot in the state's: as with buffers of their own, with a value that is not finite in
    the middle too."""
    T, H, snap = 130, 2, 40
    host = inputs(np.random.default_rng(84), T, H, scale_state=0.3)
    host[2][70, 3] = float("nan")
    _, (want_o, want_st, _) = both_routes(host, T=T, H=H, snap=snap)
    q, k, v, g, beta, st = (dev(x) for x in host)
    M.kda_scan(q, k, v, g, beta, st, v, tokens=T, heads=H, snap=snap, snap_state=st)
    torch.cuda.synchronize()
    assert_same_where_finite((v.cpu().numpy(), st.cpu().numpy()), (want_o, want_st))
