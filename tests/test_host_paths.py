"""The library's host side without a GPU: its objects linked with a HIP runtime that records allocations, frees and
launches and runs nothing (tests/cpp/fake_hip.cpp; 256 compute units). Pointers are never read."""
import ctypes
import os
import re
import subprocess
import threading
import types

import pytest

torch = pytest.importorskip("torch")

from conftest import PKG, ROOT  # noqa: E402

import mako_attn as M  # noqa: E402
import test_gpu_proj as P  # noqa: E402

U32 = 0xFFFFFFFF
FAKE_SO = os.path.join(ROOT, "tests", "cpp", "bin", "libmako_attn_fakehip.so")


@pytest.fixture
def hip(monkeypatch):
    if not os.path.exists(os.path.join(PKG, "_build", "status.o")):
        subprocess.run(["make", "-s", "-j8", "-C", PKG], check=True)
    subprocess.run(["make", "-s", "-C", os.path.join(ROOT, "tests", "cpp"), "bin/libmako_attn_fakehip.so"], check=True)
    monkeypatch.setattr(M, "LIB_PATH", FAKE_SO)
    monkeypatch.setattr(M, "_lib", None)
    L = M.lib()
    L.fake_events.restype = ctypes.c_char_p
    L.fake_alloc_limit.argtypes = [ctypes.c_size_t]
    L.fake_capture.argtypes = [ctypes.c_void_p, ctypes.c_int]
    L.fake_clear()
    yield L


def events(L, *kinds):
    return [e for e in (line.split() for line in L.fake_events().decode().splitlines()) if not kinds or e[0] in kinds]


def launches(L):
    return [e[1] for e in events(L, "launch")]


def tensor(dtype, addr=0x100000):
    return types.SimpleNamespace(dtype=dtype, data_ptr=lambda: addr)


def attn(n_q, n_k, stream, *, dim=128, heads=32, kv=8, dtype=torch.bfloat16):
    x = tensor(dtype)
    M.attn_fwd(x, x, x, x, n_q=n_q, q_pad=n_q, n_k=n_k, k_pad=n_k, heads=heads, kv_heads=kv, q_pos0=n_k - n_q,
               block=U32, dim=dim, stream=stream)


def rows(n_q, n_k, stream, *, dim=128, heads=32, kv=8):
    x = tensor(torch.float32)
    h = lambda n, r: dict(rows=r, ld=n * dim, col0=0, stride=dim, dim=dim, heads=n)  # noqa: E731
    M.attn_fwd_rows(x, x, x, tensor(torch.bfloat16), h(heads, n_q), h(kv, n_k), h(kv, n_k), n_q=n_q, n_k=n_k,
                    heads=heads, kv_heads=kv, q_pos0=n_k - n_q, block=U32, in_dtype=M.BF16, stream=stream)


@pytest.mark.parametrize("prefill", [attn, rows], ids=["tiles", "rows"])
def test_split_prefill_leaves_a_captured_calls_workspace(hip, prefill):
    """A few-row call's workspace may be in a captured graph once it has been made: a prefill on the stream, whose split
    takes more memory, neither moves nor frees it."""
    s = 0x51000
    attn(1, 4096, s)
    held = [e[1] for e in events(hip, "alloc")]
    assert len(held) == 1
    hip.fake_capture(s, 1)
    attn(1, 4096, s)
    hip.fake_capture(s, 0)
    hip.fake_clear()
    prefill(333, 9333, s)
    assert any("merge_pieces" in k for k in launches(hip)), "the prefill is not split"
    assert events(hip, "free") == []
    hip.fake_clear()
    attn(1, 4096, s)
    assert events(hip, "alloc") == []
    M.release(stream=s)
    assert held[0] in [e[1] for e in events(hip, "free")]


def test_split_prefill_without_memory_keeps_the_other_workspaces(hip):
    """Where the pieces' memory cannot be had the prefill runs unsplit, and what other calls hold stays."""
    s = 0x52000
    attn(1, 4096, s)
    hip.fake_clear()
    hip.fake_alloc_limit(1 << 20)
    try:
        attn(333, 9333, s)
    finally:
        hip.fake_alloc_limit(ctypes.c_size_t(-1).value)
    assert len(launches(hip)) == 1 and events(hip, "free") == []
    M.release(stream=s)


def proj(t, stream, k=4096, n=4096):
    M.proj_bf16(tensor(torch.bfloat16), tensor(torch.float32), tensor(torch.float32), t=t, k=k, n=n, stream=stream)


def scan(tokens, stream):
    x, o = tensor(torch.float32), tensor(torch.float32, 0x40000000)
    M.kda_scan(x, x, x, x, x, x, o, tokens=tokens, heads=4, stream=stream)


# a call whose launches pass a workspace on, and one that needs more of it
TWO_LAUNCHES = {
    "proj": (lambda s: proj(256, s), lambda s: proj(512, s)),
    "scan": (lambda s: scan(128, s), lambda s: scan(256, s)),
    "prefill": (lambda s: attn(333, 9333, s), lambda s: attn(333, 20000, s)),
    "few rows": (lambda s: attn(1, 4096, s), lambda s: attn(2, 40000, s)),
    "rows": (lambda s: rows(300, 300, s), lambda s: rows(600, 600, s)),
}


@pytest.mark.parametrize("name", TWO_LAUNCHES)
def test_threads_on_one_stream_take_turns(hip, name):
    """Another thread's call on the stream, made between a call's two launches, neither launches in between nor frees
    the buffer they share, and runs after it."""
    first, second = TWO_LAUNCHES[name]
    s = 0x53000
    other = threading.Thread(target=second, args=(s,))
    main = threading.get_ident()
    seen = []

    @ctypes.CFUNCTYPE(None, ctypes.c_char_p)
    def hook(kernel):
        seen.append(threading.get_ident() == main)
        if len(seen) == 1:
            other.start()
            other.join(0.3)  # (time enough to come between)

    hip.fake_launch_hook(hook)
    try:
        first(s)
        other.join()
    finally:
        hip.fake_launch_hook(None)
    n = seen.index(False)
    assert n >= 2 and not any(seen[n:]), seen
    kinds = [e[0] for e in events(hip, "launch", "free")]
    assert "free" not in kinds[:n]
    M.release(stream=s)


PER_THREAD = 2  # hipStreamPerThread


def test_per_thread_stream(hip):
    """hipStreamPerThread is a stream of the calling thread: a workspace that has to be is the thread's own, and calls
    that run without one do."""
    for call in (TWO_LAUNCHES["proj"][0], TWO_LAUNCHES["scan"][0], TWO_LAUNCHES["prefill"][0]):
        hip.fake_clear()
        call(PER_THREAD)
        assert events(hip, "alloc") == [] and len(launches(hip)) == 1, launches(hip)
    hip.fake_clear()

    def few_rows():
        attn(1, 4096, PER_THREAD)
        attn(1, 4096, PER_THREAD)
        M.release(stream=PER_THREAD)

    attn(1, 4096, PER_THREAD)
    other = threading.Thread(target=few_rows)
    other.start()
    other.join()
    attn(1, 4096, PER_THREAD)
    allocs, frees = ([e[1] for e in events(hip, k)] for k in ("alloc", "free"))
    assert len(allocs) == 2 and frees == allocs[1:]
    M.release(stream=PER_THREAD)


def test_release_frees_every_workspace_of_the_stream(hip):
    s, before = 0x54000, M.held_bytes()
    for first, _ in TWO_LAUNCHES.values():
        first(s)
    allocs = [e[1] for e in events(hip, "alloc")]
    assert M.held_bytes() - before == sum(int(e[2]) for e in events(hip, "alloc"))
    M.release(stream=s)
    assert sorted(e[1] for e in events(hip, "free")) == sorted(allocs) and M.held_bytes() == before


def kernels(L):
    """The projection's launches, as kernel<template arguments>."""
    out = []
    for name in launches(L):
        kernel = re.search(r"proj_few|proj_ring|proj_dma|proj_tiles|round_rows", name).group()
        args = [{"0": "false", "1": "true"}[v] if t == "b" else v for t, v in re.findall(r"L([ib])(\d+)E", name)]
        out.append(f"{kernel}<{', '.join(args)}>" if args else kernel)
    return out


@pytest.mark.parametrize("kernel,call", [(k, c) for k, calls in P.TILES.items() for c in calls])
def test_projection_tiles(hip, kernel, call):
    t, k, n, ldx, ldy = call
    f32, split = ["round_rows<false>", kernel], ["round_rows<true>", kernel]
    if call in P.SHORT_K:
        f32 = ["proj_tiles<256, true, false>"]
    if call in P.SPLIT_TILES:
        split = ["proj_tiles<128, true, true>"]
    for dtype, split, want in ((torch.bfloat16, 0, [kernel]), (torch.float32, 0, f32), (torch.float32, 1, split)):
        hip.fake_clear()
        M.proj_bf16(tensor(torch.bfloat16), tensor(dtype), tensor(torch.float32), t=t, k=k, n=n, ldx=ldx, ldy=ldy,
                    split=split, stream=0x55000)
        assert kernels(hip) == want


@pytest.mark.parametrize("kernel,call", [(k, c) for k, calls in P.FEW.items() for c in calls])
def test_projection_of_a_few_rows(hip, kernel, call):
    xd, split, t, k, n = call
    M.proj_bf16(tensor(torch.bfloat16), tensor(torch.float32 if xd == P.O.F32 else torch.bfloat16), tensor(torch.float32),
                t=t, k=k, n=n, split=split, stream=0x55000)
    assert kernels(hip)[-1] == kernel


@pytest.mark.parametrize("kernel,call", [(k, c) for k, calls in P.NO_WORKSPACE.items() for c in calls])
def test_projection_without_a_workspace(hip, kernel, call):
    t, k, n, split, ldx, ldy = call
    for stream, workspace in ((0x55000, None), (0x56000, M.LIBRARY)):
        hip.fake_clear()
        hip.fake_capture(0x56000, 1)
        M.proj_bf16(tensor(torch.bfloat16), tensor(torch.float32), tensor(torch.float32), t=t, k=k, n=n, ldx=ldx, ldy=ldy,
                    split=split, stream=stream, workspace=workspace)
        hip.fake_capture(0x56000, 0)
        assert kernels(hip) == [kernel] and events(hip, "alloc") == []


@pytest.mark.parametrize("heads,kv,n_q,n_k,q_pos0,block,split", [
    # rows on both sides of `block` in one item of query rows: its keys past the first row's stay in one piece
    (32, 8, 445, 1125, 3, 59, False), (16, 8, 867, 1563, 9, 99, False), (24, 24, 806, 7685, 186, 263, False),
    (32, 8, 200, 2100, 700, 800, False), (8, 2, 200, 2100, 700, 800, True), (32, 8, 200, 2100, 1700, 1800, True),
    (32, 8, 333, 9333, 9000, U32, True), (32, 8, 333, 9333, 0, 0, True), (32, 8, 1531, 1531, 0, U32, False),
])
def test_prefill_is_split_where_its_longest_piece_is_shorter(hip, heads, kv, n_q, n_k, q_pos0, block, split):
    assert (M.attn_fwd_workspace(n_q=n_q, q_pad=n_q, n_k=n_k, k_pad=n_k, heads=heads, kv_heads=kv, q_pos0=q_pos0,
                                 block=block, dim=128) > 0) == split


@pytest.mark.parametrize("heads,tokens,snap,chunks", [
    (1, 95, 0, False), (1, 96, 0, True), (32, 96, 0, True), (32, 4096, 0, True), (64, 96, 0, True), (64, 96, 51, False),
    (64, 100, 0, False), (64, 200, 0, True), (256, 100, 0, False), (256, 1024, 0, True), (512, 200, 0, False),
    (1024, 100, 53, False), (1024, 200, 0, False), (4000, 1024, 0, False),
])
def test_scan_goes_by_chunks_where_they_are_faster(hip, heads, tokens, snap, chunks):
    assert (M.kda_scan_workspace(tokens=tokens, heads=heads, snap=snap) > 0) == chunks
    x, o, st = (tensor(torch.float32, a) for a in (0x100000, 1 << 44, 1 << 45))
    M.kda_scan(x, x, x, x, x, x, o, tokens=tokens, heads=heads, snap=snap, snap_state=st, stream=0x57000)
    assert any("kda_scan_chunks" in k for k in launches(hip)) == chunks
    M.release(stream=0x57000)
