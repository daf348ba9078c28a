"""The library's host side without a GPU: its objects linked with a HIP runtime that records allocations, frees and
launches and runs nothing (tests/cpp/fake_hip.cpp; 256 compute units). Pointers are never read."""
import ctypes
import os
import subprocess
import types

import pytest

torch = pytest.importorskip("torch")

from conftest import PKG, ROOT  # noqa: E402

import mako_attn as M  # noqa: E402

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
