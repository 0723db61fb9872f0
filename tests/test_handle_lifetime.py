"""A handle's blob goes back to torch's allocator only when the device was
waited for: while it cannot be (a stream captures) the handle and its blob are
kept, and destroyed with a later handle."""

import ctypes
import gc

import pytest
import torch


class _Library:
    """Stands for the loaded library: a destruction that can be made to fail."""

    def __init__(self):
        self.fails = 0
        self.destroyed = []

    def fkv_attn_try_destroy(self, h):
        if self.fails:
            self.fails -= 1
            return -2
        self.destroyed.append(h.value)
        return 0

    def fkv_attn_blob_bytes(self, *shape):
        return 64


def _handle(lib, value):
    from foveated_kv_amd import ext

    h = ext.FoveatedHandle.__new__(ext.FoveatedHandle)
    h._lib, h._h = lib, ctypes.c_void_p(value)
    h._blob = torch.zeros(64, dtype=torch.uint8)
    return h


@pytest.fixture
def capturing(monkeypatch):
    state = {"now": False}
    monkeypatch.setattr(torch.cuda, "is_current_stream_capturing", lambda: state["now"])
    return state


def test_blob_is_kept_until_the_device_was_waited_for(capturing):
    import weakref

    from foveated_kv_amd import ext

    lib = _Library()
    h = _handle(lib, 11)
    blob = weakref.ref(h._blob)
    lib.fails = 1
    del h
    gc.collect()
    assert blob() is not None and lib.destroyed == []
    # while the current stream captures the device is not even waited for
    capturing["now"] = True
    h = _handle(lib, 12)
    del h
    gc.collect()
    capturing["now"] = False
    assert blob() is not None and lib.destroyed == []
    h = _handle(lib, 13)
    del h
    gc.collect()
    assert sorted(lib.destroyed) == [11, 12, 13] and blob() is None and not ext._undestroyed


def test_new_handle_destroys_the_kept_ones(capturing):
    from foveated_kv_amd import ext

    lib = _Library()
    h = _handle(lib, 21)
    lib.fails = 1
    del h
    gc.collect()
    assert lib.destroyed == [] and len(ext._undestroyed) == 1
    h = ext.FoveatedHandle.__new__(ext.FoveatedHandle)
    h.B = h.H_kv = h.D = h.N_near = h.N_far = 1
    h.device = torch.device("cpu")
    h._new_blob(lib, 0)
    assert lib.destroyed == [21] and not ext._undestroyed


def test_handle_alive_at_exit():
    """Destroyed without a message when the interpreter clears its modules."""
    import subprocess
    import sys

    code = """
import ctypes, os, torch
from foveated_kv_amd import ext
class Library:
    def fkv_attn_destroy(self, h, write=os.write):
        write(1, b"destroyed")
    fkv_attn_try_destroy = fkv_attn_destroy
h = ext.FoveatedHandle.__new__(ext.FoveatedHandle)
h._lib, h._h, h._blob = Library(), ctypes.c_void_p(5), None
torch.kept_for_the_test = h  # outlives the names of ext
"""
    r = subprocess.run([sys.executable, "-c", code], capture_output=True, text=True, timeout=300)
    assert r.returncode == 0 and r.stdout == "destroyed" and "Exception ignored" not in r.stderr


@pytest.mark.gpu
def test_handle_dropped_during_a_capture():
    """Replays of the handle's calls are in flight on another stream when it
    is dropped under capture: its blob is not handed out while they run, and
    goes back with the next handle."""
    from foveated_kv_amd import FoveatedKVCache, TierConfig, ext

    k, v = (torch.randn((2, 4, 6000, 128), device="cuda").half() for _ in range(2))
    q = torch.randn((2, 16, 1, 128), device="cuda").half()
    cache = FoveatedKVCache(TierConfig())
    cache.update(k, v, 0)
    cache.compress()
    lay = cache.layers[0]
    want = [t.clone() for t in lay.attend_fused_with_spikes(q)]
    side = torch.cuda.Stream()
    lay._kcache = None
    lay._ensure_kcache()
    h = lay._kcache.pop("cpp_handle")
    lay._kcache = None
    outs = [torch.empty_like(t) for t in want]
    h(q, out=outs)
    torch.cuda.synchronize()
    calls = torch.cuda.CUDAGraph()
    with torch.cuda.graph(calls):
        for _ in range(50):
            h(q, out=outs)
    nbytes = h._blob.numel()
    x = torch.zeros(1000, device="cuda")
    print("handle dropped under capture", flush=True)
    g = torch.cuda.CUDAGraph()
    with torch.cuda.graph(g):
        with torch.cuda.stream(side):
            for _ in range(20):
                calls.replay()
        del h
        gc.collect()
        y = x + 1
    kept = len(ext._undestroyed)
    junk = [torch.full((nbytes,), 255, dtype=torch.uint8, device="cuda") for _ in range(2)]
    torch.cuda.synchronize()
    assert kept == 1
    assert all(torch.equal(a, b) for a, b in zip(outs, want))
    x.fill_(4)
    for _ in range(3):
        g.replay()
        assert float(y.sum()) == 5000.0
    got = lay.attend_fused_with_spikes(q)  # a new handle
    assert all(torch.equal(a, b) for a, b in zip(got, want)) and not ext._undestroyed
    del junk, calls
