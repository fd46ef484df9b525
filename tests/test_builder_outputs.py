"""A builder's memory when an allocation fails: given back at once, not when the garbage collector runs."""
import gc
import weakref

import pytest
import torch

from mpserve_amd import _native
from mpserve_amd._common import BuilderOutputs


class _Args(_native.MpsFp8EncodeIn):
    pass


def _mem():
    return BuilderOutputs(torch.device("cpu"), {0: torch.uint16, 1: torch.uint8})


def test_a_failed_allocation_leaves_nothing_behind():
    mem = _mem()
    tensors = []

    def entry(_args, _stream, alloc, _ctx, _sizes, _stats):
        assert alloc(None, 0, 64) and alloc(None, -1, 256)
        tensors.extend(weakref.ref(t) for t in list(mem._out.values()) + mem._work)
        assert not alloc(None, 1, 1 << 62)  # torch has no such memory
        return 1

    gone = weakref.ref(mem)
    gc.disable()
    try:
        with pytest.raises(RuntimeError) as e:
            mem.build(entry, _Args(), 0)
        assert all(t() is None for t in tensors) and len(tensors) == 2  # while the error is still held
        del e, mem
        assert gone() is None
    finally:
        gc.enable()


def test_a_failed_build_frees_its_memory(monkeypatch):
    mem = _mem()
    monkeypatch.setattr(_native, "check", lambda rc: (_ for _ in ()).throw(RuntimeError("failed")) if rc else None)

    def entry(_args, _stream, alloc, _ctx, _sizes, _stats):
        assert alloc(None, 0, 64) and alloc(None, -1, 256)
        return 2

    with pytest.raises(RuntimeError, match="failed"):
        mem.build(entry, _Args(), 0)
    assert not mem._out and not mem._work


def test_outputs_are_kept():
    mem = _mem()
    sizes, stats = mem.build(lambda _a, _s, alloc, _c, _z, _t: 0 if alloc(None, 0, 64) else 1, _Args(), 0)
    assert mem.tensor(0, (4, 8), True).shape == (4, 8) and mem.tensor(1, (0,), True).numel() == 0
    assert len(sizes) == 17 and len(stats) == 4
