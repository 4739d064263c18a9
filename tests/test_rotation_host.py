"""Lifetime of the pivot flags that rk_power_iteration writes to pinned host
memory: however a call ends, they outlive the pending write.  The device is a
stand-in whose kernel writes when its stream or event is waited for.
"""
import gc
import types
import weakref

import pytest
import torch

from rotatek_amd import _lib, rotation


class _Flags:
    """A pinned tensor (tensors have no weak references that outlive a slot)."""

    def any(self):
        return False

    def data_ptr(self):
        return 64


class _Pending:
    """A stream or event behind which the kernel's write to ``flags`` is pending."""

    cuda_stream = 0

    def __init__(self):
        self.flags, self.written_alive = None, None

    def synchronize(self):
        self.written_alive = self.flags() is not None


def _pivots():
    flags, done = _Flags(), _Pending()
    done.flags = weakref.ref(flags)
    return rotation._Pivots(flags, done), done


def test_dropped_unchecked_waits_for_the_write():
    p, done = _pivots()
    del p
    gc.collect()
    assert done.written_alive is True


def test_checked_waits_once():
    p, done = _pivots()
    p.check()
    assert done.written_alive is True
    done.written_alive = None
    p.check()
    del p
    gc.collect()
    assert done.written_alive is None


def test_failure_behind_the_launch_waits(monkeypatch):
    """An allocation that fails between the launch and the caller's check."""
    p, done = _pivots()

    class Out:
        def reshape(self, *shape):
            raise MemoryError

    box = [p]
    del p
    monkeypatch.setattr(rotation, "_start_block", lambda cov, k, seed: torch.zeros(2, 8, k))
    monkeypatch.setattr(rotation, "_launch", lambda *a: (Out(), box.pop()))
    with pytest.raises(MemoryError):
        rotation.deferred_power_iteration(torch.zeros(2, 8, 8), 4)
    gc.collect()
    assert done.written_alive is True


@pytest.mark.parametrize("fails", ["launch", "record"])
def test_failure_inside_the_launch_waits_for_the_stream(monkeypatch, fails):
    stream, flags = _Pending(), _Flags()
    stream.flags = weakref.ref(flags)
    box = [flags]
    del flags

    class Event:
        def record(self, s):
            raise RuntimeError("record")

    cuda = types.SimpleNamespace(Event=Event, current_stream=lambda dev: stream,
                                 is_current_stream_capturing=lambda: False)
    monkeypatch.setattr(rotation, "torch", types.SimpleNamespace(
        empty_like=lambda t: t, empty=lambda *a, **k: box.pop(), int32=None, cuda=cuda))
    lib = types.SimpleNamespace(rk_power_iteration=lambda *a: _lib.RK_ERR_HIP if fails == "launch" else 0,
                                rk_strerror=lambda s: b"")
    monkeypatch.setattr(_lib, "load", lambda: lib)
    cov = types.SimpleNamespace(is_cuda=True, shape=(1, 2, 8, 8), device=None)
    monkeypatch.setattr(_lib, "desc", lambda t: _lib.RkTensor())
    with pytest.raises(RuntimeError):
        rotation._launch(cov, object(), 5, 1e-4, True)
    gc.collect()
    assert stream.written_alive is True
