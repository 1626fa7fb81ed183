"""Plan.execute on device tensors returns with its work queued: the tensors of
every queued call stay alive until that call's work is done, not until some
later call.  On the CPU with a stand-in for the library and its events; on the
GPU with plans on streams of their own and results that are dropped."""
import ctypes as C
import gc
import weakref
from collections import deque

import numpy as np
import pytest
import torch

from mp_tools_amd import nufft


class _Lib:
    @staticmethod
    def mpsq_execute_dev(h, c, f):
        return 0

    @staticmethod
    def mpsq_setpts_dev(h, m, x, y, z):
        return 0


class _Event:
    def __init__(self, log):
        self.done, self.log = False, log

    def query(self):
        return self.done

    def synchronize(self):
        self.log.append(self)
        self.done = True


class _Plan(nufft.Plan):
    """A 1D FP64 plan on a stream of its own, without a device."""

    def __init__(self):
        self._L, self._pre, self._h = _Lib(), "mpsq", C.c_void_p()
        self.n_modes, self.dim, self.n_trans, self.single = (8,), 1, 1, False
        self.rdtype, self.M, self._keep, self._device, self._stream = np.float64, 4, None, 0, 0
        self._inflight = deque()
        self.events, self.waits = [], []

    def _mark(self):
        self.events.append(_Event(self.waits))
        return self.events[-1]


def _call(p):
    """One execute whose strengths and result the caller drops."""
    c, out = torch.zeros(4, dtype=torch.complex128), torch.zeros(8, dtype=torch.complex128)
    refs = weakref.ref(c), weakref.ref(out)
    p.execute(c, out=out)
    del c, out
    gc.collect()
    return refs


def _alive(refs):
    gc.collect()
    return [r() is not None for r in refs]


def test_tensors_of_each_queued_call_are_held():
    p = _Plan()
    a, b = _call(p), _call(p)
    assert _alive(a) == _alive(b) == [True, True]  # neither call's work is known to be done
    p.events[0].done = True
    c = _call(p)
    assert _alive(a) == [False, False]
    assert _alive(b) == _alive(c) == [True, True]


def test_held_calls_are_bounded():
    p = _Plan()
    refs = [_call(p) for _ in range(10)]
    alive = [all(_alive(r)) for r in refs]
    assert alive == [False] * (9 - p.HOLD) + [True] * (p.HOLD + 1)
    assert p.waits == p.events[:9 - p.HOLD]  # each dropped call was waited for


def test_setpts_waits_and_drops():
    p = _Plan()
    a = _call(p)
    p.setpts(torch.zeros(4, dtype=torch.float64))
    assert _alive(a) == [False, False]
    assert not p.events  # one execute per setpts records no event


@pytest.mark.gpu
@pytest.mark.parametrize("dtype", ["complex64", "complex128"])
def test_dropped_results_of_two_plans(gpu_lib, dtype):
    """Back-to-back calls of two plans on streams of their own, every result
    but the last one dropped at once: equal to the same calls waited for."""
    g = torch.Generator(device="cuda")
    g.manual_seed(5)
    cdt = getattr(torch, dtype)
    rdt = torch.float64 if dtype == "complex128" else torch.float32
    m, nm = 20000, (64, 64, 16)
    x = [(torch.rand(m, generator=g, device="cuda", dtype=rdt) - 0.5) * 6.28 for _ in range(3)]
    c = [torch.randn(m, generator=g, device="cuda", dtype=cdt) for _ in range(4)]
    plans = [nufft.Plan(1, nm, eps=1e-6, isign=s, dtype=dtype) for s in (-1, 1)]
    for p in plans:
        p.setpts(*x)
    ref = []
    for p in plans:
        ref.append([])
        for v in c:
            ref[-1].append(p.execute(v).clone())
            torch.cuda.synchronize()
    for _ in range(5):
        kept = []
        for k in range(4):
            for i, p in enumerate(plans):
                p.execute(c[(k + 1) % 4] * 1.0)
                p.execute(c[(k + 2) % 4] * 1.0)
                kept.append((i, k, p.execute(c[k] * 1.0)))
        torch.cuda.synchronize()
        for i, k, f in kept:
            d = (f - ref[i][k]).abs().max().item()
            # atomics add in another order from run to run: rounding of the sum
            assert d <= (1e-5 if dtype == "complex64" else 1e-13) * ref[i][k].abs().max().item()
