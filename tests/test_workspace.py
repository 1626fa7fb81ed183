"""Engine grids in a buffer of the caller's: buffers the kernels could not
write are refused before the library sees them, and lent and own grids give the
same amplitudes."""
import ctypes as C

import numpy as np
import pytest
import torch

from mp_tools_amd.sqw import SqwEngine


class _Buf:
    """What set_workspace looks at in a tensor."""

    def __init__(self, cuda=True, index=0, contiguous=True):
        self.is_cuda, self.device, self._c = cuda, torch.device("cuda", index), contiguous

    def is_contiguous(self):
        return self._c

    def numel(self):
        return 1 << 20

    def element_size(self):
        return 1

    def data_ptr(self):
        return 1 << 12


class _Lib:
    def __init__(self):
        self.calls = []

    def mpsq_sqw_set_workspace(self, *a):
        self.calls.append(a)
        return 0


def _engine():
    e = object.__new__(SqwEngine)
    e._L, e._h, e.device = _Lib(), C.c_void_p(), 0
    return e


@pytest.mark.parametrize("buf", [_Buf(cuda=False), _Buf(index=1), _Buf(contiguous=False), torch.zeros(1 << 20, dtype=torch.uint8)])
def test_unusable_buffers_are_refused(buf):
    e = _engine()
    with pytest.raises(ValueError):
        e.set_workspace(buf)
    assert not e._L.calls


def test_usable_buffers_pass():
    e = _engine()
    e.set_workspace(_Buf())
    e.set_workspace(None)
    assert len(e._L.calls) == 2


@pytest.mark.gpu
@pytest.mark.parametrize("precision", ["fp32", "fp64"])
@pytest.mark.parametrize("nm,kw", [((24, 20, 12), {}), ((24, 20, 12), dict(q0=(0.25, 0.0, 0.0))), ((32, 31), {}),
                                   ((24, 20, 12), dict(table=True)), ((16, 12, 8), dict(combine=False))])
def test_lent_and_own_grids_agree(gpu_lib, precision, nm, kw):
    from mp_tools_amd._lib import MpsqError
    kw, g = dict(kw), np.random.default_rng(3)
    T, counts = 5, (300, 200)
    pos = np.zeros((T, 500, 4), np.float32)
    pos[..., :3] = g.uniform(0.1, 6.1, (T, 500, 3))
    pos = torch.tensor(pos, device="cuda")
    if kw.pop("table", False):
        kw["weight_table"] = g.uniform(0.5, 2.0, (2, int(np.prod(nm)))).astype(np.float32)
    eng = SqwEngine(len(nm), nm, counts, precision=precision, **kw)
    own = eng.amplitudes(pos).clone()

    def same(frames):
        # FP64 cells are added by atomics, in another order from run to run
        d = (eng.amplitudes(pos[:frames]) - own[:frames]).abs().max().item()
        return d <= (0.0 if precision == "fp32" else 1e-13) * own.abs().max().item()

    for frames in (1, T):
        n = eng.workspace_bytes(frames)
        buf = torch.empty(n + 256, dtype=torch.uint8, device="cuda")
        with pytest.raises(MpsqError):
            eng.set_workspace(buf[:n - 1], frames)
        with pytest.raises(MpsqError):
            eng.set_workspace(buf[1:], frames)
        eng.set_workspace(buf[:n], frames)
        buf[n:] = 77
        assert same(frames)
        assert (buf[n:] == 77).all()  # nothing past the bytes asked for
        buf[:n] = 0
        assert same(frames) and bool(buf[:n].any())  # the grids are in the buffer
        assert same(T)  # more frames than lent for: memory of the engine's own
        eng.set_workspace(buf[:n], frames)
        eng.set_workspace(None)
        buf[:n] = 0
        assert same(T) and not bool(buf[:n].any())
    eng.destroy()
    assert eng._ws is None
