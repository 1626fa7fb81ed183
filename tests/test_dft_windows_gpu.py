"""The DFT reductions (sliding windows; one window over a frame count without
a radix plan) at the edges of their groups: columns around a wave, frequency
counts around the per-wave groups, window lengths from one frame up, negative
first frequencies, cuts, and both amplitude precisions."""
import math

import numpy as np
import pytest
import torch

from mp_tools_amd import sqw

pytestmark = pytest.mark.gpu


def _ref(C, n, kind, m_lo, n_f, nat, dt, mean, qfac):
    T = C.shape[0]
    tot = (np.abs(C) ** 2).sum(0) / (T * nat * nat)
    if mean:
        C = C - C.mean(0)
    C = C * qfac
    i = np.arange(n)
    if n == 1:
        w = np.ones(1)
    else:
        w = 0.5 * (1 - np.cos(2 * math.pi * (i + 1) / (n + 1))) if kind else 0.5 * (1 - np.cos(2 * math.pi * i / (n - 1)))
    m = m_lo + np.arange(n_f)
    W = np.exp(-2j * math.pi * (np.outer(m, i) % n) / n) * w
    S = sum(np.abs(W @ C[s:s + n]) ** 2 for s in range(T - n + 1))
    return S * dt / (nat * nat * 0.5 * (T - n + 1) * n), tot


@pytest.mark.parametrize("precision", ["fp32", "fp64"])
@pytest.mark.parametrize("nx,ny,T,n_int,kind,m_lo,n_f,mean,cut", [
    (1, 1, 2, 1, 0, 0, 1, True, 0),
    (9, 7, 12, 2, 0, 0, 2, True, 0),
    (8, 8, 12, 2, 1, -1, 2, False, 0),
    (13, 5, 37, 11, 0, 0, 6, True, 0),
    (13, 5, 37, 11, 1, -7, 19, True, 0),
    (16, 16, 64, 33, 0, 0, 17, True, 0),
    (150, 150, 21, 11, 0, 0, 7, True, 0),
    (40, 40, 50, 25, 0, 0, 25, True, 33),
    (9, 7, 37, 37, 0, 0, 18, True, 0),
    (200, 200, 11, 11, 0, 0, 5, True, 0),
    (13, 5, 97, 97, 1, -48, 97, False, 0),
    (40, 40, 53, 53, 0, 0, 53, True, 65),
    (1, 1, 7, 7, 0, 3, 1, True, 0),
    (1, 1, 1, 1, 0, 0, 0, True, 0),
    (65, 3, 1, 1, 0, 0, 1, False, 0),
    (65, 3, 20, 20, 0, 0, 20, True, 0),
    (65, 3, 20, 20, 0, 0, 0, True, 0),
    (65, 3, 64, 64, 1, 0, 0, True, 33),
])
def test_dft_reductions(precision, nx, ny, T, n_int, kind, m_lo, n_f, mean, cut):
    g = np.random.default_rng(T * 1000 + n_f)
    nq = nx * ny
    C = g.standard_normal((T, nq)) + 1j * g.standard_normal((T, nq)) + 5.0
    C = C.astype(np.complex64 if precision == "fp32" else np.complex128)
    qf = g.uniform(0.5, 2.0, nq).astype(np.float32)
    eng = sqw.SqwEngine(2, (nx, ny), (10, 10), precision=precision)
    qidx = None
    if cut:
        qidx = torch.tensor(g.integers(0, nq, cut), dtype=torch.int32, device="cuda:0")
    S, St = eng.reduce(torch.tensor(C, device="cuda:0"), n_int=n_int, win_kind=kind, dt=0.01, nat=10.0, m_lo=m_lo,
                       n_f=n_f, subtract_mean=mean, qfac=torch.tensor(qf, device="cuda:0"), qidx=qidx)
    C = C.astype(np.complex128)
    q = np.arange(nq) if qidx is None else qidx.cpu().numpy()
    S0, T0 = _ref(C[:, q], n_int, kind, m_lo, n_f, 10.0, 0.01, mean, qf[q].astype(np.float64))
    # FP64 sums of at most ~100 unit-size terms per window: 1e-12 of the
    # largest value covers their rounding a thousandfold
    assert n_f == 0 or np.abs(S.cpu().numpy() - S0).max() <= 1e-12 * max(np.abs(S0).max(), np.abs(C).max() ** 2 * 1e-4)
    assert np.abs(St.cpu().numpy() - T0).max() <= 1e-12 * T0.max()


def test_one_frequency_of_a_long_series():
    """400 frames of 4,096 columns: one frequency takes no longer than half
    again as long as four (direct sums, a wave walking the frames alone, took
    1.8 times)."""
    eng = sqw.SqwEngine(2, (64, 64), (10, 10), precision="fp32")
    amp = torch.randn((400, 4096), device="cuda:0", dtype=torch.complex64)

    def fastest(n_f):
        out = eng.reduce(amp, n_int=400, n_f=n_f)
        best = 1e9
        for _ in range(30):
            eng.set_timing(True)
            eng.reduce(amp, n_int=400, n_f=n_f, out=out[0], out_tot=out[1])
            best = min(best, eng.timing()["reduce"][0])
        return best

    assert fastest(1) < 1.5 * fastest(4)
