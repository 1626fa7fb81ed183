"""mp_dos spectra over more column groups than workgroups (each keeps its sums
over several groups, the last one ragged), a single group, and more sums than
a workgroup's registers keep, with the species in blocks and interleaved."""
import math

import numpy as np
import pytest
import torch

from mp_tools_amd import sqw

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("precision,tol", [("fp32", 1e-6), ("fp64", 1e-13)])
@pytest.mark.parametrize("T,n,nsp,mixed", [(64, 17000, 3, False), (60, 40003, 5, True), (512, 5001, 4, True),
                                           (512, 3, 2, False), (500, 700, 20, True), (1, 9, 2, True), (1200, 40, 3, True),
                                           (8192, 5, 2, False)])
def test_dos_column_groups(gpu_lib, precision, tol, T, n, nsp, mixed):
    g = np.random.default_rng(T + n)
    v = np.zeros((T, n, 4), np.float32)
    v[..., :3] = g.standard_normal((T, n, 3))
    ind = np.zeros((n, 4), np.int32)
    ind[:, 3] = (np.arange(n) % nsp if mixed else np.arange(n) * nsp // n) + 1
    nf = T // 2 + 1
    w = np.ones(1) if T == 1 else 0.5 * (1 - np.cos(2 * math.pi * np.arange(1, T + 1) / (T + 1)))
    p = np.empty((nf, n))
    for a in range(0, n, 2000):
        p[:, a:a + 2000] = (np.abs(np.fft.fft(v[:, a:a + 2000, :3].astype(np.float64) * w[:, None, None], axis=0)[:nf]) ** 2).sum(2) / T
    ref = np.stack([p[:, ind[:, 3] == s + 1].sum(1) for s in range(nsp)], 1)
    got = sqw.dos_spectra(torch.tensor(v, device="cuda"), torch.tensor(ind, device="cuda"), nsp, nf, precision=precision)
    # each power to FP32 (FP64) rounding of a T-point transform, summed in FP64
    assert np.abs(got.cpu().numpy() - ref).max() <= tol * np.abs(ref).max()
