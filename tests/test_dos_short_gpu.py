"""mp_dos spectra of short series, whose groups hold up to 512 columns, with the
species in blocks, in layers (the type changes from group to group),
interleaved, and more of them than one table of types holds; and what a short
series costs."""
import math

import numpy as np
import pytest
import torch

from mp_tools_amd import sqw

pytestmark = pytest.mark.gpu


def _types(n, nsp, order):
    a = np.arange(n)
    return {"blocks": a * nsp // n, "layers": a // 512 % nsp, "mixed": a % nsp,
            "outside": a % (nsp + 2) - 1}[order]  # some types of no species: they count for nothing


@pytest.mark.parametrize("precision,tol", [("fp32", 1e-6), ("fp64", 1e-13)])
@pytest.mark.parametrize("T,n,nsp,order", [(20, 150001, 5, "blocks"), (20, 150001, 5, "layers"), (8, 140003, 3, "mixed"),
                                           (2, 140000, 2, "blocks"), (3, 140000, 2, "outside"), (1, 300001, 2, "mixed"),
                                           (50, 3001, 130, "mixed"), (200, 900, 70, "outside"), (128, 40000, 3, "layers"),
                                           (1200, 60, 3, "layers"), (2048, 33, 5, "mixed")])
def test_short_series(gpu_lib, precision, tol, T, n, nsp, order):
    g = np.random.default_rng(T + n)
    v = np.zeros((T, n, 4), np.float32)
    v[..., :3] = g.standard_normal((T, n, 3))
    ty = _types(n, nsp, order)
    ind = np.zeros((n, 4), np.int32)
    ind[:, 3] = ty + 1
    nf = T // 2 + 1
    w = np.ones(1) if T == 1 else 0.5 * (1 - np.cos(2 * math.pi * np.arange(1, T + 1) / (T + 1)))
    p = np.empty((nf, n))
    for a in range(0, n, 20000):
        p[:, a:a + 20000] = (np.abs(np.fft.fft(v[:, a:a + 20000, :3].astype(np.float64) * w[:, None, None], axis=0)[:nf]) ** 2).sum(2) / T
    ref = np.stack([p[:, ty == s].sum(1) for s in range(nsp)], 1)
    got = sqw.dos_spectra(torch.tensor(v, device="cuda"), torch.tensor(ind, device="cuda"), nsp, nf, precision=precision)
    # each power to FP32 (FP64) rounding of a T-point transform, summed in FP64
    assert np.abs(got.cpu().numpy() - ref).max() <= tol * np.abs(ref).max()


def test_short_series_cost_less(gpu_lib):
    """20 frames of 40,000 atoms take less time than 200 of them (a third of it;
    a partial row per share of the columns made them take longer)."""
    def fastest(T, n=40000):
        v = torch.randn((T, n, 4), device="cuda")
        ind = torch.zeros((n, 4), dtype=torch.int32, device="cuda")
        ind[:, 3] = torch.arange(n, device="cuda", dtype=torch.int32) * 5 // n + 1
        best = 1e9
        for _ in range(20):
            e = [torch.cuda.Event(enable_timing=True) for _ in range(2)]
            e[0].record()
            sqw.dos_spectra(v, ind, 5, T // 2)
            e[1].record()
            e[1].synchronize()
            best = min(best, e[0].elapsed_time(e[1]))
        return best

    assert fastest(20) < fastest(200)
