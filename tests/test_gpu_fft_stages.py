"""Grids whose column and row transforms end in every radix, with the twiddles of
the power-of-two stages taken inside their butterflies: powers at sampled
frequencies against FP64 direct sums.

The window (exponential of a semicircle, sigma = 1.5, m = 6) is good to 1e-7, and
the transforms' FP32 error is below 4e-6 of their RMS output (about sqrt(N)
times a deviate); 300 points of unit weight keep the amplitudes' rounding to
4e-6 / sqrt(300) = 2e-7 of the root of chi2_0, amplified by the deconvolution
at the band's edge (up to 10): 2 sqrt(P) times that is below 5e-6.
"""
import numpy as np
import pytest

from cuvarbase_amd import _lib, engine
from oracle import gls as og

pytestmark = pytest.mark.gpu

TOL = 5e-6


@pytest.mark.parametrize("spread", [_lib.SPREAD_FLOAT, _lib.SPREAD_FIXED], ids=["float", "fixed"])
@pytest.mark.parametrize("n1,p2", [(16, 12), (40, 11), (48, 10), (72, 9), (80, 8), (128, 7),
                                   (144, 6), (200, 9), (256, 8), (384, 7), (400, 6), (405, 6),
                                   (432, 6), (640, 6), (648, 6), (768, 6), (1080, 6), (1152, 6),
                                   (1280, 6), (2048, 6), (2160, 6), (2304, 6),
                                   (3072, 6), (3200, 6), (3240, 6), (3456, 6), (4096, 6)])
def test_stages_against_direct_sums(n1, p2, spread):
    rng = np.random.default_rng(n1)
    nf = int((n1 << p2) / 1.5) - 2
    T = 50.0
    freqs = (20 + np.arange(nf)) / (5 * T)   # from four cycles over the baseline on
    data = []
    for _ in range(2):
        t = np.sort(rng.uniform(0, T, 300))
        y = np.sin(2 * np.pi * t / 1.7) + rng.normal(0, 0.4, 300)
        data.append((t, y, rng.uniform(0.3, 0.6, 300)))
    engine.set_grid_cost(n1, p2, 1e-6)   # makes it the plan's choice of size
    try:
        b = engine.LombBatch(data, [freqs, freqs], sigma=1.5, m=6, window=_lib.WINDOW_ES,
                             spread=spread)
    finally:
        engine.set_grid_cost(n1, p2, 0.0)
    assert b.plan.geometry(1)[1:3] == (n1, 1 << p2)
    out = b.run()
    at = np.unique(np.concatenate([np.arange(40), nf - 1 - np.arange(40), nf // 2 + np.arange(-20, 20),
                                   rng.integers(0, nf, 200)]))
    for p, d in zip(out, data):
        assert np.max(np.abs(p[at] - og.gls_direct(*d, freqs[at]))) < TOL
