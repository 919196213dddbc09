"""Pass-1 tiles on both sides of the point count from which a thread spreads all the
columns of a point, not one: powers at sampled frequencies against FP64 direct
sums.

The tolerance is that of a transform's FP32 error, 4e-6 of its RMS output of
sqrt(N) deviates: 4e-6 / sqrt(N) of the root of chi2_0, times 10 for the
deconvolution at the band's edge, 2 sqrt(P) <= 2 for the square and 2 for normal
matrices that are not diagonal at 60 points.
"""
import numpy as np
import pytest

from cuvarbase_amd import _lib, engine
from oracle import gls as og

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("spread", [_lib.SPREAD_FLOAT, _lib.SPREAD_FIXED], ids=["float", "fixed"])
@pytest.mark.parametrize("window", [_lib.WINDOW_ES, _lib.WINDOW_GAUSSIAN], ids=["es", "gaussian"])
@pytest.mark.parametrize("n1,p2", [(16, 6), (72, 6), (216, 6), (432, 6), (1280, 6)])
def test_points_per_tile(n1, p2, window, spread):
    # 64 columns, c1 of them per tile and a window of 2 m + 1: a tile sees
    # N (c1 + 2 m) / 64 points, its threads take a column each up to 512 / c1
    m = 6 if window == _lib.WINDOW_ES else 12
    sizes = (60, 64, 100, 180, 260, 500, 700, 1100, 1500, 2500)
    rng = np.random.default_rng(n1 + m)
    nf = int((n1 << p2) / 2.0) - 2
    T = 50.0
    freqs = (20 + np.arange(nf)) / (5 * T)
    data = []
    for n in sizes:
        t = np.sort(rng.uniform(0, T, n))
        data.append((t, np.sin(2 * np.pi * t / 1.7) + rng.normal(0, 0.4, n),
                     rng.uniform(0.3, 0.6, n)))
    engine.set_grid_cost(n1, p2, 1e-6)   # makes it the plan's choice of size
    try:
        b = engine.LombBatch(data, [freqs] * len(data), sigma=2.0, m=m, window=window,
                             spread=spread)
    finally:
        engine.set_grid_cost(n1, p2, 0.0)
    assert b.plan.geometry(0)[1:3] == (n1, 1 << p2)
    at = np.unique(np.concatenate([np.arange(40), nf - 1 - np.arange(40), rng.integers(0, nf, 200)]))
    for p, d, n in zip(b.run(), data, sizes):
        assert np.max(np.abs(p[at] - og.gls_direct(*d, freqs[at]))) < 1.6e-4 / np.sqrt(n), n
