"""The leading frequencies of a curve, |f| (t_max - t_min) < 3, against FP64 direct
sums at the point counts where the kernel changes its ways: one wave or a
workgroup for a few frequencies, slices of curves above 16,384 points, more
curves than workgroups per curve.

The NFFT runs at a coarse setting (Gaussian, sigma = 1.25, m = 2: |dP| ~ 1e-3), so
that only the direct sums can meet the tolerance, 1e-5: from one cycle over the
baseline on, the weights' rounding to FP32 (6e-8 of each) moves the power by
less than 100 of it (below, the normal matrix is nearly singular).
"""
import numpy as np
import pytest

from oracle import gls as og

pytestmark = pytest.mark.gpu

TOL = 1e-5


def _curve(seed, n, T=60.0):
    rng = np.random.default_rng(seed)
    t = np.sort(rng.uniform(0, T, n))
    y = np.sin(2 * np.pi * t / 9.0) + rng.normal(0, 0.5, n)
    return t, y, rng.uniform(0.3, 0.6, n)


@pytest.mark.parametrize("sizes", [(60, 255, 256, 257), (4097, 16384), (16385, 40000),
                                   (100, 20000, 700, 17000), (300,) * 600],
                         ids=["short", "block", "wide", "mixed", "many"])
@pytest.mark.parametrize("per_cycle", [5, 23])
def test_low_frequencies(sizes, per_cycle):
    from cuvarbase_amd.engine import LombBatch

    data = [_curve(i, n) for i, n in enumerate(sizes)]
    freqs = [(1 + np.arange(900)) / (per_cycle * np.ptp(t)) for t, _, _ in data]
    out = LombBatch(data, freqs, sigma=1.25, m=2).run()
    check = range(len(sizes)) if len(sizes) < 10 else (0, 1, 299, 598, 599)
    for i in check:
        f = freqs[i]
        low = np.flatnonzero((f * np.ptp(data[i][0]) < 3.0) & (f * np.ptp(data[i][0]) >= 1.0))
        assert len(low) >= 2 * per_cycle - 1
        assert np.max(np.abs(out[i][low] - og.gls_direct(*data[i], f[low]))) < TOL
