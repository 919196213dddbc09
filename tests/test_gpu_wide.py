"""Preparation of curves above 16,384 points over chunks of 1,024: around whole
chunks, beyond 1,024 chunks (longer chunks), and with the most buckets a grid
has (rows of 4,096 cells, one column per tile), in a batch and alone.

Tolerance: sigma = 2, m = 8 meets |dP| <= 2e-5 from one cycle over the baseline
on (alias 3e-7, FP32 grid round-off 1e-6 amplified by the deconvolution below 10).
"""
import numpy as np
import pytest

from oracle import gls as og

pytestmark = pytest.mark.gpu

TOL = 2e-5


def _curve(seed, n, T=400.0):
    rng = np.random.default_rng(seed)
    t = np.sort(rng.uniform(0, T, n))
    y = 15.0 + np.sin(2 * np.pi * t / 1.7) + rng.normal(0, 0.5, n)
    return t, y, rng.uniform(0.3, 0.6, n)


def _check(d, f, p, count=60):
    sel = np.unique(np.linspace(12, len(f) - 1, count).astype(int))
    assert np.max(np.abs(p[sel] - og.gls_direct(*d, f[sel]))) < TOL


@pytest.mark.parametrize("sizes", [(16385, 17408, 17409), (65536, 16384, 40961)])
def test_around_whole_chunks(sizes):
    from cuvarbase_amd import _lib
    from cuvarbase_amd.engine import LombBatch

    data = [_curve(n, n) for n in sizes]
    f = (1 + np.arange(6000)) / 2000.0
    kw = dict(sigma=2, m=8, spread=_lib.SPREAD_FIXED)
    out = LombBatch(data, [f] * len(data), **kw).run()
    for d, p in zip(data, out):
        _check(d, f, p)
        assert np.array_equal(p, LombBatch([d], [f], **kw).run()[0])


def test_weighted_input_and_missing_times():
    from cuvarbase_amd.engine import LombBatch

    t, y, dy = _curve(3, 30_001)
    f = (1 + np.arange(6000)) / 2000.0
    w = og.weights(dy)
    ybar = float(np.dot(w, y))
    yy = float(np.dot(w, (y - ybar) ** 2))
    args = dict(sigma=2, m=8, input_kind="weighted", ybar=[ybar], yy=[yy])
    _check((t, y, dy), f, LombBatch([(t, w * (y - ybar), w)], [f], **args).run()[0])
    # points without a time contribute nothing to the sums
    t2 = np.concatenate([t, np.full(5, np.nan)])
    w2, y2 = np.concatenate([w, np.zeros(5)]), np.concatenate([y, np.full(5, ybar)])
    _check((t, y, dy), f, LombBatch([(t2, w2 * (y2 - ybar), w2)], [f], **args).run()[0])


def test_more_than_1024_chunks():
    from cuvarbase_amd.engine import LombBatch

    d = _curve(5, (1 << 20) + 1025)
    f = (1 + np.arange(4000)) / 2000.0
    _check(d, f, LombBatch([d], [f], sigma=2, m=8).run()[0], count=12)


def test_most_buckets():
    from cuvarbase_amd.engine import LombBatch

    d = _curve(6, 16_500)
    f = (1 + np.arange(4_300_000)) / 2000.0
    b = LombBatch([d], [f], sigma=2, m=8)
    assert b.plan.geometry(0)[2] // b.plan.tiles(0)[0] == 4096
    _check(d, f, b.run()[0])
