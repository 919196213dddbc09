"""Direct sums at the edges of their tiles: a wave takes 512 frequencies of a
linear grid (16 rows of 32) or 64 of a list, 4 points at a time, and 1, 2, 4 or
8 waves share a tile.

Tolerance: a sum of unit phasors with weights adding to one is off by at most
about 8 FP32 roundings of each term, 8 x 6e-8 = 5e-7; the power is a ratio of
quadratic forms in the sums, each form a few times a sum's error where the
normal matrix is within a factor 2 of a half (determinant 1/16 or more): 1e-5.
Below that the weights' own rounding to FP32 decides (5 points: 3e-5 at the
worst frequency of half of all curves, with or without matrix instructions).
"""
import numpy as np
import pytest

from oracle import gls as og

pytestmark = pytest.mark.gpu

TOL = 1e-5


def _curve(seed, n, T=20.0):
    rng = np.random.default_rng(seed)
    t = np.sort(rng.uniform(0, T, n))
    y = 2.0 + 0.8 * np.sin(2 * np.pi * t / 1.7) + rng.normal(0, 0.3, n)
    return t, y, rng.uniform(0.2, 0.5, n)


def _error(d, f, p):
    """max |dP| over the well-conditioned frequencies, as the tolerance assumes."""
    t, y, dy = d
    C, S, C2, S2 = og.direct_sums(t, og.weights(dy), np.zeros(len(t)), f)[:4]
    det = ((0.5 * (1 + C2) - C * C) * (0.5 * (1 - C2) - S * S) - (0.5 * S2 - C * S) ** 2)
    e = np.abs(p - og.gls_direct(t, y, dy, f))
    return float(np.max(e[det >= 1 / 16], initial=0.0))


def _powers(data, freqs, **kw):
    from cuvarbase_amd.engine import LombBatch

    return LombBatch(data, freqs, use_fft=False, **kw).run()


@pytest.mark.parametrize("custom", [False, True])
@pytest.mark.parametrize("nfs", [(2, 31, 32, 33), (63, 64, 65, 511), (512, 513, 1025, 4097)])
def test_tile_edges(nfs, custom):
    # 5 .. 260 points: partial groups of 4, one group per wave and several
    data = [_curve(i, n) for i, n in enumerate((5, 31, 64, 260))]
    freqs = [0.15 + 0.01 * np.arange(nf) for nf in nfs]
    if custom:
        freqs = [f[::-1].copy() for f in freqs]
    for d, f, p in zip(data, freqs, _powers(data, freqs, custom_freqs=custom)):
        assert p.shape == f.shape
        assert _error(d, f, p) < TOL


# waves per tile 1, 2, 4, 8 (300 points) and 1 (60 points)
@pytest.mark.parametrize("n, nf", [(300, 2_097_160), (300, 1_048_600), (300, 524_300),
                                   (300, 5000), (60, 5000)])
@pytest.mark.parametrize("custom", [False, True])
def test_waves_per_tile(n, nf, custom):
    if custom:
        nf //= 8   # 64 frequencies per wave instead of 512
    d = _curve(n, n)
    f = 0.15 + 2e-4 * np.arange(nf)
    p = _powers([d], [f], custom_freqs=custom)[0]
    sel = np.unique(np.concatenate([np.arange(40), np.arange(nf - 40, nf),
                                    np.random.default_rng(1).integers(0, nf, 300)]))
    assert _error(d, f[sel], p[sel]) < TOL


def test_double_output_and_missing_values():
    t, y, dy = _curve(3, 131)
    f = 0.15 + 0.01 * np.arange(700)
    p = _powers([(t, y, dy)], [f], use_double=True)[0]
    assert p.dtype == np.float64 and _error((t, y, dy), f, p) < TOL
    t[7] = np.nan   # a point without a time makes every power of its curve invalid
    p, q = _powers([(t, y, dy), _curve(4, 50)], [f, f])
    assert np.all(p == -1.0) and np.all(q >= 0.0)
