"""Descriptors of a plan on their way to the device: as arguments of the first
launch (up to 3,584 bytes: about a dozen curves), or through the staging ring,
whose spans are reused after 16 MiB, also when the stream that read them is gone.

With fixed-point spreading a curve's powers are bitwise the same in any batch.
"""
import numpy as np
import pytest

from oracle import gls as og

pytestmark = pytest.mark.gpu


def _curve(seed, n=40):
    rng = np.random.default_rng(seed)
    t = np.sort(rng.uniform(0, 30.0, n))
    return t, np.sin(2 * np.pi * t / 1.7) + rng.normal(0, 0.3, n), rng.uniform(0.2, 0.5, n)


FREQS = 0.02 * (5 + np.arange(300))


def _powers(data, use_fft=True):
    from cuvarbase_amd import _lib
    from cuvarbase_amd.engine import LombBatch

    return LombBatch(data, [FREQS] * len(data), use_fft=use_fft, spread=_lib.SPREAD_FIXED)


@pytest.mark.parametrize("use_fft", [True, False])
@pytest.mark.parametrize("count", [1, 10, 13, 14, 15, 300])
def test_batch_sizes_around_the_limit(count, use_fft):
    data = [_curve(i) for i in range(count)]
    out = _powers(data, use_fft).run()
    for i in {0, count // 2, count - 1}:
        assert np.array_equal(out[i], _powers([data[i]], use_fft).run()[0])
        assert np.max(np.abs(out[i] - og.gls_direct(*data[i], FREQS))) < 1e-4


def test_wide_curve_alone_and_after_small_ones():
    wide, small = _curve(1, 17_000), [_curve(i) for i in range(3)]
    alone = _powers([wide]).run()[0]
    assert np.array_equal(_powers(small + [wide]).run()[3], alone)
    assert np.max(np.abs(alone - og.gls_direct(*wide, FREQS))) < 1e-4


def test_ring_reuse_after_streams_are_gone():
    from cuvarbase_amd._device import Stream

    data = [_curve(i % 50) for i in range(6000)]   # 1.5 MB of descriptors
    batch = _powers(data).allocate()
    first = None
    for _ in range(24):
        s = Stream()
        batch.upload(stream=s)
        batch.execute(stream=s)
        p = batch.download_async(stream=s)
        s.synchronize()
        first = p if first is None else first
        assert np.array_equal(p, first)
        del s
    for i in (0, 49, 50, 5999):
        assert np.array_equal(batch.split(first)[i], _powers([data[i]]).run()[0])
