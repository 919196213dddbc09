"""Runs of one process share memory kept between them: results stay their own
while the caller holds them, whatever is run, dropped or deleted meanwhile.
Direct sums repeat bitwise, so their results are compared exactly."""
import gc

import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def _curve(seed, n=400):
    rng = np.random.default_rng(seed)
    t = np.sort(rng.uniform(0, 20.0, n))
    return t, np.sin(2 * np.pi * t / 1.7) + rng.normal(0, 0.3, n), rng.uniform(0.2, 0.5, n)


FREQS = 0.02 * (5 + np.arange(1500))


def _alone(d, **kw):
    from cuvarbase_amd.lombscargle import LombScargleAsyncProcess

    proc = LombScargleAsyncProcess(sigma=2, m=8)
    out = proc.run([d], freqs=FREQS, **kw)
    proc.finish()
    return np.array(out[0][1])


def test_results_survive_later_runs_and_the_process():
    from cuvarbase_amd.lombscargle import LombScargleAsyncProcess

    want = [_alone(_curve(i), use_fft=False) for i in range(6)]
    proc = LombScargleAsyncProcess(sigma=2, m=8)
    held = []
    for i in range(3):                      # enqueued together, one dropped before finish
        held.append(proc.run([_curve(i)], freqs=FREQS, use_fft=False))
    del held[1]
    proc.finish()
    for i in range(3, 6):                   # finished one by one, on reused memory
        held.append(proc.run([_curve(i)], freqs=FREQS, use_fft=False))
        proc.finish()
    del proc
    gc.collect()
    for i, r in zip((0, 2, 3, 4, 5), held):
        assert np.array_equal(r[0][1], want[i])


def test_sizes_and_methods_alternate_on_one_process():
    from cuvarbase_amd.lombscargle import LombScargleAsyncProcess

    proc = LombScargleAsyncProcess(sigma=2, m=8)
    for n in (50, 3000, 400, 17_000, 400):
        for use_fft in (True, False):
            d = _curve(n, n)
            out = proc.run([d], freqs=FREQS, use_fft=use_fft)
            proc.finish()
            assert np.max(np.abs(out[0][1] - _alone(d, use_fft=use_fft))) < 2e-5
