"""Host side of the batched runs: the block pool, centring and significances of
many curves at a time (no device calls)."""
import ctypes as C

import numpy as np
import pytest

from cuvarbase_amd import _device, lombscargle as ls, utils


class _Allocator:
    """Stands for the library's allocation entry points."""

    def __init__(self):
        self.live, self.made, self.keep = {}, 0, []

    def call(self, name, *args):
        if name in ("gls_malloc", "gls_host_alloc"):
            buf = C.create_string_buffer(args[1].value)
            addr = C.addressof(buf)
            args[0]._obj.value = addr
            self.live[addr] = buf
            self.made += 1
        else:
            self.live.pop(args[0].value)


@pytest.fixture
def allocator(monkeypatch):
    a = _Allocator()
    monkeypatch.setattr(_device._lib, "call", a.call)
    monkeypatch.setattr(_device._lib, "_lib", a)
    return a


@pytest.mark.parametrize("kind", ["malloc", "host_alloc"])
def test_pool_reuses_bounds_and_gives_back(allocator, kind):
    pool = _device.BufferPool(device_limit=100_000, host_limit=100_000)
    p, cap = pool.take(kind, 5000)
    assert cap >= 5000
    pool.give(kind, p, cap)
    assert pool.take(kind, cap) == (p, cap) and allocator.made == 1
    q = [pool.take(kind, 40_000) for _ in range(3)]
    for ptr, c in q:
        pool.give(kind, ptr, c)       # two fit under the limit
    assert len(allocator.live) == 3   # p (taken) and two kept
    big, c = pool.take(kind, 200_000)
    pool.give(kind, big, c)           # above the limit: freed at once
    assert big not in allocator.live
    pool.close()
    assert list(allocator.live) == [p]
    pool.give(kind, p, cap)           # after close: freed
    assert not allocator.live


def test_pool_size_classes():
    for n in (1, 4096, 4097, 5000, 65536, 65537, 10**6 + 7):
        cap = _device.BufferPool._class(n)
        assert max(n, 4096) <= cap <= max(4096, 1.25 * n + 1)
        assert _device.BufferPool._class(cap) == cap


def _curves(count, seed):
    rng = np.random.default_rng(seed)
    return [(np.sort(rng.uniform(0, 90, n)), rng.normal(15, 1, n), rng.uniform(0.1, 0.3, n))
            for n in rng.integers(5, 400, count)]


def test_centring_many_matches_one_by_one():
    data = _curves(40, 1)
    data[3][1][2] = np.nan
    data[5][0][0] = np.nan
    before = [tuple(c.copy() for c in d) for d in data]
    out = utils.centre_light_curves(data)
    for got, want, was, d in zip(out, utils.normalize_light_curves(data), before, data):
        for a, b in zip(got, want):
            np.testing.assert_allclose(a, b, rtol=0, atol=1e-12)
        for a, b in zip(was, d):
            np.testing.assert_array_equal(a, b)
    # lists, other types and ragged columns take the curve-by-curve way
    out = utils.centre_light_curves([([1, 2, 6], [2, 2, 5], [1, 1, 1])])
    np.testing.assert_allclose(out[0][0], [-2, -1, 3])
    assert utils.centre_light_curves([]) == []


def test_significances_match_one_by_one():
    data = _curves(30, 2)
    z = np.random.default_rng(3).uniform(0.02, 0.95, len(data))
    z[7] = np.nan
    got = ls._significances(data, z, 40.0)
    for c, p, s in zip(data, z, got):
        if np.isnan(p):
            assert np.isnan(s)
        else:
            assert abs(s - (1 - ls.fap_baluev(c[0], c[2], np.array([p]), 40.0)[0])) < 1e-12
    assert len(ls._significances([], np.zeros(0), 1.0)) == 0
