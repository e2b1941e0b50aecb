"""The wave-parallel ordered sum (sb_debug_ordered_sum_device) against the one-at-a-time
sum: equal bits, over sums that stay in a binade, cross binades, cancel, hit rounding ties at
every step, or hold zeros, subnormals, infinities and NaN; sizes around a wave's 1,024 terms.
"""
import ctypes

import numpy as np
import pytest

import stormbird_amd as sb

pytestmark = pytest.mark.gpu

_dp = ctypes.POINTER(ctypes.c_double)


def gpu_sum(t, s0):
    L = sb.lib()
    L.sb_debug_ordered_sum_device.argtypes = [_dp, ctypes.c_size_t, ctypes.c_double, _dp]
    out = np.zeros(1)
    assert L.sb_debug_ordered_sum_device(t.ctypes.data_as(_dp), t.size, s0, out.ctypes.data_as(_dp)) == 0
    return out[0]


def terms(kind, n, rng):
    u = 2.0 ** -52
    if kind == "positive":
        return rng.uniform(0.0, 1.0, n), 0.0
    if kind == "signed":
        return rng.standard_normal(n), 0.0
    if kind == "decaying":
        return rng.standard_normal(n) / (1.0 + np.arange(n)) ** 2, 0.0
    if kind == "ties":  # multiples of half an ulp of the sum, which stays in [1, 2)
        return rng.integers(-3, 4, n) * (0.5 * u), 1.5
    if kind == "ties_up":  # always a tie: every step's rounding depends on the parity of the sum
        return np.full(n, 0.5 * u), 1.0 + u
    if kind == "ties_negative":
        return rng.integers(-3, 4, n) * (0.5 * u), -1.25
    if kind == "binade_edge":  # back and forth over a power of two
        return np.where(np.arange(n) % 2 == 0, 1.0, -1.0) * rng.uniform(0.9, 1.1, n) * 1e-3, 2.0
    if kind == "cancelling":
        a = rng.standard_normal(n) * 1e8
        a[1::2] = -a[:n // 2 * 2:2] + rng.standard_normal(n // 2)
        return a, 0.0
    if kind == "wide":
        return rng.standard_normal(n) * 10.0 ** rng.uniform(-30, 30, n), 0.0
    if kind == "mostly_zero":
        return np.where(rng.uniform(size=n) < 0.97, 0.0, rng.standard_normal(n)), 0.0
    if kind == "signed_zeros":
        return np.where(rng.uniform(size=n) < 0.5, 0.0, -0.0), 0.0
    if kind == "subnormal":
        return rng.integers(-50, 50, n) * 5e-324, 0.0
    if kind == "leaves_subnormal":
        return rng.integers(0, 1 << 50, n) * 5e-324, 0.0
    if kind == "infinite":
        t = rng.standard_normal(n)
        t[n // 2] = np.inf
        return t, 1.0
    if kind == "overflow":
        return rng.uniform(0.0, 1e308, n), 0.0
    t = rng.standard_normal(n)
    t[n // 3] = np.nan
    return t, 0.0


@pytest.mark.parametrize("kind", ["positive", "signed", "decaying", "ties", "ties_up", "ties_negative", "binade_edge",
                                  "cancelling", "wide", "mostly_zero", "signed_zeros", "subnormal",
                                  "leaves_subnormal", "infinite", "overflow", "nan"])
def test_ordered_sum_equals_the_sequential_sum(kind):
    rng = np.random.default_rng(11)
    for n in (1, 15, 16, 17, 63, 1023, 1024, 1025, 2048, 5000, 40000):
        t, s0 = terms(kind, n, rng)
        t = np.ascontiguousarray(t, dtype=np.float64)
        with np.errstate(over="ignore", invalid="ignore"):
            want = np.add.accumulate(np.concatenate([[s0], t]))[-1]  # one addition after another
        got = gpu_sum(t, s0)
        assert got == want or (np.isnan(got) and np.isnan(want)), (kind, n, got.hex(), float(want).hex())
        assert np.signbit(got) == np.signbit(want) or np.isnan(want), (kind, n)
