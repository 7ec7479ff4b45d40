"""Rows split over 1 .. 16 waves: the cross-wave combination of a row's sum
(RMSNorm, softmax) and maximum (softmax) at every wave count, with the row's
largest value and a NaN placed in the first and in the last wave.

The sum over waves has a fixed order, so its result is compared with the same
order in float32: lane partials, a fixed 64-lane tree, then the waves from the
first to the last.  A power-of-two row makes every operation exact, so the
RMSNorm bound is the rounding of one division, one rsqrt (2 ulp) and two
products: 6 * 2^-24 relative.  Softmax of a row with one dominant value is
bounded by its n exponentials at 1e-6 each.
"""
import numpy as np
import pytest

import fence_ops as F
from gpu_util import dev, host, stream

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("waves", list(range(1, 17)))
def test_rms_norm_at_every_wave_count(waves):
    n = 4 * 64 * waves  # one row: one float4 per lane
    x = np.where(np.arange(n) // 256 % 2 == 0, 2.0, 0.5).astype(np.float32)
    w = np.ones(n, np.float32)
    out = dev(np.zeros(n, np.float32))
    F.rms_norm(out.data_ptr(), dev(x).data_ptr(), dev(w).data_ptr(), n, 0.0, stream())
    ref = x / np.sqrt(np.mean(x.astype(np.float64) ** 2))
    assert np.max(np.abs(host(out) - ref) / np.abs(ref)) <= 6 * 2.0 ** -24
    for at in (0, n - 1):
        y = x.copy()
        y[at] = np.nan
        F.rms_norm(out.data_ptr(), dev(y).data_ptr(), dev(w).data_ptr(), n, 0.0, stream())
        assert np.all(np.isnan(host(out)))
        y[at] = np.inf
        F.rms_norm(out.data_ptr(), dev(y).data_ptr(), dev(w).data_ptr(), n, 0.0, stream())
        got = host(out)  # inf * rsqrt(inf) = nan at the infinite value, 0 elsewhere
        assert np.isnan(got[at]) and np.count_nonzero(got != 0) == 1


@pytest.mark.parametrize("waves", list(range(1, 17)))
def test_softmax_at_every_wave_count(waves):
    n = 4 * 64 * waves
    for at in (0, n - 1):
        x = np.full(n, -np.inf, np.float32)
        x[at], x[n // 2] = 3.0, 2.0
        d = dev(x)
        F.softmax(d.data_ptr(), n, stream())
        e = np.exp(x.astype(np.float64) - 3.0)
        assert np.max(np.abs(host(d) - e / e.sum())) <= 2e-6
        d = dev(np.full(n, -np.inf, np.float32))  # a fully masked row: 0 / 0, as the formula gives
        F.softmax(d.data_ptr(), n, stream())
        assert np.all(np.isnan(host(d)))
        x[at] = np.nan  # the maximum passes it by, the sum does not
        d = dev(x)
        F.softmax(d.data_ptr(), n, stream())
        assert np.all(np.isnan(host(d)))
