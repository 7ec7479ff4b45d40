"""Rows split over 1 .. 16 waves: the cross-wave combination of a row's sum
(RMSNorm, softmax) and maximum (softmax) at every wave count.

One float4 per lane, so a row of 256 w floats takes w waves.  RMSNorm folds
the waves' sums at two waves and more; softmax has kernels of its own for up
to 256 lanes (w <= 4, with 3 rounded up to 4) and folds sums and maxima from
five waves on.

Values: rows of powers of two, where every operation is exact in any order,
against float64.  The RMSNorm bound is the rounding of one division, one rsqrt
(2 ulp) and two products: 6 * 2^-24 relative.  Softmax of a row with one
dominant value is bounded by its n exponentials at 1e-6 each.

Order: the sum runs over the waves from the first to the last.  With 2^24 in
the first wave and 1 in each later one every addition rounds back to 2^24,
with 2^24 in the last wave the ones add up before it; either total is also
that of a row with one nonzero wave, whose result no order can change, and
the two must agree bit for bit.

Maximum: a value 198 above the rest, in each wave in turn, makes the row
exactly one-hot; were it lost, the others' exponentials would not be.
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


def normed(x):
    out = dev(np.zeros(len(x), np.float32))
    F.rms_norm(out.data_ptr(), dev(x).data_ptr(), dev(np.ones(len(x), np.float32)).data_ptr(), len(x), 0.0, stream())
    return host(out)


@pytest.mark.parametrize("waves", list(range(2, 17)))
def test_waves_are_added_first_to_last(waves):
    n = 4 * 64 * waves
    for big in (0, waves - 1):
        x = np.zeros(n, np.float32)
        x[0::256] = 1.0  # each wave's sum
        x[256 * big] = 4096.0
        total = np.float32(0.0)
        for w in range(waves):
            total = np.float32(total + x[256 * w] * x[256 * w])
        one = np.zeros(n, np.float32)  # the same total from the big wave alone
        one[256 * big] = 4096.0
        rest = int(total) - 2 ** 24
        assert rest in (0, 2, 4, 6, 8, 10, 12, 14, 16)
        at = 256 * big + 128  # in the wave's upper half, which is summed before the lower one joins it
        while rest:  # small squares that add up to the rest, one per lane
            r = int(np.sqrt(rest))
            one[at] = r
            rest -= r * r
            at += 4
        assert normed(x)[256 * big] == normed(one)[256 * big]


@pytest.mark.parametrize("waves", list(range(1, 17)))
def test_softmax_maximum_in_each_wave(waves):
    n = 4 * 64 * waves
    for w in range(waves):
        for at in (256 * w, 256 * w + 255):
            x = np.full(n, 2.0, np.float32)
            x[at] = 200.0
            d = dev(x)
            F.softmax(d.data_ptr(), n, stream())
            want = np.zeros(n, np.float32)
            want[at] = 1.0
            assert np.array_equal(host(d), want)
