"""Q6_K rows on four waves: x read through LDS once per workgroup (rows of
33-48 blocks, 16-byte aligned x, where the row count suits it) gives the bits
of a wave's own loads (any other alignment), at the fewest and most blocks of
each layout, odd row counts (a last workgroup with one row of its two) and
several matrices.
"""
import ctypes

import numpy as np
import pytest

import fence_ops as F
from gpu_util import assert_bits_equal, dev, host, stream

pytestmark = pytest.mark.gpu


def blocks(rng, rows, nb):
    w = rng.integers(0, 256, (rows, nb, 210), dtype=np.uint8)
    d = (rng.random((rows, nb)) * 0.01).astype(np.float16)
    w[:, :, 208:210] = d[..., None].view(np.uint8).reshape(rows, nb, 2)
    return w


@pytest.mark.parametrize("nb", [13, 16, 33, 38, 48, 49, 64])
@pytest.mark.parametrize("rows", [8, 24, 3072, 4608, 3 * 8 * 257])  # the largest that share x, and more
def test_x_alignment_does_not_change_the_bits(nb, rows):
    rng = np.random.default_rng(nb * 1000 + rows)
    x = rng.standard_normal(256 * nb).astype(np.float16)
    w = dev(blocks(rng, rows, nb))
    ys = []
    for off in (0, 1, 4):  # 16-, 2- and 8-byte aligned
        xb = dev(np.concatenate([np.zeros(off, np.float16), x]))
        y = dev(np.full(rows, np.nan, np.float32))
        F.gemv_q6k(w.data_ptr(), xb.data_ptr() + 2 * off, y.data_ptr(), rows, 256 * nb, stream())
        ys.append(host(y))
    assert np.all(np.isfinite(ys[0]))
    assert_bits_equal(ys[0], ys[1], "2-byte aligned x")
    assert_bits_equal(ys[0], ys[2], "8-byte aligned x")
    # two matrices in one launch: the rows of each alone
    half = 8 * (rows // 16) or 8
    if half < rows:
        lib, vp = F.lib(), ctypes.c_void_p
        y = dev(np.full(rows, np.nan, np.float32))
        W = (vp * 2)(w.data_ptr(), w.data_ptr() + half * nb * 210)
        Y = (vp * 2)(y.data_ptr(), y.data_ptr() + 4 * half)
        xb = dev(x)
        assert lib.fence_gemv_q6k_multi(2, W, Y, None, (ctypes.c_int * 2)(half, rows - half), vp(xb.data_ptr()),
                                        256 * nb, vp(stream())) == 0
        assert_bits_equal(host(y), ys[0], "two matrices")


@pytest.mark.parametrize("nb", [16, 40, 48])  # odd row counts are staged where a row is a multiple of 8 blocks
@pytest.mark.parametrize("rows", [1, 3, 265, 511, 1535, 1537, 3071, 4607, 4609])
def test_odd_row_counts(nb, rows):
    rng = np.random.default_rng(nb * 1000 + rows)
    x = rng.standard_normal(256 * nb).astype(np.float16)
    w = dev(blocks(rng, rows, nb))
    ys = []
    for off in (0, 1):  # 16- and 2-byte aligned
        xb = dev(np.concatenate([np.zeros(off, np.float16), x]))
        y = dev(np.full(rows + 16, 12345.0, np.float32))
        F.gemv_q6k(w.data_ptr(), xb.data_ptr() + 2 * off, y.data_ptr(), rows, 256 * nb, stream())
        ys.append(host(y))
    assert np.all(np.isfinite(ys[0])) and np.all(ys[0][rows:] == 12345.0) and np.all(ys[1][rows:] == 12345.0)
    assert_bits_equal(ys[0], ys[1], "2-byte aligned x")
    first = rows // 2 | 1  # an odd first matrix: the second starts in the middle of a workgroup
    if first < rows:
        y = dev(np.full(rows + 16, 12345.0, np.float32))
        F.gemv_q6k_multi([w.data_ptr(), w.data_ptr() + first * nb * 210], dev(x).data_ptr(),
                         [y.data_ptr(), y.data_ptr() + 4 * first], [first, rows - first], 256 * nb, stream=stream())
        assert_bits_equal(host(y), ys[0], "two matrices")
