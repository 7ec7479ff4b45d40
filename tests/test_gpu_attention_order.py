"""The order attention adds its positions in, bit for bit.

With q = 0 every score is 0, every weight exactly 1 and the sum of weights
the number of positions, a power of two here, so an output is the sum of the
attended V values in the kernel's order, divided exactly: each of the 16
position groups adds its own positions (t % 16) in order, and the groups are
added in order from 0.  V spans 2^-14 .. 2^15, so another order rounds
differently.  No score_buf: one split, and nothing after the sum.
"""
import numpy as np
import pytest

import fence_ops as F
from gpu_util import assert_bits_equal, dev, host, stream

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("seq", [16, 64, 256])
@pytest.mark.parametrize("n_q,n_kv", [(32, 8), (8, 8), (12, 4)])
def test_positions_are_added_in_group_order(n_q, n_kv, seq):
    hd = 128
    rng = np.random.default_rng(100 * n_q + seq)
    v = np.ldexp(rng.uniform(-1, 1, (seq, n_kv * hd)), rng.integers(-14, 16, (seq, n_kv * hd))).astype(np.float16)
    k = rng.standard_normal((seq, n_kv * hd)).astype(np.float16)
    out = dev(np.full(n_q * hd, np.nan, np.float32))
    F.gqa_attention(out.data_ptr(), dev(np.zeros(n_q * hd, np.float32)).data_ptr(), dev(k).data_ptr(),
                    dev(v).data_ptr(), hd, n_q, n_kv, seq, seq, None, stream())
    groups = np.zeros((16, n_kv * hd), np.float32)
    for t in range(seq):
        groups[t % 16] += v[t].astype(np.float32)
    acc = np.zeros(n_kv * hd, np.float32)
    for g in groups:
        acc = acc + g
    ref = (acc / np.float32(seq)).reshape(n_kv, hd)
    assert_bits_equal(host(out).reshape(n_q, hd), ref[np.arange(n_q) // (n_q // n_kv)], f"{seq} positions")
