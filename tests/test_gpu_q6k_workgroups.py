"""Which Q6_K launches read x through LDS (8-wave workgroups of two rows) and
which let each wave load its own (4-wave workgroups of one), by the placement
records of the instrumented library: consecutive workgroups go to different
XCDs, the waves of one workgroup share theirs.

Two rows at a time must not cost more than they save: a CU whose share of the
rows is odd gets one row more.  Row counts on both sides of each bound, on 256
CUs that hold three such workgroups each.
"""
import ctypes
import os

import numpy as np
import pytest

import fence_ops as F
from gpu_util import dev, stream, torch_mod

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def clock():
    torch_mod()  # its HIP runtime is the one to bind to
    return ctypes.CDLL(os.path.join(os.path.dirname(F.LIB_PATH), "libfence_ops_waveclock.so"))


def workgroup_waves(clock, rows, nb, x_offset=0):
    torch = torch_mod()
    w = torch.zeros(rows * nb * 210, dtype=torch.uint8, device="cuda")
    x = dev(np.zeros(256 * nb + 8, np.float16))
    y = torch.empty(rows, device="cuda")
    torch.cuda.synchronize()
    vp = ctypes.c_void_p
    assert clock.fence_wave_clock_clear() == 0
    assert clock.fence_gemv_q6k(vp(w.data_ptr()), vp(x.data_ptr() + x_offset), vp(y.data_ptr()), rows, 256 * nb,
                                vp(stream())) == 0
    rec = np.zeros((1 << 16, 4), np.uint64)
    assert clock.fence_wave_clock_read(vp(rec.ctypes.data), ctypes.c_int64(len(rec))) == 0
    n = int(np.count_nonzero(rec[:, 0]))
    assert n >= 64 and n % 8 == 0 and np.all(rec[:n, 0] != 0)
    xcc = (rec[:n, 2] >> np.uint64(32)).astype(np.int64) & 15
    return 8 if np.array_equal(xcc[0::8], xcc[4::8]) else 4


@pytest.mark.parametrize("nb", [33, 40, 48])
@pytest.mark.parametrize("rows,waves", [
    (128, 4), (256, 4), (264, 8), (512, 8), (520, 4), (768, 4), (776, 8), (1280, 4), (1536, 8),  # the first round
    (1792, 8), (1808, 8), (2056, 4), (2304, 4), (2560, 8), (2816, 4), (3072, 8),  # the second
    (3328, 8), (3840, 8), (3856, 8), (4104, 4), (4352, 4), (4608, 8), (4624, 4), (6144, 4)])  # the third, and past it
def test_three_pass_rows_share_x_where_it_pays(clock, nb, rows, waves):
    assert torch_mod().cuda.get_device_properties(0).multi_processor_count == 256
    assert workgroup_waves(clock, rows, nb) == waves


@pytest.mark.parametrize("rows,nb,offset", [(512, 13, 0), (1536, 16, 0), (2816, 16, 0), (1536, 49, 0), (1536, 64, 0),
                                            (1536, 33, 2), (1536, 48, 8)])
def test_other_rows_and_alignments_load_their_own_x(clock, rows, nb, offset):
    assert workgroup_waves(clock, rows, nb, offset) == 4
