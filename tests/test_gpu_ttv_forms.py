"""Which form of the TTV unit kernel runs. The one by whole fibres sums exact
products in FP64, so every entry is the 64-bit result rounded once; the one with
a window of c sums long fibres in FP32. Up to 2048 nonzeros a fibre and 2048
units of 512 the first is taken, beyond either the second."""

import numpy as np
import pytest

import oracle
import tentaco_amd as tt
from helpers import REL_L2_TOL

pytestmark = pytest.mark.gpu


def _run(sizes, bands, seed):
    rng = np.random.default_rng(seed)
    fib = np.repeat(np.arange(sizes.size), sizes)
    leaf = np.concatenate([rng.choice(5000, n, replace=False) for n in sizes])
    B = tt.Csf.from_coo((sizes.size, 5000), np.stack([fib, leaf]).astype(np.int32),
                        rng.uniform(-1, 1, fib.size).astype(np.float32))
    c = rng.uniform(-1, 1, 5000).astype(np.float32)
    H = tt.DeviceCsf(B)
    H.set_ttv_bands(bands)
    y = tt.DeviceArray.empty((sizes.size,))
    tt.ktimer_start()
    H.ttv(tt.DeviceArray.from_numpy(c), y)
    assert tt.ktimer_stop()[2] == "ttv_unit_kernel"
    got = y.numpy()
    H.close()
    # (an oracle of its own: the 64-bit sum of the exact products)
    ref = np.add.reduceat(B.vals.astype(np.float64) * c[B.crd[1]], B.pos[1][:-1])
    assert oracle.rel_l2(got, ref) <= REL_L2_TOL
    return np.array_equal(got, ref.astype(np.float32))


@pytest.mark.parametrize("sizes,whole", [([2048] * 40 + [7, 300] * 50, True), ([2048] * 40 + [2049] + [7, 300] * 50, False),
                                         ([512] * 2048, True), ([512] * 2048 + [1], False)])
def test_form_by_sizes(gpu, sizes, whole):
    sizes = np.array(sizes)
    assert _run(sizes, 0, 1) == whole
    assert not _run(sizes, 1, 1)  # the window, by request
