"""GPU parity of AUTO's slice-row kernels for short fibres and short slices:
slices summed a few to a wave (below 12 nonzeros a slice on average), one and
two waves a slice, at every rank layout; empty slices at the start, in runs
and at the end, slices longer than a batch of the kernel, and as many
nonzeros as one wave's share and one more."""

import numpy as np
import pytest

import oracle
import tentaco_amd as tt
from helpers import REL_L2_TOL

pytestmark = pytest.mark.gpu


def _slices(rng, sizes, d1, d2):
    rows = np.repeat(np.arange(sizes.size), sizes)
    n = rows.size
    coords = np.stack([rows, rng.integers(0, d1, n), rng.integers(0, d2, n)]).astype(np.int32)
    return tt.Csf.from_coo((sizes.size, d1, d2), coords, rng.uniform(-1, 1, n).astype(np.float32))


def _sizes(rng, case):
    if case == "mean5":
        s = rng.integers(1, 10, 4000)
        s[:70] = 0
        s[1000:1200] = 0
        s[-130:] = 0
        s[500] = 38  # past a batch, within 8 x the mean
    elif case == "mean11":
        s = rng.integers(4, 19, 3000)
        s[7] = 80
        s[-1] = 80
    elif case == "share":  # exactly 64 x the waves, then one more
        s = np.full(2048, 8)
    elif case == "share+1":
        s = np.full(2049, 8)
        s[-1] = 1
    elif case == "mean30":
        s = rng.integers(1, 60, 2500)
        s[rng.random(2500) < 0.1] = 0
    else:  # mean80
        s = rng.integers(40, 120, 2200)
    return s


@pytest.mark.parametrize("R", [2, 10, 16, 20, 32, 50, 64, 100, 128, 200])
@pytest.mark.parametrize("case", ["mean5", "mean11", "share", "share+1", "mean30", "mean80"])
def test_auto_short_slices(gpu, case, R):
    rng = np.random.default_rng(len(case) * 1000 + R)
    B = _slices(rng, _sizes(rng, case), 30000, 20000)
    assert B.nnz * 4 <= B.nodes(1) * 5
    facs = [rng.uniform(-1, 1, (d, R)).astype(np.float32) for d in B.dims[1:]]
    ref = oracle.mttkrp(B, facs, "taco", fp64=True)
    H = tt.DeviceCsf(B)
    assert tt.variants()[H.resolve(R)] == "sr_b256"
    fd = [tt.DeviceArray.from_numpy(f) for f in facs]
    A = tt.DeviceArray.from_numpy(np.full((B.dims[0], R), 3.0, np.float32))
    tt.ktimer_start()
    H.mttkrp(fd, A, R)
    name = tt.ktimer_stop()[2]
    if not case.startswith("mean30") and not case.startswith("mean80"):
        assert name == "slice_group_kernel"
    got = A.numpy()
    assert oracle.rel_l2(got, ref) <= REL_L2_TOL
    per_slice = np.diff(np.asarray(B.pos[2])[np.asarray(B.pos[1])])
    assert not got[per_slice == 0].any()
    H.mttkrp(fd, A, R)
    assert np.array_equal(A.numpy(), got)  # no atomics
    H.close()
