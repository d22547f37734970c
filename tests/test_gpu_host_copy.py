"""Factors read back through pinned slabs: sizes around a slab (512 KB), around
all slabs (2 MB) and past them; host-pointer calls with pageable and pinned
operands; and a fault in an array that is copied while it is being checked."""

import numpy as np
import pytest

import oracle
import tentaco_amd as tt
from helpers import REL_L2_TOL

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("R,dims", [(32, (4095, 4096, 4097)), (32, (16384, 16385, 1)),
                                    (32, (32769, 45000, 2)), (16, (8191, 8193, 1)), (64, (1, 2049, 16_385))])
def test_cpd_factor_round_trip(gpu, R, dims):
    """set_factor then factor gives the same bytes back, and weights."""
    rng = np.random.default_rng(R)
    n = 500
    coords = np.stack([rng.integers(0, d, n) for d in dims]).astype(np.int32)
    B = tt.Csf.from_coo(dims, coords, rng.uniform(-1, 1, n).astype(np.float32))
    c = tt.Cpd([[tt.DeviceCsf(b) for b in B.mode_csfs()]], R, seed=1)
    facs = [rng.uniform(-1, 1, (d, R)).astype(np.float32) for d in dims]
    for m, f in enumerate(facs):
        c.set_factor(0, m, f)
    for _ in range(2):
        for m, f in enumerate(facs):
            a, lam = c.factor(0, m)
            assert np.array_equal(a, f)
            assert np.array_equal(lam, np.ones(R, np.float32))


@pytest.mark.parametrize("pinned", [False, True])
def test_host_mttkrp_operands(gpu, pinned):
    rng = np.random.default_rng(11)
    dims, n, R = (3001, 40_009, 9001), 1_300_003, 32
    B = tt.Csf.from_coo(dims, np.stack([rng.integers(0, d, n) for d in dims]).astype(np.int32),
                        rng.uniform(-1, 1, n).astype(np.float32))
    facs = [rng.uniform(-1, 1, (d, R)).astype(np.float32) for d in dims[1:]]
    ref = oracle.mttkrp(B, facs, "taco", fp64=True)
    got = tt.mttkrp(B, [tt.pinned_copy(f) for f in facs] if pinned else facs)
    assert oracle.rel_l2(got, ref) <= REL_L2_TOL


@pytest.mark.parametrize("level", [1, 2])
@pytest.mark.parametrize("at", [0, -1])
def test_bad_coordinate_in_a_copied_level(gpu, level, at):
    """A coordinate outside its dimension is refused, the first one named."""
    rng = np.random.default_rng(12)
    dims, n = (2003, 5003, 7001), 1_200_000
    B = tt.Csf.from_coo(dims, np.stack([rng.integers(0, d, n) for d in dims]).astype(np.int32),
                        rng.uniform(-1, 1, n).astype(np.float32))
    crd = [np.array(x) for x in B.crd]
    crd[level][at] = dims[level]
    bad = tt.Csf(3, dims, B.pos, crd, B.vals, _owner=B._owner)
    where = crd[level].size - 1 if at else 0
    with pytest.raises(tt.TentacoError, match=rf"level {level} crd\[{where}\]={dims[level]}"):
        tt.DeviceCsf(bad)
    H = tt.DeviceCsf(B)
    assert H.nnz == B.nnz
    H.close()
