"""GPU parity of the rank layouts at their edges: ranks 1-3 (scalar columns),
and every runtime-rank layout at its smallest, an odd and its largest rank
(4..16, 17..32, 33..64, 65..128, 129..256 columns), for one tile of each
MTTKRP family and for the one-CSF modes."""

import numpy as np
import pytest

import oracle
import tentaco_amd as tt
from helpers import REL_L2_TOL, factors_for, skewed_coo

pytestmark = pytest.mark.gpu

RANKS = [1, 2, 3, 4, 5, 15, 17, 18, 31, 33, 50, 63, 65, 100, 127, 129, 254, 255, 256]
TILES = ["es_b256_g16", "ep_b256_g16", "ep_b512_g64", "sr_b256"]


@pytest.mark.parametrize("order", [2, 3, 4, 5])
@pytest.mark.parametrize("R", RANKS)
def test_rank_layouts(gpu, order, R):
    rng = np.random.default_rng(1000 * order + R)
    dims = {2: (60, 500), 3: (45, 60, 70), 4: (31, 20, 25, 30), 5: (17, 9, 10, 11, 12)}[order]
    coords, vals = skewed_coo(rng, dims, 5000, hot_slice=3)
    B = tt.Csf.from_coo(dims, coords, vals)
    facs = factors_for(rng, B, R)
    ref = oracle.mttkrp(B, facs, "taco", fp64=True)
    H = tt.DeviceCsf(B)
    fd = [tt.DeviceArray.from_numpy(f) for f in facs]
    names = tt.variants()
    for name in TILES:
        v = names.index(name)
        if not tt.variant_fits(order, R, v):
            continue
        A = tt.DeviceArray.from_numpy(np.full((dims[0], R), np.nan, np.float32))
        H.mttkrp(fd, A, R, v)
        assert oracle.rel_l2(A.numpy(), ref) <= REL_L2_TOL, (name, order, R)
    # the one-CSF modes: the mode at the leaf level, and at level 1
    root = rng.uniform(-1, 1, (dims[0], R)).astype(np.float32)
    full = [root] + facs
    fdl = [tt.DeviceArray.from_numpy(f) for f in full]
    for level in sorted({1, order - 1}):
        Bm = B.reorder([level] + [k for k in range(order) if k != level])
        refl = oracle.mttkrp(Bm, [full[k] for k in range(order) if k != level], "taco", fp64=True)
        out = tt.DeviceArray.from_numpy(np.full((dims[level], R), np.nan, np.float32))
        H.mttkrp_level(level, fdl, out, R)
        assert oracle.rel_l2(out.numpy(), refl) <= REL_L2_TOL, (level, order, R)
    H.close()
