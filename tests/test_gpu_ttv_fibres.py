"""GPU parity of the TTV kernel that sums whole fibres by the wave (few
nonzeros, no long or empty fibre), against the oracle and against the window
kernel (set_ttv_bands(1)): nonzeros around the 512 of a unit and the 2048 of a
workgroup, fibres that start, end and cross at unit edges, fibres as long as
several units, and one nonzero past the length the kernel takes."""

import numpy as np
import pytest

import oracle
import tentaco_amd as tt
from helpers import REL_L2_TOL

pytestmark = pytest.mark.gpu

CASES = {
    "one": [1],
    "ones": [1] * 3000,
    "unit": [512],
    "unit+1": [512, 1],
    "edges": [511, 1, 1, 511, 513, 511, 64, 63, 65, 256, 64],
    "workgroup": [2048],
    "workgroup+1": [2047, 2],
    "long": [3, 2048, 1, 1500, 700, 2048, 5],
    "past": [3, 2049, 1, 1500, 7],
    "mixed": None,
}


@pytest.mark.parametrize("order", [2, 3, 4])
@pytest.mark.parametrize("case", list(CASES))
def test_ttv_whole_fibres(gpu, case, order):
    rng = np.random.default_rng(len(case) + order)
    sizes = CASES[case]
    if sizes is None:
        sizes = np.minimum(2048, (rng.pareto(0.8, 6000) * 3 + 1).astype(int))
    sizes = np.asarray(sizes)
    nf, kdim = sizes.size, 5000
    fib = np.repeat(np.arange(nf), sizes)
    leaf = np.concatenate([rng.choice(kdim, s, replace=False) for s in sizes])
    lead = {2: [fib], 3: [fib // 7, fib % 7], 4: [fib // 15, fib % 15 // 5, fib % 5]}[order]
    dims = tuple(int(x.max()) + 1 for x in lead) + (kdim,)
    coords = np.stack([*lead, leaf]).astype(np.int32)
    B = tt.Csf.from_coo(dims, coords, rng.uniform(-1, 1, fib.size).astype(np.float32))
    assert B.nodes(order - 2) == nf
    c = rng.uniform(-1, 1, kdim).astype(np.float32)
    ref = oracle.ttv(B, c, "taco", fp64=True)
    cd = tt.DeviceArray.from_numpy(c)
    got = []
    for bands in (0, 1, 0):
        H = tt.DeviceCsf(B)
        H.set_ttv_bands(bands)
        y = tt.DeviceArray.from_numpy(np.full(nf, np.nan, np.float32))
        H.ttv(cd, y)
        got.append(y.numpy())
        assert H.ttv_layout() == (1, 0)
        # an entry is a sum of at most 2049 products below 1 in magnitude
        assert oracle.rel_l2(got[-1], ref) <= REL_L2_TOL
        H.close()
    assert np.array_equal(got[0], got[2])
