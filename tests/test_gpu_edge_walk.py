"""The edge walk where a wave's chunk of 64 nonzeros holds many slices, one, or
parts of several: slices of one to five nonzeros, of exactly 64 and one more
and less, slices of several chunks among them, and empty root nodes at the
start, in runs and at the end; on the first call of a handle, on its second,
after a reserve, and by the call that allocates nothing (whose waves search
for their starts); explicit tiles and the sized one."""

import ctypes

import numpy as np
import pytest

import oracle
import tentaco_amd as tt
from helpers import REL_L2_TOL

pytestmark = pytest.mark.gpu


def _sizes(rng, case):
    if case == "ones":
        return np.ones(5000, int)
    if case == "few":
        return rng.integers(0, 6, 4000)
    if case == "chunks":
        return np.array([64] * 20 + [63, 65, 1, 128, 64, 1, 1, 62, 64, 192] + [32] * 40)
    if case == "gaps":
        s = rng.integers(1, 9, 3000)
        s[:200] = 0
        s[900:1300] = 0
        s[-150:] = 0
        return s
    s = rng.integers(1, 4, 2500)  # "long": long slices among short ones
    s[[0, 700, 701, 2499]] = [5000, 900, 3000, 2100]
    return s


@pytest.mark.parametrize("order,R", [(2, 32), (3, 16), (3, 32), (3, 50), (3, 128), (4, 64), (5, 3), (5, 20), (5, 32)])
@pytest.mark.parametrize("case", ["ones", "few", "chunks", "gaps", "long"])
def test_edge_walk_slices(gpu, case, order, R):
    rng = np.random.default_rng(order * 1000 + R)
    sizes = _sizes(rng, case)
    dims = (sizes.size,) + (40, 30, 50)[: order - 2] + (20_000,)
    rows = np.repeat(np.arange(sizes.size), sizes)
    coords = np.stack([rows, *[rng.integers(0, d, rows.size) for d in dims[1:]]]).astype(np.int32)
    B = tt.Csf.from_coo(dims, coords, rng.uniform(-1, 1, rows.size).astype(np.float32))
    facs = [rng.uniform(-1, 1, (d, R)).astype(np.float32) for d in dims[1:]]
    ref = oracle.mttkrp(B, facs, "taco", fp64=True)
    fd = [tt.DeviceArray.from_numpy(f) for f in facs]
    names = tt.variants()
    A = tt.DeviceArray.empty((dims[0], R))
    for v in [names.index(n) for n in ("ep_b256_g16", "ep_b128_g4", "es_b256_g8", "ep_b512_g64")] + [tt.VARIANT_AUTO]:
        if v >= 0 and not tt.variant_fits(order, R, v):
            continue
        H = tt.DeviceCsf(B)
        reserved = tt.DeviceCsf(B)
        reserved.reserve(R, v)
        for what, h in (("first", H), ("second", H), ("reserved", reserved)):
            A.upload(np.full((dims[0], R), 7.0, np.float32))
            h.mttkrp(fd, A, R, v)
            assert oracle.rel_l2(A.numpy(), ref) <= REL_L2_TOL, (v, what)
        arr = (ctypes.c_void_p * len(fd))(*[f.ptr for f in fd])
        A.upload(np.full((dims[0], R), 7.0, np.float32))
        bare = tt.DeviceCsf(B)
        assert tt.lib().tentaco_mttkrp_dev_noalloc(bare.h, R, arr, A.ptr, dims[0], v, None) == tt.OK
        assert oracle.rel_l2(A.numpy(), ref) <= REL_L2_TOL, (v, "noalloc")
        for h in (H, reserved, bare):
            h.close()


@pytest.mark.parametrize("order,R", [(2, 32), (3, 16), (3, 32), (3, 50), (4, 64), (4, 3), (5, 100), (5, 200)])
def test_edge_walk_shared_rows(gpu, order, R):
    """More than 2048 workgroups of an edge-parallel tile add to the rows that
    they share in FP64: slices over many workgroups, over two, starting with a
    workgroup and ending with one, and shorter than one; rows without a root
    node and rows past the tensor's are zeroed, on every call and replay-like
    repetition, also when the calls alternate with another rank's."""
    rng = np.random.default_rng(R)
    nb = 128 * 4 // max(1, next(p for p in (4, 8, 16, 32, 64, 128, 256) if p >= R) // 4) if R > 3 else 128 * 4
    nb = max(nb, 32)
    sizes = np.concatenate([[30 * nb, nb, nb, nb // 2, nb // 2, 2 * nb + 5, nb - 5], rng.integers(0, 3, 700),
                            [nb] * 900, rng.integers(1, 3 * nb, 700), [0] * 40, [300 * nb], [0] * 33])
    dims = (sizes.size + 10,) + (40, 30, 50)[: order - 2] + (60_000,)
    rows = np.repeat(np.arange(sizes.size), sizes)
    coords = np.stack([rows, *[rng.integers(0, d, rows.size) for d in dims[1:]]]).astype(np.int32)
    B = tt.Csf.from_coo(dims, coords, rng.uniform(-1, 1, rows.size).astype(np.float32))
    more = dims[0] + 45
    facs = [rng.uniform(-1, 1, (d, R)).astype(np.float32) for d in dims[1:]]
    ref = np.zeros((more, R))
    ref[: dims[0]] = oracle.mttkrp(B, facs, "taco", fp64=True)
    fd = [tt.DeviceArray.from_numpy(f) for f in facs]
    half = [tt.DeviceArray.from_numpy(np.ascontiguousarray(f[:, :1])) for f in facs]
    A, A1 = tt.DeviceArray.empty((more, R)), tt.DeviceArray.empty((dims[0], 1))
    v = tt.variants().index("ep_b128_g4")
    if not tt.variant_fits(order, R, v):
        pytest.skip("tile over the limit")
    H = tt.DeviceCsf(B)
    for rep in range(3):
        A.upload(np.full((more, R), 7.0 + rep, np.float32))
        H.mttkrp(fd, A, R, v, a_rows=more)
        got = A.numpy()
        # FP32 products and sums of a workgroup, FP64 across workgroups
        assert oracle.rel_l2(got, ref) <= REL_L2_TOL, rep
        assert np.all(got[np.all(ref == 0, axis=1)] == 0), rep
        H.mttkrp(half, A1, 1, v)
        assert oracle.rel_l2(A1.numpy(), oracle.mttkrp(B, [f[:, :1].copy() for f in facs], "taco", fp64=True)) <= REL_L2_TOL
    H.close()
