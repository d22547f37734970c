"""Sums of many nonzeros in FP32 take them in levels. One nonzero of 2^24 and
many of 1, all factors 1: a sum that adds them to the large one one by one
loses every 1 (2^24 + 1 rounds to 2^24), one that adds partial sums keeps them."""

import numpy as np
import pytest

import tentaco_amd as tt

pytestmark = pytest.mark.gpu

BIG = 2.0 ** 24


def _ones(dims, R):
    return [tt.DeviceArray.from_numpy(np.ones((d, R), np.float32)) for d in dims]


def _groups(R):
    """Row groups of a wave (lanes that share a factor row)."""
    p = next(p for p in (16, 32, 64, 128, 256) if p >= max(R, 16))
    return 16 if R < 4 else 64 // min(16, p // 4)


@pytest.mark.parametrize("order,R", [(3, 16), (3, 32), (3, 50), (4, 64), (4, 20), (5, 32), (5, 128)])
def test_inner_mode_row(gpu, order, R):
    # one output row of 8192 level N-2 nodes with 8 nonzeros each
    n = np.arange(65536)
    lead = [n // 8] if order == 3 else [n // 64, n // 8 % 8] if order == 4 else [n // 512, n // 64 % 8, n // 8 % 8]
    coords = np.stack([lead[0], np.zeros_like(n), *lead[1:], n % 8]).astype(np.int32)
    dims = tuple(int(c.max()) + 1 for c in coords)
    vals = np.ones(n.size, np.float32)
    vals[0] = BIG
    H = tt.DeviceCsf(tt.Csf.from_coo(dims, coords, vals))
    A = tt.DeviceArray.empty((1, R))
    H.mttkrp_level(1, _ones(dims, R), A, R)
    # what is added to the large one alone: its chunk's 64 / groups nonzeros of
    # its row group; every other partial sum below 2^24 is exact, and adding an
    # odd one to a total past 2^24 rounds by 1, at most once a wave of 8
    got = A.numpy().astype(np.float64)
    assert np.max(np.abs(got - (BIG + n.size - 1))) <= 64 // _groups(R) + 9
    H.close()


@pytest.mark.parametrize("order,R", [(2, 32), (3, 2), (3, 16), (3, 32), (3, 50), (3, 128), (4, 64), (4, 20), (5, 32), (5, 256)])
def test_edge_walk_run(gpu, order, R):
    # two slices of 8192 nonzeros, 8 to a fibre
    n = np.arange(16384)
    lead = {2: [n // 8192], 3: [n // 8192, n // 8 % 1024], 4: [n // 8192, n // 64 % 128, n // 8 % 8],
            5: [n // 8192, n // 512 % 16, n // 64 % 8, n // 8 % 8]}[order]
    coords = np.stack([*lead, n % 8192 if order == 2 else n % 8]).astype(np.int32)
    dims = tuple(int(c.max()) + 1 for c in coords)
    vals = np.ones(n.size, np.float32)
    vals[[0, 8192]] = BIG
    names = tt.variants()
    H = tt.DeviceCsf(tt.Csf.from_coo(dims, coords, vals))
    A = tt.DeviceArray.empty((2, R))
    fd = _ones(dims[1:], R)
    ran = 0
    for v in ("ep_b512_g64", "ep_b256_g64", "ep_b128_g32", "es_b512_g64", "es_b128_g64"):
        if not tt.variant_fits(order, R, names.index(v)):
            continue
        ran += 1
        H.mttkrp(fd, A, R, names.index(v))
        # the large one's chunk of its row group, then a rounding by 1 for every
        # odd total that a wave, a workgroup or (FP32 atomics, at most 32
        # workgroups a slice) the output row adds to 2^24
        got = A.numpy().astype(np.float64)
        assert np.max(np.abs(got - (BIG + 8191))) <= 64 // _groups(R) + 6, v
    assert ran >= 3
    H.close()


@pytest.mark.parametrize("R", [2, 16, 20, 32, 50, 100, 128, 200])
def test_short_slices(gpu, R):
    # slices of 6 on average, 40 at most, one nonzero a fibre (the AUTO kernel of
    # short slices); every slice starts with the large one
    rng = np.random.default_rng(R)
    sizes = np.where(rng.random(5000) < 0.02, 40, rng.integers(1, 12, 5000))
    row = np.repeat(np.arange(sizes.size), sizes)
    at = np.arange(row.size) - np.repeat(np.cumsum(sizes) - sizes, sizes)
    coords = np.stack([row, at, rng.integers(0, 9, row.size)]).astype(np.int32)
    vals = np.where(at == 0, BIG, 1.0).astype(np.float32)
    dims = tuple(int(c.max()) + 1 for c in coords)
    H = tt.DeviceCsf(tt.Csf.from_coo(dims, coords, vals))
    A = tt.DeviceArray.empty((dims[0], R))
    tt.ktimer_start()
    H.mttkrp(_ones(dims[1:], R), A, R, tt.VARIANT_AUTO)
    assert tt.ktimer_stop()[2] == "slice_group_kernel"
    # FP64 sums: one rounding
    ref = (BIG + sizes - 1).astype(np.float32)
    assert np.array_equal(A.numpy(), np.repeat(ref[:, None], R, axis=1))
    H.close()


@pytest.mark.parametrize("order,R", [(2, 32), (3, 16), (3, 32), (3, 50), (4, 20), (5, 32)])
def test_edge_walk_many_slices(gpu, order, R):
    # chunks of several slices, whose sums are FP64; every slice starts with the
    # large one, none crosses a workgroup's first or last nonzero but the two of
    # its ends
    rng = np.random.default_rng(R)
    sizes = rng.integers(1, 6, 400)
    row = np.repeat(np.arange(sizes.size), sizes)
    at = np.arange(row.size) - np.repeat(np.cumsum(sizes) - sizes, sizes)
    coords = np.stack([row, *[at] * (order - 1)]).astype(np.int32)
    dims = tuple(int(c.max()) + 1 for c in coords)
    vals = np.where(at == 0, BIG, 1.0).astype(np.float32)
    names = tt.variants()
    H = tt.DeviceCsf(tt.Csf.from_coo(dims, coords, vals))
    A = tt.DeviceArray.empty((dims[0], R))
    fd = _ones(dims[1:], R)
    ref = (BIG + sizes - 1)[:, None]
    for v in ("ep_b512_g64", "ep_b256_g64", "es_b512_g64"):
        if not tt.variant_fits(order, R, names.index(v)):
            continue
        H.mttkrp(fd, A, R, names.index(v))
        got = A.numpy().astype(np.float64)
        # a slice inside a batch of products is its FP64 sum rounded once; one cut
        # by a batch, chunk, run or workgroup adds parts in FP32, and may lose its 1s
        cut = np.abs(got - ref).max(axis=1)
        assert np.max(cut) <= 5 and np.mean(cut > 1) <= 0.2, v
    H.close()
