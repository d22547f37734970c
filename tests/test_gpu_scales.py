"""Products of four and five rows whose partial products leave FP32's range
while value times leaf row times the rows one by one does not: small factors
under large values, large ones under small values, rows of both kinds and of
ordinary size in one tensor, and factors with many zeros."""

import numpy as np
import pytest

import tentaco_amd as tt

pytestmark = pytest.mark.gpu

# All terms of an entry are positive and pass at most about 80 roundings of
# 2^-24 one after another (a lane group's run of nonzeros, the wave's and the
# workgroup's sums): 4.8e-6.
ROW_TOL = 1e-5


def _case(rng, dims, R, mode, sizes, kind):
    """Entries with sizes[j] of them at coordinate j of `mode`. Rows of the lower
    half of every other factor's coordinates have size 1, of the upper half the
    kind's; an output row uses one half only, with values that fit it."""
    order = len(dims)
    rows = np.repeat(np.arange(sizes.size), sizes)
    upper = rows % 2 == 1 if kind == "mixed" else np.full(rows.size, kind != "zeros")
    coords = np.stack([rows if m == mode else rng.integers(0, d // 2, rows.size) + upper * (d // 2)
                       for m, d in enumerate(dims)]).astype(np.int32)
    vals = rng.uniform(0.5, 1.5, rows.size).astype(np.float32)
    big = kind == "large" or (kind == "mixed" and order == 4)
    row, val = {4: (1e-23, 1e37), 5: (1e-15, 1e35)}[order]
    if big:
        row, val = {4: (1e22, 1e-34), 5: (1e14, 1e-34)}[order]
    vals[upper] *= np.float32(val)
    facs = [rng.uniform(0.5, 1.5, (d, R)).astype(np.float32) for d in dims]
    others = [m for m in range(order) if m != mode]
    for m in others[:-1]:
        facs[m][dims[m] // 2:] *= np.float32(row)
        if kind == "zeros":
            facs[m][rng.random(facs[m].shape) < 0.3] = 0
    B = tt.Csf.from_coo(dims, coords, vals)
    p = vals.astype(np.float64)[:, None]
    for m in others:
        p = p * facs[m][coords[m]].astype(np.float64)
    ref = np.zeros((dims[mode], R))
    np.add.at(ref, coords[mode], p)
    used = ref[ref > 0]
    assert used.max() < 1e37 and used.min() > 1e-30
    return B, facs, ref


def _check(got, ref, what):
    zero = ref == 0
    assert np.all(got[zero] == 0), what
    e = np.abs(got[~zero] - ref[~zero]) / ref[~zero]
    assert np.max(e) <= ROW_TOL, (what, np.max(e))


KINDS = ["small", "large", "mixed", "zeros"]


@pytest.mark.parametrize("order,R", [(4, 2), (4, 16), (4, 32), (4, 50), (4, 128), (5, 3), (5, 20), (5, 32), (5, 64), (5, 200)])
@pytest.mark.parametrize("kind", KINDS)
@pytest.mark.parametrize("sizes", ["long", "short"])
def test_edge_walk(gpu, sizes, kind, order, R):
    rng = np.random.default_rng(order * 1000 + R)
    n = rng.integers(20, 900, 60) if sizes == "long" else rng.integers(0, 7, 3000)
    dims = (n.size,) + (10, 12, 14)[: order - 2] + (5000,)
    B, facs, ref = _case(rng, dims, R, 0, n, kind)
    fd = [tt.DeviceArray.from_numpy(f) for f in facs[1:]]
    names = tt.variants()
    H = tt.DeviceCsf(B)
    A = tt.DeviceArray.empty(ref.shape)
    for v in [names.index(x) for x in ("ep_b128_g4", "ep_b512_g64", "es_b256_g8")] + [tt.VARIANT_AUTO]:
        if v >= 0 and not tt.variant_fits(order, R, v):
            continue
        A.upload(np.full(ref.shape, 7.0, np.float32))
        H.mttkrp(fd, A, R, v)
        _check(A.numpy(), ref, v)
    H.close()


@pytest.mark.parametrize("R", [16, 32, 64])
@pytest.mark.parametrize("kind", KINDS)
def test_batch(gpu, kind, R):
    rng = np.random.default_rng(R)
    cases = [_case(rng, (n,) + (10, 12, 14)[: order - 2] + (5000,), R, 0, rng.integers(0, 400, n), kind)
             for order, n in ((4, 70), (5, 60))]
    tasks = [tt.DeviceCsf(B) for B, _, _ in cases]
    outs = [tt.DeviceArray.from_numpy(np.full(ref.shape, 7.0, np.float32)) for _, _, ref in cases]
    bt = tt.Batch(tasks, R)
    bt.set_operands([[tt.DeviceArray.from_numpy(f) for f in facs[1:]] for _, facs, _ in cases], outs,
                    [ref.shape[0] for _, _, ref in cases])
    for tile in (None, (1, 128, 4), (1, 512, 64)):
        if tile:
            bt.configure(*tile)
        bt.run()
        for t, (o, (_, _, ref)) in enumerate(zip(outs, cases)):
            _check(o.numpy(), ref, (tile, t))


@pytest.mark.parametrize("order,R", [(4, 2), (4, 16), (4, 32), (4, 50), (4, 128), (5, 3), (5, 20), (5, 32), (5, 64), (5, 200)])
@pytest.mark.parametrize("kind", KINDS)
@pytest.mark.parametrize("sizes", ["long", "short"])
def test_inner_modes(gpu, sizes, kind, order, R):
    rng = np.random.default_rng(order * 1000 + R)
    n = rng.integers(20, 900, 60) if sizes == "long" else rng.integers(0, 7, 3000)
    for level in range(1, order - 1):
        dims = [10, 12, 14, 16, 5000][5 - order:]
        dims[level] = n.size
        B, facs, ref = _case(rng, tuple(dims), R, level, n, kind)
        H = tt.DeviceCsf(B)
        A = tt.DeviceArray.from_numpy(np.full(ref.shape, 7.0, np.float32))
        H.mttkrp_level(level, [tt.DeviceArray.from_numpy(f) for f in facs], A, R)
        _check(A.numpy(), ref, level)
        H.close()


def _raised(rng, dims, R, mode, sizes):
    """Order 5: two of the other rows underflow together (1e-23 each) and a third
    brings their product back (1e22), whichever is multiplied first; or two
    overflow together and a third holds zeros."""
    B, facs, _ = _case(rng, dims, R, mode, sizes, "zeros")
    others = [m for m in range(5) if m != mode]
    out = []
    for big in others[:-1]:
        f = [x.copy() for x in facs]
        for m in others[:-1]:
            f[m][f[m] == 0] = 1
            f[m] *= np.float32(1e22 if m == big else 1e-23)
        out.append(f)
        g = [x.copy() for x in facs]
        for m in others[:-1]:
            if m != big:
                g[m][g[m] == 0] = 1
                g[m] *= np.float32(1e20)
        g[others[-1]] *= np.float32(1e-38)
        out.append(g)
    B.vals = B.vals * np.float32(1e10)  # (the rows one by one, in either order, stay in range)
    return B, out


@pytest.mark.parametrize("R", [3, 16, 32, 50, 64])
@pytest.mark.parametrize("mode", [0, 1, 2, 3])
def test_products_lost_on_the_way(gpu, mode, R):
    rng = np.random.default_rng(R)
    n = rng.integers(20, 400, 40)
    dims = [10, 12, 14, 16, 3000]
    dims[mode] = n.size
    B, cases = _raised(rng, tuple(dims), R, mode, n)
    # (the tensor's coordinates and values, from its CSF)
    node = np.arange(B.nnz)
    coords = [None] * 4 + [B.crd[4]]
    for m in range(4, 0, -1):
        node = np.searchsorted(B.pos[m], node, side="right") - 1
        coords[m - 1] = B.crd[m - 1][node]
    H = tt.DeviceCsf(B)
    A = tt.DeviceArray.empty((dims[mode], R))
    for facs in cases:
        p = B.vals.astype(np.float64)[:, None]
        for m in range(5):
            if m != mode:
                p = p * facs[m][coords[m]].astype(np.float64)
        ref = np.zeros((dims[mode], R))
        np.add.at(ref, coords[mode], p)
        used = ref[ref > 0]
        assert used.max() < 1e37 and used.min() > 1e-30
        fd = [tt.DeviceArray.from_numpy(f) for f in facs]
        A.upload(np.full(ref.shape, 7.0, np.float32))
        if mode == 0:
            H.mttkrp(fd[1:], A, R, tt.variants().index("ep_b256_g16"))
        else:
            H.mttkrp_level(mode, fd, A, R)
        _check(A.numpy(), ref, mode)
    H.close()
