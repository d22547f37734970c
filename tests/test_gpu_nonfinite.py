"""Infinities and NaN in factor rows stay where they belong. Row 0 of every
factor is NaN and infinite and no nonzero uses it; the last row of every factor
holds an infinity and is used by the last nonzero of some output rows only. So
lanes without a nonzero of their own must add nothing at all (0 times such a
row would be NaN): rows that use no such factor row are finite and right, and
the others infinite in the columns that are."""

import numpy as np
import pytest

import oracle
import tentaco_amd as tt
from helpers import REL_L2_TOL

pytestmark = pytest.mark.gpu


def _case(rng, dims, R, mode, sizes):
    """COO entries with sizes[j - 1] of them at coordinate j of `mode`, the
    factors, and the 64-bit MTTKRP of that mode."""
    rows = 1 + np.repeat(np.arange(sizes.size), sizes)
    coords = np.stack([rows if m == mode else rng.integers(1, d - 1, rows.size) for m, d in enumerate(dims)])
    some = 1 + np.arange(0, sizes.size, 5)
    last = np.stack([some if m == mode else np.full(some.size, d - 1) for m, d in enumerate(dims)])
    coords = np.concatenate([coords, last], axis=1).astype(np.int32)
    vals = rng.uniform(0.5, 1.5, coords.shape[1]).astype(np.float32)
    facs = [rng.uniform(0.5, 1.5, (d, R)).astype(np.float32) for d in dims]
    for m, f in enumerate(facs):
        f[0, 0::2] = np.nan
        f[0, 1::2] = np.inf
        f[-1, m % R] = np.inf
    B = tt.Csf.from_coo(dims, coords, vals)
    p = vals.astype(np.float64)[:, None]
    for m, f in enumerate(facs):
        if m != mode:
            p = p * f[coords[m]].astype(np.float64)
    ref = np.zeros((dims[mode], R))
    np.add.at(ref, coords[mode], p)
    assert np.isinf(ref).any() and not np.isnan(ref).any()
    return B, facs, ref


def _check(got, ref, what):
    fin = np.isfinite(ref)
    assert np.array_equal(got[~fin], ref[~fin].astype(np.float32)), what
    assert np.all(np.isfinite(got[fin])), what
    assert oracle.rel_l2(got[fin], ref[fin]) <= REL_L2_TOL, what


@pytest.mark.parametrize("R", [2, 3, 7, 16, 20, 32, 50, 64, 100, 128])
def test_short_fibre_slice_rows(gpu, R):
    rng = np.random.default_rng(R)
    # one slice too long for the padded and paired layouts
    sizes = np.concatenate([rng.integers(1, 130, 300), [64, 128, 63, 65, 1, 2, 700]])
    B, facs, ref = _case(rng, (sizes.size + 2, 4000, 3000), R, 0, sizes)
    fd = [tt.DeviceArray.from_numpy(f) for f in facs[1:]]
    names = tt.variants()
    H = tt.DeviceCsf(B)
    A = tt.DeviceArray.empty(ref.shape)
    for v in ("sr_b128", "sr_b256", "sr_b512"):
        A.upload(np.full(ref.shape, 7.0, np.float32))
        H.mttkrp(fd, A, R, names.index(v))
        _check(A.numpy(), ref, v)
    H.close()


@pytest.mark.parametrize("order,R", [(2, 3), (2, 16), (2, 32), (2, 50), (2, 128), (4, 2), (4, 32), (4, 100), (5, 20), (5, 64)])
def test_slice_rows(gpu, order, R):
    rng = np.random.default_rng(order * 1000 + R)
    sizes = np.concatenate([rng.integers(1, 130, 150), [64, 128, 63, 65, 1, 2, 700]])
    dims = (sizes.size + 2,) + (12, 9, 8)[: order - 2] + (3000,)
    B, facs, ref = _case(rng, dims, R, 0, sizes)
    fd = [tt.DeviceArray.from_numpy(f) for f in facs[1:]]
    names = tt.variants()
    H = tt.DeviceCsf(B)
    A = tt.DeviceArray.empty(ref.shape)
    for v in ("sr_b128", "sr_b256", "sr_b512"):
        A.upload(np.full(ref.shape, 7.0, np.float32))
        H.mttkrp(fd, A, R, names.index(v))
        _check(A.numpy(), ref, v)
    H.close()


@pytest.mark.parametrize("R", [16, 32, 64])
def test_paired_slices(gpu, R):
    rng = np.random.default_rng(R)
    sizes = rng.integers(60, 190, 300)  # two slices to a workgroup
    B, facs, ref = _case(rng, (sizes.size + 2, 4000, 3000), R, 0, sizes)
    fd = [tt.DeviceArray.from_numpy(f) for f in facs[1:]]
    H = tt.DeviceCsf(B)
    A = tt.DeviceArray.from_numpy(np.full(ref.shape, 7.0, np.float32))
    tt.ktimer_start()
    H.mttkrp(fd, A, R, tt.variants().index("sr_b256"))
    assert tt.ktimer_stop()[2] == "slice_pair_kernel"
    _check(A.numpy(), ref, "sr_b256")
    H.close()


@pytest.mark.parametrize("order,R", [(2, 32), (3, 3), (3, 16), (3, 32), (3, 50), (3, 128), (4, 64), (4, 20), (5, 200), (5, 32)])
@pytest.mark.parametrize("case", ["long", "short"])
def test_edge_walk(gpu, case, order, R):
    rng = np.random.default_rng(order * 1000 + R)
    # slices of several chunks of a wave, and many to a chunk
    sizes = rng.integers(20, 900, 60) if case == "long" else rng.integers(0, 7, 3000)
    dims = (sizes.size + 2,) + (40, 30, 50)[: order - 2] + (20_000,)
    B, facs, ref = _case(rng, dims, R, 0, sizes)
    fd = [tt.DeviceArray.from_numpy(f) for f in facs[1:]]
    names = tt.variants()
    H = tt.DeviceCsf(B)
    A = tt.DeviceArray.empty(ref.shape)
    for v in [names.index(n) for n in ("ep_b128_g4", "ep_b256_g16", "ep_b512_g64", "es_b256_g8")] + [tt.VARIANT_AUTO]:
        if v >= 0 and not tt.variant_fits(order, R, v):
            continue
        A.upload(np.full(ref.shape, 7.0, np.float32))
        H.mttkrp(fd, A, R, v)
        _check(A.numpy(), ref, v)
    H.close()


@pytest.mark.parametrize("R", [16, 32, 64])
def test_batch(gpu, R):
    rng = np.random.default_rng(R)
    cases = [_case(rng, (n + 2,) + (40, 30, 50)[: order - 2] + (9000,), R, 0, rng.integers(0, 400, n))
             for order, n in ((2, 50), (3, 90), (4, 70), (5, 60))]
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


@pytest.mark.parametrize("order,R", [(2, 32), (3, 3), (3, 16), (3, 32), (3, 50), (3, 128), (4, 64), (4, 20), (5, 200), (5, 32)])
@pytest.mark.parametrize("sizes", ["long", "short"])
def test_level_modes(gpu, sizes, order, R):
    rng = np.random.default_rng(order * 1000 + R)
    n = rng.integers(20, 900, 60) if sizes == "long" else rng.integers(0, 7, 3000)
    for level in range(1, order):
        dims = [60, 40, 30, 50, 20_000][5 - order:]
        dims[level] = n.size + 2
        B, facs, ref = _case(rng, tuple(dims), R, level, n)
        H = tt.DeviceCsf(B)
        A = tt.DeviceArray.from_numpy(np.full(ref.shape, 7.0, np.float32))
        H.mttkrp_level(level, [tt.DeviceArray.from_numpy(f) for f in facs], A, R)
        _check(A.numpy(), ref, level)
        H.close()
