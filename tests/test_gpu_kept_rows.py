"""The FP64 rows that a handle keeps for tiles of many workgroups: a sweep, which
runs every such tile, leaves none behind but the handle's own, and the tiles
that calls name have them whatever was swept or called before (at most 8 are
kept, the least recently used goes)."""

import ctypes

import numpy as np
import pytest

import tentaco_amd as tt
from test_gpu_graph import _hip

pytestmark = pytest.mark.gpu


def _free_bytes(hip):
    free, total = ctypes.c_size_t(), ctypes.c_size_t()
    assert hip.hipMemGetInfo(ctypes.byref(free), ctypes.byref(total)) == 0
    return free.value


def _ones(dims, R):
    return [tt.DeviceArray.from_numpy(np.ones((d, R), np.float32)) for d in dims]


def test_sweep_keeps_no_rows(gpu):
    hip = _hip()
    n = np.arange(1 << 22)
    coords = np.stack([n >> 12, n >> 3 & 511, n & 7]).astype(np.int32)
    dims = (1024, 512, 8)
    R = 64
    H = tt.DeviceCsf(tt.Csf.from_coo(dims, coords, np.ones(n.size, np.float32)))
    fd = _ones(dims[1:], R)
    A = tt.DeviceArray.empty((dims[0], R))
    H.reserve(R)
    H.mttkrp(fd, A, R)
    tt.synchronize()
    before = _free_bytes(hip)
    H.sweep(fd, A, R, reps=1)
    # the smallest tile's rows alone take 16 R B for each of 131072 workgroups
    assert before - _free_bytes(hip) < 16 * R * (1 << 22) // 32 // 4
    H.autotune(fd, A, R, reps=1)
    assert before - _free_bytes(hip) <= 16 * R * (1 << 22) // 32 + (32 << 20)
    H.close()


def test_later_ranks_have_rows(gpu):
    # one slice, 2^24 in its first workgroup, then parts that FP32 additions to
    # 2^24 would lose (see test_gpu_auto_rows)
    n = np.arange(1 << 20)
    coords = np.stack([np.zeros_like(n), n // 8, n % 8]).astype(np.int32)
    vals = np.full(n.size, 2.0 ** -11, np.float32)
    vals[:4096] = 0
    vals[0] = 2.0 ** 24
    dims = (1, n.size // 8, 8)
    total = np.float32(2.0 ** 24 + (n.size - 4096) / 2048)
    H = tt.DeviceCsf(tt.Csf.from_coo(dims, coords, vals))
    names = tt.variants()
    fd = _ones(dims[1:], 32)
    A = tt.DeviceArray.empty((1, 32))
    H.sweep(fd, A, 32, reps=1)
    ranks = [16, 64, 128, 20, 48, 8, 100, 12, 24, 16, 32]
    ops = {R: (_ones(dims[1:], R), tt.DeviceArray.empty((1, R))) for R in ranks}
    for v in ("ep_b128_g4", "ep_b128_g8"):
        for R in ranks:
            f, out = ops[R]
            for _ in range(2):
                out.upload(np.full((1, R), 7.0, np.float32))
                H.mttkrp(f, out, R, names.index(v))
                assert np.all(out.numpy() == total), (v, R)
    H.close()


def _lossy_slice():
    n = np.arange(1 << 20)
    coords = np.stack([np.zeros_like(n), n // 8, n % 8]).astype(np.int32)
    vals = np.full(n.size, 2.0 ** -11, np.float32)
    vals[:4096] = 0
    vals[0] = 2.0 ** 24
    dims = (1, n.size // 8, 8)
    return tt.Csf.from_coo(dims, coords, vals), dims, np.float32(2.0 ** 24 + (n.size - 4096) / 2048)


def test_a_choice_after_reserve_has_rows(gpu):
    """A handle reserved for AUTO, then given a selector: its pick's tables are
    built with the pick, as later calls build none."""
    B, dims, total = _lossy_slice()
    R = 32
    H = tt.DeviceCsf(B)
    fd = _ones(dims[1:], R)
    A = tt.DeviceArray.empty((1, R))
    pick = tt.variants().index("ep_b128_g4")
    sel = tt.Selector()
    p = np.zeros_like(sel.params())
    p[-len(tt.variants()):] = 1.0  # the output layer's biases
    p[-len(tt.variants()) + pick] = -1.0
    sel.set_params(p)
    assert sel.select(3, R, H.features(R))[0] == pick
    H.reserve(R)
    H.set_selector(sel, 0.0)
    for _ in range(3):
        A.upload(np.full((1, R), 7.0, np.float32))
        H.mttkrp(fd, A, R)
        assert H.tuned(R)[0] == pick
        assert np.all(A.numpy() == total)
    H.close()
    sel.close()


def test_streams_and_a_graph_on_one_handle(gpu):
    """Calls that add to one handle's rows on two streams wait for each other, and
    a captured call's replays, which use none, run between them."""
    from test_gpu_graph import _capture

    hip = _hip()
    n = np.arange(1 << 18)
    rng = np.random.default_rng(5)
    coords = np.stack([n >> 15, n >> 3 & 4095, n & 7]).astype(np.int32)
    vals = rng.integers(-8, 9, n.size).astype(np.float32)  # whole numbers: every sum is exact
    dims = (8, 4096, 8)
    R = 32
    B = tt.Csf.from_coo(dims, coords, vals)
    H = tt.DeviceCsf(B)
    v = tt.variants().index("ep_b128_g4")  # 4096 workgroups
    facs = [rng.integers(-2, 3, (d, R)).astype(np.float32) for d in dims[1:]]
    other = [rng.integers(-2, 3, (d, R)).astype(np.float32) for d in dims[1:]]

    def exact(f):
        ref = np.zeros((8, R))
        np.add.at(ref, coords[0], vals[:, None].astype(np.float64) * f[0][coords[1]] * f[1][coords[2]])
        assert np.abs(ref).max() < 2 ** 24
        return ref

    refs = [exact(facs), exact(other)]
    ops = [[tt.DeviceArray.from_numpy(x) for x in f] for f in (facs, other)]
    outs = [[tt.DeviceArray.empty((8, R)) for _ in range(6)] for _ in range(2)]
    streams = [tt.Stream(), tt.Stream()]
    H.reserve(R, v)
    G = tt.DeviceArray.empty((8, R))
    g, ex = _capture(hip, streams[0], lambda: H.mttkrp(ops[1], G, R, v, stream=streams[0].h))
    try:
        for rep in range(3):
            for o in outs[0] + outs[1] + [G]:
                o.upload(np.full((8, R), 7.0 + rep, np.float32))
            for i in range(6):
                for k in (0, 1):
                    H.mttkrp(ops[k], outs[k][i], R, v, stream=streams[k].h)
                # (a replay writes the handle's workspace: it waits for the calls)
                for s in streams:
                    s.synchronize()
                assert hip.hipGraphLaunch(ex, streams[0].h) == 0
                streams[0].synchronize()
                assert np.array_equal(G.numpy(), refs[1]), (rep, i)
            for k in (0, 1):
                for o in outs[k]:
                    assert np.array_equal(o.numpy(), refs[k]), (rep, k)
        for i in range(6):  # without a wait between them
            for k in (0, 1):
                H.mttkrp(ops[k], outs[k][i], R, v, stream=streams[k].h)
        for s in streams:
            s.synchronize()
        for k in (0, 1):
            for o in outs[k]:
                assert np.array_equal(o.numpy(), refs[k]), k
    finally:
        hip.hipGraphExecDestroy(ex)
        hip.hipGraphDestroy(g)
    H.close()
    for s in streams:
        s.close()
