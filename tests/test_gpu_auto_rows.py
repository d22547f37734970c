"""AUTO's tile, which is smaller than the variant it stands for, adds a long
slice's parts in FP64 or is not run. The slice's first workgroup holds 2^24, and
every one of the variant's other workgroups adds 2, which FP32 keeps whatever
the order (its steps at 2^24 are 2). The sized tile's workgroups add 1/2, which
FP32 atomics would lose and FP64 rows keep. So every kind of call has the exact
sum: eager ones, first or later, on a handle reserved for AUTO or for something
else, two streams in turn, a captured graph's replays between eager calls, the
allocation-free call and the host calls."""

import ctypes

import numpy as np
import pytest

import tentaco_amd as tt
from test_gpu_graph import _capture, _hip

pytestmark = pytest.mark.gpu

R = 32


def _tensor():
    nb = 4096  # nonzeros of a workgroup of the variant (512 threads x 64, rank 32)
    assert tt.variant_params(tt.variants().index("ep_b512_g64"))[1:] == (512, 64)
    n = np.arange(256 * nb)
    coords = np.stack([np.zeros_like(n), n // 8, n % 8]).astype(np.int32)
    vals = np.full(n.size, 2.0 / nb, np.float32)
    vals[:nb] = 0
    vals[0] = 2.0 ** 24
    dims = (2, n.size // 8, 8)
    return tt.Csf.from_coo(dims, coords, vals), dims, 2.0 ** 24 + 2 * 255


def test_every_kind_of_call(gpu):
    hip = _hip()
    B, dims, total = _tensor()
    host = [np.ones((d, R), np.float32) for d in dims[1:]]
    fd = [tt.DeviceArray.from_numpy(f) for f in host]
    half = [tt.DeviceArray.from_numpy(np.ones((d, 16), np.float32)) for d in dims[1:]]
    arr = (ctypes.c_void_p * 2)(*[f.ptr for f in fd])
    A = tt.DeviceArray.empty((2, R))
    A16 = tt.DeviceArray.empty((2, 16))
    ref = np.zeros((2, R), np.float32)
    ref[0] = total

    def check(what, call):
        A.upload(np.full((2, R), 7.0, np.float32))
        call()
        tt.synchronize()
        assert np.array_equal(A.numpy(), ref), (what, A.numpy()[0, 0] - total)

    first = tt.DeviceCsf(B)
    assert tt.variants()[first.resolve(R)] == "ep_b512_g64"
    for what in ("first", "second"):
        check(what, lambda: first.mttkrp(fd, A, R))
    reserved = tt.DeviceCsf(B)
    reserved.reserve(R)
    check("reserved", lambda: reserved.mttkrp(fd, A, R))
    other = tt.DeviceCsf(B)
    other.reserve(16, tt.default_variant())
    check("reserved for something else", lambda: other.mttkrp(fd, A, R))
    other.mttkrp(half, A16, 16)
    # two streams on one handle, ranks in between, the outputs of both
    s, s2 = tt.Stream(), tt.Stream()
    A2 = tt.DeviceArray.empty((2, R))

    def turns():
        for _ in range(8):
            first.mttkrp(fd, A, R, stream=s.h)
            first.mttkrp(fd, A2, R, stream=s2.h)
        first.mttkrp(half, A16, 16, stream=s.h)
        first.mttkrp(fd, A, R, stream=s.h)
        s.synchronize()
        s2.synchronize()

    check("streams", turns)
    assert np.array_equal(A2.numpy(), ref)
    for h in (reserved, first):
        g, ex = _capture(hip, s, lambda: h.mttkrp(fd, A, R, stream=s.h))
        try:
            for rep in range(3):
                def replay():
                    assert hip.hipGraphLaunch(ex, s.h) == 0
                    s.synchronize()
                check(("replay", rep), replay)
                check(("between", rep), lambda: h.mttkrp(fd, A, R, stream=s2.h))
        finally:
            hip.hipGraphExecDestroy(ex)
            hip.hipGraphDestroy(g)
    for h in (first, other, tt.DeviceCsf(B)):
        def noalloc():
            assert tt.lib().tentaco_mttkrp_dev_noalloc(h.h, R, arr, A.ptr, 2, tt.VARIANT_AUTO, None) == tt.OK
        check("noalloc", noalloc)
    assert np.array_equal(tt.mttkrp(B, host, tt.VARIANT_AUTO), ref)
    up = tt.DeviceCsf.upload_async(B, s)
    out = np.full((2, R), 7.0, np.float32)
    for _ in range(2):
        up.mttkrp_host_async(host, out, R, s)
        s.synchronize()
        assert np.array_equal(out, ref)
    for h in (first, reserved, other, up):
        h.close()
    s.close()
    s2.close()
