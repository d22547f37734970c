"""Batches of several orders with more work items than the one launch for all
orders takes (10 a workgroup of it; at most 16 workgroups of 128 threads on each
of 256 CUs): a launch per order, at every rank, with written and retained
outputs, eagerly and replayed."""

import numpy as np
import pytest

import oracle
import tentaco_amd as tt
from helpers import REL_L2_TOL

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("R", [16, 32, 64])
def test_more_items_than_one_launch_takes(gpu, R):
    rng = np.random.default_rng(R)
    per_item = 128 // (R // 4)  # nonzeros of an item of 128 threads, one a lane group
    total = 10 * 16 * 256 * per_item
    cases = []
    for dims, share in (((900, 2100), 0.2), ((300, 500, 700), 0.45), ((5000, 40, 60, 50), 0.3), ((120, 30, 40, 20, 50), 0.3)):
        n = int(total * share)
        B = tt.Csf.from_coo(dims, np.stack([rng.integers(0, d, n) for d in dims]).astype(np.int32),
                            rng.uniform(-1, 1, n).astype(np.float32))
        f = [rng.uniform(-1, 1, (d, R)).astype(np.float32) for d in dims[1:]]
        cases.append((B, f, oracle.mttkrp(B, f, "taco", fp64=True)))
    tasks = [tt.DeviceCsf(B) for B, _, _ in cases]
    outs = [tt.DeviceArray.empty(ref.shape) for _, _, ref in cases]
    bt = tt.Batch(tasks, R)
    bt.set_operands([[tt.DeviceArray.from_numpy(x) for x in f] for _, f, _ in cases], outs,
                    [ref.shape[0] for _, _, ref in cases])
    bt.configure(1, 128, 1)
    items = sum(-(-B.nnz // per_item) for B, _, _ in cases)
    assert items > 10 * 16 * 256
    for mode in (bt.OUTPUTS_WRITTEN, bt.OUTPUTS_RETAINED):
        for o in outs:
            o.upload(np.full(o.shape, 7.0, np.float32))
        bt.set_output_mode(mode)
        bt.run()
        bt.capture()
        for rep in range(3):
            for t, (o, (_, _, ref)) in enumerate(zip(outs, cases)):
                assert oracle.rel_l2(o.numpy(), ref) <= REL_L2_TOL, (mode, rep, t)
            bt.launch()
            tt.synchronize()
    bt.close()
