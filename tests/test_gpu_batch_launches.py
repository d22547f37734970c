"""The batch's two ways to launch several orders (one launch for all; one per
order, on queues of their own), over which choices of tile and schedule take
each, with written and retained outputs, eagerly and as a replayed graph."""

import numpy as np
import pytest

import oracle
import tentaco_amd as tt
from helpers import REL_L2_TOL

pytestmark = pytest.mark.gpu


def _one_order_tiles(bt):
    for order in range(2, 6):
        bt.configure_order(order, 1, 256, 16, 0)


def _mixed_blocks(bt):
    _one_order_tiles(bt)
    bt.configure_order(4, 1, 128, 8, 0)


def _mixed_schedules(bt):
    _one_order_tiles(bt)
    bt.configure_order(5, 1, 256, 16, 1)


def _many_items(bt):
    bt.configure(1, 128, 1)  # far past the one launch's limit of items


def _static(bt):
    bt.configure(1, 256, 64)
    bt.set_schedule(1)


@pytest.mark.parametrize("R", [16, 32, 64])
@pytest.mark.parametrize("tiles", [_one_order_tiles, _mixed_blocks, _mixed_schedules, _many_items, _static])
def test_batch_launch_forms(gpu, tiles, R):
    rng = np.random.default_rng(R)
    shapes = [((900, 2100), 30_000), ((300, 500, 700), 150_000), ((5000, 40, 60, 50), 60_000),
              ((120, 30, 40, 20, 50), 90_000), ((70_000, 3, 3), 64)]
    Bs, facs = [], []
    for dims, n in shapes:
        Bs.append(tt.Csf.from_coo(dims, np.stack([rng.integers(0, d, n) for d in dims]).astype(np.int32),
                                  rng.uniform(-1, 1, n).astype(np.float32)))
        facs.append([rng.uniform(-1, 1, (d, R)).astype(np.float32) for d in dims[1:]])
    refs = [oracle.mttkrp(B, f, "taco", fp64=True) for B, f in zip(Bs, facs)]
    tasks = [tt.DeviceCsf(B) for B in Bs]
    outs = [tt.DeviceArray.empty((d[0], R)) for d, _ in shapes]
    bt = tt.Batch(tasks, R)
    bt.set_operands([[tt.DeviceArray.from_numpy(f) for f in fs] for fs in facs], outs, [d[0] for d, _ in shapes])
    tiles(bt)

    def check(what):
        for t, (o, ref) in enumerate(zip(outs, refs)):
            assert oracle.rel_l2(o.numpy(), ref) <= REL_L2_TOL, (what, t)

    for mode in (bt.OUTPUTS_WRITTEN, bt.OUTPUTS_RETAINED):
        for o in outs:
            o.upload(np.full(o.shape, 7.0, np.float32))
        bt.set_output_mode(mode)  # retained: zeroes the rows no launch stores
        bt.run()
        check((mode, "run"))
        bt.capture()
        for rep in range(3):
            if mode == bt.OUTPUTS_WRITTEN:
                for o in outs:
                    o.upload(np.full(o.shape, float(rep), np.float32))
            bt.launch()
            check((mode, rep))
