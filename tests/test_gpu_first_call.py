"""The hot-region timer of a process's first host calls holds the kernels alone:
loading an order's code object (milliseconds) falls before it. A fresh process,
one small tensor of every order, each of them the first of its order."""

import os
import subprocess
import sys

import pytest

pytestmark = pytest.mark.gpu

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))

SOURCE = """
import numpy as np
import tentaco_amd as tt
rng = np.random.default_rng(1)
for order in (3, 5, 2, 4):
    dims = (60, 50, 40, 30, 20)[:order]
    B = tt.Csf.from_coo(dims, np.stack([rng.integers(0, d, 2000) for d in dims]).astype(np.int32),
                        rng.uniform(-1, 1, 2000).astype(np.float32))
    tt.mttkrp(B, [rng.uniform(-1, 1, (d, 32)).astype(np.float32) for d in dims[1:]], tt.default_variant())
    print(order, tt.last_timer_ms(), flush=True)
"""


def test_first_call_of_each_order_times_the_kernels(gpu):
    r = subprocess.run([sys.executable, "-u", "-c", SOURCE], cwd=ROOT, stdout=subprocess.PIPE, text=True, timeout=100)
    assert r.returncode == 0, r.stdout
    ms = {int(l.split()[0]): float(l.split()[1]) for l in r.stdout.splitlines()}
    assert sorted(ms) == [2, 3, 4, 5]
    assert all(0 < t < 1 for t in ms.values()), ms  # (0.03; with the load 3.8)
