"""The node-parallel stage at the edges of its launch forms: block orders
(device tuning 0, 1, 2), one block per element, per task and resident grids
give the same bits, at element counts around a task, a cube of 64 tasks
and a group of 512."""
import numpy as np
import pytest

import bfam_amd as bx
import bfam_amd.workloads as W
from util import random_elastic

pytestmark = pytest.mark.gpu


def _final(cfg, q0, prec, N, kind, remap, steps=2):
    dev = bx.Device(0)
    dev.set_tuning(remap)
    dev.set_kernel(prec, N, kind)
    sub = W.upload(dev, cfg, prec)
    sub.set_fields(q0, 0.0, cfg["dt"])
    sub.step(steps)
    q = sub.download()
    sub.close()
    dev.close()
    return q


# elements of a brick: one; around a task (8, 4, 2 elements); past 64 tasks,
# with a remainder; past 512 one-element tasks, with a remainder
BRICKS = [(1, 1, 1), (3, 1, 1), (3, 3, 1), (5, 13, 1), (19, 7, 1), (9, 9, 7)]


@pytest.mark.parametrize("prec", [bx.FP32, bx.FP32_RHS, bx.FP64])
@pytest.mark.parametrize("N", [3, 4, 5, 6, 7])
@pytest.mark.parametrize("n", BRICKS, ids=lambda n: "x".join(map(str, n)))
def test_launch_forms_agree(n, N, prec):
    cfg, q0 = random_elastic(n, N, seed=N)
    ref = _final(cfg, q0, prec, N, 1, 0)
    assert np.isfinite(ref).all() and np.abs(ref - q0).max() > 0
    for kind, remap in ((1, 1), (1, 2), (2, 0), (2, 1), (2, 2)):
        np.testing.assert_array_equal(_final(cfg, q0, prec, N, kind, remap), ref)
