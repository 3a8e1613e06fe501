"""The node-parallel stage at the edges of its launch forms: block orders
(device tuning 0, 1, 2), one block per element, per task and resident grids
give the same bits, at element counts around a task, a cube of 64 tasks, a
group of 512 and, FP64 N = 4, where blocks take whole tasks."""
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


@pytest.mark.parametrize("nx", [28, 27])
def test_fp64_n4_whole_and_split_tasks(nx):
    """7168 tasks of four elements take whole tasks, 6912 one block per
    element; the two forms compute an element alike up to the rounding of a
    differently contracted sum (states of order 1, ten stages: 1e-13)."""
    N = 4
    mesh = W.Mesh(3, [nx, 32, 32], N, L=[1.0, 1.0, 1.0])
    assert (mesh.K >= 4 * 7168) == (nx == 28)
    cfg, q0 = random_elastic((nx, 32, 32), N, seed=nx)
    a = _final(cfg, q0, bx.FP64, N, 1, 2)
    b = _final(cfg, q0, bx.FP64, N, 3, 2)
    scale = np.abs(a).max()
    assert np.isfinite(a).all()
    assert np.abs(a - b).max() <= 1e-13 * scale
