"""The node-parallel stage on resident grids whose blocks take several turns:
the same bits as one block per task or element, in every block order.

A CU holds at most 32 wavefronts.  With residency capped at half, a resident
grid has at most 16 / W blocks per CU, W wavefronts each, and 16 times that
where an order's blocks take part of a task (N = 3..5); the bricks have more
work than that, with a partial last task and a partial last group of 512
blocks, so that every block loops over its share and the shares are uneven."""
import numpy as np
import pytest

import bfam_amd as bx
import bfam_amd.workloads as W
from util import random_elastic

pytestmark = pytest.mark.gpu

# order -> brick, elements of a task
BRICKS = {3: ((41, 41, 41), 8), 4: ((33, 33, 31), 4), 5: ((27, 25, 25), 2), 6: ((11, 9, 7), 1),
          7: ((11, 9, 7), 1)}


def _turns(dev, N, prec, K, epb):
    """blocks' worth of work over the most blocks that the grid can have"""
    waves = -(-epb * (N + 1) ** 3 // 64)
    task = BRICKS[N][1]
    resident = 16 // waves * dev.info()[0] * (16 if epb < task else 1)
    work = -(-K // task) * (task // epb)
    assert work % 512 and (task == 1 or K % task)
    return work / resident


@pytest.mark.parametrize("prec", [bx.FP32, bx.FP32_RHS, bx.FP64])
@pytest.mark.parametrize("N", sorted(BRICKS))
def test_turns_of_a_resident_grid(N, prec):
    print(f"resident grid N={N} prec={prec}", flush=True)
    n, task = BRICKS[N]
    cfg, q0 = random_elastic(n, N, seed=N)
    dev = bx.Device(0)
    # elements per block (N = 3: FP64 blocks of two), and per block of kinds 3, 4
    assert _turns(dev, N, prec, cfg["mesh"].K, 2 if N == 3 and prec == bx.FP64 else 1) > 1
    pairs = [((1, 0), ((2, 0), (2, 1), (2, 2), (1, 1), (1, 2)))]
    if N <= 5:
        assert _turns(dev, N, prec, cfg["mesh"].K, task) > 1
        pairs.append(((3, 0), ((4, 0), (4, 1), (4, 2))))

    def final(kind, remap):
        dev.set_tuning(remap)
        dev.set_kernel(prec, N, kind)
        sub.set_fields(q0, 0.0, cfg["dt"])
        rate = sub.rhs(0.1)
        sub.step(1)
        return rate, sub.download()

    sub = W.upload(dev, cfg, prec)
    for slot in (1, 2):
        dev.set_occupancy(prec, N, slot, 2)
    for base, others in pairs:
        rate, want = final(*base)
        assert np.isfinite(want).all() and np.abs(want - q0).max() > 0
        for form in others:
            r, q = final(*form)
            assert np.array_equal(r, rate) and np.array_equal(q, want), form
    sub.close()
    dev.close()
