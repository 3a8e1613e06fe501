"""The order launches of a mixed batch without mortars run as chains of stages
on several streams that meet where the clocks advance: every member takes the
bits it takes alone, whatever the number of orders, in eager runs past one
refill of the clocks and in replays of a captured graph."""
import numpy as np
import pytest

import bfam_amd as bx
import bfam_amd.workloads as W
from util import random_elastic

pytestmark = pytest.mark.gpu

# (order, elements per axis): one to five orders, an order with two members
SETS = [[(3, 2), (3, 3)], [(4, 3), (7, 1)], [(6, 1), (3, 3), (5, 2)],
        [(7, 2), (3, 4), (5, 2), (4, 3), (6, 1), (3, 1)]]


@pytest.mark.parametrize("prec", [bx.FP32, bx.FP64])
@pytest.mark.parametrize("members", SETS, ids=lambda m: "-".join(str(n) for n, _ in m))
def test_members_step_as_alone(members, prec):
    print(f"chains {members} prec={prec}", flush=True)
    dev = bx.Device(0)
    steps = 11  # past one refill (eight steps of five stages)
    cfgs, subs, alone = [], [], []
    for s, (N, n) in enumerate(members):
        cfg, q0 = random_elastic((n, n, n), N, seed=s)
        cfgs.append((cfg, q0))
        sub = W.upload(dev, cfg, prec)
        sub.set_fields(q0, 0.0, cfg["dt"])
        sub.step(steps)
        alone.append(sub.download())
        subs.append(sub)

    def reset():
        for sub, (cfg, q0) in zip(subs, cfgs):
            sub.set_fields(q0, 0.0, cfg["dt"])

    b = bx.Batch(dev, subs)
    for parts in ((11,), (1, 9, 1)):
        reset()
        for k in parts:
            b.step(k)
        for sub, q in zip(subs, alone):
            assert np.isfinite(q).all()
            np.testing.assert_array_equal(sub.download(), q)
    b.capture(1)
    reset()
    for i in range(steps):
        b.launch_graph()
        if i % 4 == 1:
            dev.sync()
    for sub, q in zip(subs, alone):
        np.testing.assert_array_equal(sub.download(), q)
    b.capture(9)  # a refill within the graph
    reset()
    b.launch_graph()
    b.step(2)
    for sub, q in zip(subs, alone):
        np.testing.assert_array_equal(sub.download(), q)
    b.close()
    for sub in subs:
        sub.close()
    dev.close()
