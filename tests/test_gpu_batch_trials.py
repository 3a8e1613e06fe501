"""Mixed batches in the serving loop's default precision (FP32 rates) and
under the autotuner's trials of whole steps: every member takes the bits it
takes alone."""
import numpy as np
import pytest

import bfam_amd as bx
import bfam_amd.workloads as W
from util import random_elastic

pytestmark = pytest.mark.gpu

SETS = [[(3, 2), (3, 3)], [(4, 3), (7, 1)], [(6, 1), (3, 3), (5, 2)],
        [(7, 2), (3, 4), (5, 2), (4, 3), (6, 1), (3, 1)]]


def _members(dev, members, prec):
    cfgs, subs = [], []
    for s, (N, n) in enumerate(members):
        cfg, q0 = random_elastic((n, n, n), N, seed=s)
        cfgs.append((cfg, q0))
        subs.append(W.upload(dev, cfg, prec))
    return cfgs, subs


def _reset(cfgs, subs):
    for sub, (cfg, q0) in zip(subs, cfgs):
        sub.set_fields(q0, 0.0, cfg["dt"])


@pytest.mark.parametrize("members", SETS, ids=lambda m: "-".join(str(n) for n, _ in m))
def test_fp32_rates_step_as_alone(members):
    print(f"chains {members} FP32 rates", flush=True)
    dev = bx.Device(0)
    cfgs, subs = _members(dev, members, bx.FP32_RHS)
    _reset(cfgs, subs)
    alone = []
    for sub in subs:
        sub.step(11)  # past one refill of the clocks
        alone.append(sub.download())
    b = bx.Batch(dev, subs)
    _reset(cfgs, subs)
    for k in (1, 9, 1):
        b.step(k)
    for sub, q in zip(subs, alone):
        np.testing.assert_array_equal(sub.download(), q)
    b.capture(1)
    _reset(cfgs, subs)
    for i in range(11):
        b.launch_graph()
        if i % 4 == 1:
            dev.sync()
    for sub, q in zip(subs, alone):
        assert np.isfinite(q).all()
        np.testing.assert_array_equal(sub.download(), q)
    b.close()
    for sub in subs:
        sub.close()
    dev.close()


@pytest.mark.parametrize("prec", [bx.FP32, bx.FP32_RHS, bx.FP64])
@pytest.mark.parametrize("members", SETS[1:], ids=lambda m: "-".join(str(n) for n, _ in m))
def test_trials_of_the_strategy_leave_no_trace(members, prec):
    """Every order on the line kernel, so that the autotuner times the two
    strategies, in the middle of a step: the run goes on as without it."""
    print(f"strategy trials {members} prec={prec}", flush=True)
    dev = bx.Device(0)
    for N, _ in members:
        dev.set_kernel(prec, N, 0)
    cfgs, subs = _members(dev, members, prec)
    _reset(cfgs, subs)
    alone = []
    for sub in subs:
        sub.step(4)
        alone.append(sub.download())
    _reset(cfgs, subs)
    for sub in subs:
        for _ in range(7):
            sub.stage()
    b = bx.Batch(dev, subs)
    b.autotune(2)
    b.step(2)
    b.close()
    for sub, q in zip(subs, alone):
        for _ in range(3):
            sub.stage()
        np.testing.assert_array_equal(sub.download(), q)
        sub.close()
    dev.close()
