"""The stage parameters a subdomain's clock holds ahead (source and forcing
scalars, LSRK coefficients, ping-pong parity of the next 40 stages): a run
gives the same bits however its stages are divided into calls, across the
refill of the clock, for tables of 1, 2, 3 and 5 stages, and a batch steps as
its member does alone."""
import numpy as np
import pytest

import bfam_amd as bx
import bfam_amd.workloads as W
from util import random_elastic

pytestmark = pytest.mark.gpu


def _problem(forced):
    cfg, q0 = random_elastic((2, 3, 2), 3, seed=4)
    if forced:
        cfg.update({"k": 2 * np.pi, "omega": 3.0, "F": np.linspace(-1, 1, 9)})
    return cfg, q0


def _run(cfg, q0, prec, method, advance):
    dev = bx.Device(0)
    sub = W.upload(dev, cfg, prec, lsrk_method=method)
    sub.set_fields(q0, 0.1, cfg["dt"])
    try:
        advance(dev, sub)
        return sub.download(), sub.time()
    finally:
        sub.close()
        dev.close()


def _graph(steps, per):
    def go(dev, sub):
        b = bx.Batch(dev, [sub])
        b.capture(per)
        for _ in range(steps // per):
            b.launch_graph()
        dev.sync()
        b.close()
    return go


def _mixed(steps):
    """single stages to the middle of a step, then a batch, then the rest"""
    def go(dev, sub):
        ns = sub.nstages
        for _ in range(ns + 1):
            sub.stage()
        b = bx.Batch(dev, [sub])
        b.step(steps - 3)
        dev.sync()
        b.close()
        for _ in range(2 * ns - 1):
            sub.stage()
    return go


@pytest.mark.parametrize("method", [bx.LSRK_KC54, bx.LSRK_FE, bx.LSRK_HEUN, bx.LSRK_W33])
@pytest.mark.parametrize("prec", [bx.FP64, bx.FP32])
def test_divided_runs_agree(method, prec):
    cfg, q0 = _problem(forced=True)
    ns = {bx.LSRK_KC54: 5, bx.LSRK_FE: 1, bx.LSRK_HEUN: 2, bx.LSRK_W33: 3}[method]
    steps = 6 * (40 // ns // 6 + 2)  # past one refill of the clock, a multiple of 6
    cfg["dt"] *= 0.2
    q, t = _run(cfg, q0, prec, method, lambda d, s: s.step(steps))
    assert np.isfinite(q).all() and t[1] == steps * ns
    for go in (lambda d, s: [s.stage() for _ in range(steps * ns)],
               lambda d, s: [s.step(1) for _ in range(steps)], _graph(steps, 6), _graph(steps, 1),
               _mixed(steps)):
        q2, t2 = _run(cfg, q0, prec, method, go)
        assert t2 == t
        assert np.array_equal(q2, q)


def test_source_set_during_a_run():
    """a new source takes effect from the next stage on"""
    cfg, q0 = _problem(forced=False)
    s = cfg["src"]

    def change(d, sub):
        sub.step(3)
        sub.set_source(s["elem"], s["weights"], s["amp"], 2 * s["f0"], 0.1)
        sub.step(9)

    def change_by_stages(d, sub):
        for _ in range(15):
            sub.stage()
        sub.set_source(s["elem"], s["weights"], s["amp"], 2 * s["f0"], 0.1)
        for _ in range(45):
            sub.stage()

    a, ta = _run(cfg, q0, bx.FP64, bx.LSRK_KC54, change)
    b, tb = _run(cfg, q0, bx.FP64, bx.LSRK_KC54, change_by_stages)
    c, _ = _run(cfg, q0, bx.FP64, bx.LSRK_KC54, lambda d, sub: sub.step(12))
    assert ta == tb and np.array_equal(a, b)
    assert not np.array_equal(a, c)
