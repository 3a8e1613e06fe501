"""Stages captured by the caller on the device's stream (bfamx_device_stream)
and replayed there: the capture itself runs none, and every query afterwards
sees the stages replayed, an odd number of them included.  Replays mix with
eager runs of the same subdomain through other descriptors: a batch keeps
those of its creation, and a later source is the subdomain's own."""
import ctypes as C

import numpy as np
import pytest

import bfam_amd as bx
import bfam_amd.workloads as W
from util import random_acoustic, random_elastic

pytestmark = pytest.mark.gpu


class Capture:
    """What `run` enqueues on the device's stream, as a graph to launch."""

    def __init__(self, dev, run):
        self.hip = bx.lib()  # its HIP runtime's symbols
        self.st = C.c_void_p(bx.lib().bfamx_device_stream(dev.h))
        graph = C.c_void_p()
        self.exe = C.c_void_p()
        self.call("hipStreamBeginCapture", self.st, C.c_int(1))
        run()
        self.call("hipStreamEndCapture", self.st, C.byref(graph))
        self.call("hipGraphInstantiate", C.byref(self.exe), graph, None, None, C.c_size_t(0))
        self.call("hipGraphDestroy", graph)

    def call(self, name, *args):
        f = getattr(self.hip, name)
        f.restype = C.c_int
        assert f(*args) == 0, name

    def launch(self):
        self.call("hipGraphLaunch", self.exe, self.st)

    def close(self):
        self.call("hipGraphExecDestroy", self.exe)


def _sub(dev, prec, seed, acoustic=False, N=4):
    cfg, q0 = random_acoustic((3, 2), 4, seed) if acoustic else random_elastic((2, 1, 2), N, seed)
    return W.upload(dev, cfg, prec), cfg, q0


@pytest.mark.parametrize("prec", [bx.FP64, bx.FP32, bx.FP32_RHS, bx.FP64_PLAIN])
@pytest.mark.parametrize("acoustic", [False, True], ids=["elastic", "acoustic"])
@pytest.mark.parametrize("what", ["stage", "step"])
def test_captured_by_the_caller(what, acoustic, prec):
    print(f"caller's capture {what} acoustic={acoustic} prec={prec}", flush=True)
    dev = bx.Device(0)
    sub, cfg, q0 = _sub(dev, prec, 3, acoustic)
    ref, _, _ = _sub(dev, prec, 3, acoustic)
    for x in (sub, ref):
        x.set_fields(q0, 0.0, cfg["dt"])
    start = ref.download()
    g = Capture(dev, sub.stage if what == "stage" else sub.step)
    np.testing.assert_array_equal(sub.download(), start)
    for replay in range(4):
        g.launch()
        (ref.stage if what == "stage" else ref.step)()
        np.testing.assert_array_equal(sub.download(), ref.download())
        assert sub.energy() == ref.energy() and sub.time() == ref.time()
        assert sub.l2_diff(ref) == ref.l2_diff(ref)
        if replay == 2:  # eager work between the replays
            sub.step(1)
            ref.step(1)
    np.testing.assert_array_equal(sub.download(), ref.download())
    g.close()
    sub.close()
    ref.close()
    dev.close()


@pytest.mark.parametrize("prec", [bx.FP64, bx.FP32, bx.FP32_RHS])
def test_batch_captured_by_the_caller(prec):
    print(f"caller's capture of a batch prec={prec}", flush=True)
    dev = bx.Device(0)
    subs, refs = [], []
    for N in (3, 5, 4):
        for xs in (subs, refs):
            s, cfg, q0 = _sub(dev, prec, N, N=N)
            s.set_fields(q0, 0.0, cfg["dt"])
            xs.append(s)
    b, r = bx.Batch(dev, subs), bx.Batch(dev, refs)
    g = Capture(dev, b.step)
    for replay in range(3):
        g.launch()
        r.step()
        for s, t in zip(subs, refs):
            np.testing.assert_array_equal(s.download(), t.download())
        if replay == 1:
            b.step(2)
            r.step(2)
    g.close()
    for x in (b, r, *subs, *refs):
        x.close()
    dev.close()


@pytest.mark.parametrize("replayed", ["subdomain", "batch"])
@pytest.mark.parametrize("acoustic", [False, True], ids=["elastic", "acoustic"])
def test_replays_mix_with_runs_of_other_descriptors(acoustic, replayed):
    print(f"mixed descriptors acoustic={acoustic} replayed={replayed}", flush=True)
    dev = bx.Device(0)

    def state():
        cfg, q0 = random_acoustic((3, 2), 4, 3) if acoustic else random_elastic((2, 1, 2), 4, 3)
        src = dict(cfg["src"], t0=6 * cfg["dt"], f0=0.02 / cfg["dt"])
        cfg["src"] = src
        s = W.upload(dev, cfg, bx.FP64)
        b = bx.Batch(dev, [s])
        # the subdomain's own source from here on
        s.set_source(src["elem"], src["weights"], [3.0 * a for a in src["amp"]],
                     2.3 * src["f0"], src["t0"])
        s.set_fields(q0, 0.0, cfg["dt"])
        return s, b

    sub, batch = state()
    ref, rbatch = state()
    own, other = (sub.step, batch.step) if replayed == "subdomain" else (batch.step, sub.step)
    rown, rother = (ref.step, rbatch.step) if replayed == "subdomain" else (rbatch.step, ref.step)
    g = Capture(dev, own)
    for turn in range(6):
        g.launch()
        rown()
        if turn % 3 != 1:
            other(1 + turn % 2)
            rother(1 + turn % 2)
        np.testing.assert_array_equal(sub.download(), ref.download())
    g.close()
    for x in (batch, rbatch, sub, ref):
        x.close()
    dev.close()
