"""Host field arrays to and from the device (set_fields, download, rhs), in
one piece by the calling thread, in two by two threads and in many by eight,
with a ragged last piece: every value arrives, rounded once to the state
type, and a state survives the way there and back."""
import numpy as np
import pytest

import bfam_amd as bx
import bfam_amd.workloads as W
from util import random_acoustic, random_elastic

pytestmark = pytest.mark.gpu

# (dims, N): 21 KB to 190 MB of FP64 state
SIZES = [((1, 2, 1), 3), ((4, 3, 3), 4), ((7, 5, 3), 5), ((9, 8, 7), 6), ((17, 13, 11), 7),
         ((19, 17, 15), 7)]


@pytest.mark.parametrize("dims,N", SIZES)
@pytest.mark.parametrize("prec", [bx.FP64, bx.FP64_PLAIN, bx.FP32_RHS, bx.FP32])
def test_round_trip(dims, N, prec):
    cfg, _ = random_elastic(dims, N, seed=1, src=False)
    K, Np = cfg["mesh"].K, cfg["mesh"].Np
    q0 = np.random.default_rng(2).standard_normal((9, K * Np))
    dev = bx.Device(0)
    sub = W.upload(dev, cfg, prec)
    for q in (q0, q0[::-1]):
        sub.set_fields(q, 0.0, cfg["dt"])
        want = q.astype(np.float32).astype(np.float64) if prec == bx.FP32 else q
        assert np.array_equal(sub.download(), want)
    sub.close()
    dev.close()


def test_download_follows_the_steps():
    """the copy out waits for the stages launched before it"""
    cfg, q0 = random_elastic((9, 9, 9), 6, seed=3)
    dev = bx.Device(0)
    sub = W.upload(dev, cfg, bx.FP32)
    sub.set_fields(q0, 0.0, cfg["dt"])
    sub.step(3)
    dev.sync()
    a = sub.download()
    sub.set_fields(q0, 0.0, cfg["dt"])
    for _ in range(15):
        sub.stage()
    assert np.array_equal(sub.download(), a)
    sub.close()
    dev.close()


@pytest.mark.parametrize("dims,N", [((3, 2, 2), 4), ((12, 12, 12), 7)])
def test_rhs_matches_the_strided_copy(dims, N):
    cfg, q0 = random_elastic(dims, N, seed=5)
    dev = bx.Device(0)
    sub = W.upload(dev, cfg, bx.FP64)
    sub.set_fields(q0, 0.0, cfg["dt"])
    assert np.array_equal(sub.rhs(0.1), sub.rhs_noalloc(0.1))
    sub.close()
    dev.close()


def test_acoustic_round_trip():
    cfg, q0 = random_acoustic((300, 211), 5, seed=6)
    dev = bx.Device(0)
    sub = W.upload(dev, cfg, bx.FP64)
    sub.set_fields(q0, 0.0, cfg["dt"])
    assert np.array_equal(sub.download(), q0)
    sub.close()
    dev.close()
