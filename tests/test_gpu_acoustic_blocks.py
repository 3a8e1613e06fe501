"""Acoustic stage: a subdomain of few tasks launches blocks of one wavefront,
others blocks of up to 256 threads, and one of several members reads its tasks
from the table: a member alone and the same member in a batch agree, at one
element, remainders of both block sizes and around the 128 tasks where the
block size changes.  The forms compute an element alike up to the rounding of
a differently contracted sum: 5 steps of 5 stages, some 100 operations a node
and stage on states of order 1, so 25 * 100 * eps bounds the difference."""
import numpy as np
import pytest

import bfam_amd as bx
import bfam_amd.workloads as W
from util import random_acoustic

pytestmark = pytest.mark.gpu


def _edges(N):
    e = 256 // (N + 1) ** 2
    return [(1, 1), (7, 3), (e, 128), (e + 1, 128)]


@pytest.mark.parametrize("prec", [bx.FP64, bx.FP32, bx.FP32_RHS])
@pytest.mark.parametrize("N,n", [(N, n) for N in (1, 2, 4, 7, 8) for n in _edges(N)])
def test_alone_equals_batched(N, n, prec):
    dev = bx.Device(0)
    cfg, q0 = random_acoustic(n, N, seed=N)
    cfg2, p0 = random_acoustic((5, 4), N, seed=N + 1)
    sub, other = W.upload(dev, cfg, prec), W.upload(dev, cfg2, prec)
    sub.set_fields(q0, 0.0, cfg["dt"])
    sub.step(5)
    alone = sub.download()
    sub.set_fields(q0, 0.0, cfg["dt"])
    other.set_fields(p0, 0.0, cfg2["dt"])
    b = bx.Batch(dev, [other, sub])
    b.step(5)
    got = sub.download()
    b.close()
    sub.close()
    other.close()
    dev.close()
    eps = np.finfo(np.float64 if prec == bx.FP64 else np.float32).eps
    assert np.isfinite(alone).all() and np.abs(alone - q0).max() > 0
    assert np.abs(got - alone).max() <= 2500 * eps * np.abs(alone).max()
