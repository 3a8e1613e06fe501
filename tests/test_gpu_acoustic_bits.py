"""Acoustic stage, to the last bit.

The update d = A d + dt L, q = q + B d has one order of rounding whatever the
block form: A d is rounded, dt L is added to it with one rounding, and B d to
q with one.  The rates are the device's own (no source: they do not depend on
time), so the expected state follows exactly, in rational arithmetic.

The block forms (one wavefront, up to 256 threads, tasks from the table in a
batch) differ in how elements are dealt to threads only: a member alone and
the same member in a batch agree to the last bit."""
from fractions import Fraction as Q

import numpy as np
import pytest

import bfam_amd as bx
import bfam_amd.workloads as W
from util import random_acoustic

pytestmark = pytest.mark.gpu


def _q(a):
    return np.array([Q(float(x)) for x in np.ravel(a)], dtype=object)


def _round(v, T):
    """Rationals to the nearest T; to float32 by way of 64 bits of mantissa, so
    that a second rounding could differ only within 2^-40 of a tie."""
    if T is np.float64:
        return np.array([float(x) for x in v])
    hi = np.array([float(x) for x in v])
    lo = np.array([float(x - Q(h)) for x, h in zip(v, hi)])
    return (hi.astype(np.longdouble) + lo.astype(np.longdouble)).astype(np.float32)


@pytest.mark.parametrize("prec", [bx.FP32_RHS, bx.FP64, bx.FP32])
@pytest.mark.parametrize("N,n", [(1, (3, 1)), (2, (5, 2)), (4, (3, 2)), (8, (2, 1))])
def test_update_rounds_in_one_order(N, n, prec):
    print(f"acoustic update N={N} n={n} prec={prec}", flush=True)
    TS = np.float32 if prec == bx.FP32 else np.float64  # state
    TR = np.float64 if prec == bx.FP64 else np.float32  # rates
    rebuilt = prec != bx.FP32_RHS  # B d of the last stage is taken as q - q_before
    A, B, _ = bx.lsrk_init()
    dev = bx.Device(0)
    cfg, q0 = random_acoustic(n, N, seed=N)
    cfg.pop("src")
    sub, other = W.upload(dev, cfg, prec), W.upload(dev, cfg, prec)
    sub.set_fields(q0, 0.0, cfg["dt"])
    q = [sub.download().astype(TS).ravel()]
    d = np.zeros(q0.size, TR)
    for s in range(5):
        rate = sub.rhs(0.0).astype(TR).ravel()
        a = A[s]
        if rebuilt and s:
            a = A[s] / B[s - 1]
            d = q[-1] - q[-2]
        ad = _round(_q(d) * Q(float(TR(a))), TR)
        d = _round(_q(rate) * Q(float(TR(cfg["dt"]))) + _q(ad), TR)
        q.append(_round(_q(d) * Q(float(TS(B[s]))) + _q(q[-1]), TS))
        sub.stage()
        np.testing.assert_array_equal(sub.download().astype(TS).ravel(), q[-1])
    b = bx.Batch(dev, [sub, other])
    for x in (sub, other):
        x.set_fields(q0, 0.0, cfg["dt"])
    b.step(1)
    for x in (sub, other):
        np.testing.assert_array_equal(x.download().astype(TS).ravel(), q[-1])
    b.close()
    sub.close()
    other.close()
    dev.close()


def _edges(N):
    e = 256 // (N + 1) ** 2
    return [(1, 1), (7, 3), (e, 128), (e + 1, 128)]


@pytest.mark.parametrize("prec", [bx.FP64, bx.FP32, bx.FP32_RHS])
@pytest.mark.parametrize("N,n", [(N, n) for N in range(1, 9) for n in _edges(N)])
def test_alone_and_batched_to_the_last_bit(N, n, prec):
    print(f"acoustic alone, batched N={N} n={n} prec={prec}", flush=True)
    dev = bx.Device(0)
    cfg, q0 = random_acoustic(n, N, seed=N)
    cfg2, p0 = random_acoustic((5, 4), N, seed=N + 1)
    sub, other = W.upload(dev, cfg, prec), W.upload(dev, cfg2, prec)
    sub.set_fields(q0, 0.0, cfg["dt"])
    rate = sub.rhs(0.1)
    sub.step(5)
    alone = sub.download()
    sub.set_fields(q0, 0.0, cfg["dt"])
    other.set_fields(p0, 0.0, cfg2["dt"])
    b = bx.Batch(dev, [other, sub])
    np.testing.assert_array_equal(b.rhs(0.1)[1], rate)
    b.step(5)
    np.testing.assert_array_equal(sub.download(), alone)
    assert np.isfinite(alone).all() and np.abs(alone - q0).max() > 0
    b.close()
    sub.close()
    other.close()
    dev.close()
