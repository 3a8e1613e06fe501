"""The transfer kernel at every pair of orders and of state types: one
destination element kept, one a child of its source, one coarsened from eight
sources of two orders, against the oracle's transfer of the same state: the
arithmetic is FP64 in sums of at most 8^3 * 8 terms (1e-12 of the largest
value), each value rounded once to its state type (2^-24 for FP32)."""
import numpy as np
import pytest

import bfam_amd as bx
import bfam_amd.workloads as W
import oracle
from util import random_elastic

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("sp,dp", [(bx.FP64, bx.FP64), (bx.FP32, bx.FP32), (bx.FP64, bx.FP32),
                                   (bx.FP32, bx.FP64)])
@pytest.mark.parametrize("Nd", [3, 4, 5, 6, 7])
@pytest.mark.parametrize("Ns", [3, 4, 5, 6, 7])
def test_order_pairs(Ns, Nd, sp, dp):
    dev = bx.Device(0)
    Nt = 10 - Ns  # the other source's order
    src, qs = [], []
    for s, (N, n) in enumerate(((Ns, (2, 2, 2)), (Nt, (2, 1, 1)))):
        cfg, q0 = random_elastic(n, N, seed=s, src=False)
        sub = W.upload(dev, cfg, sp)
        sub.set_fields(q0, 0.0, cfg["dt"])
        src.append(sub)
        qs.append(sub.download())
    cfg, _ = random_elastic((3, 1, 1), Nd, seed=9, src=False)
    dst = W.upload(dev, cfg, dp)
    m = {"num_dst": 3, "num_coarse_dst": 1,
         "dst_to_adapt_flags": [bx.FLAG_REFINE, bx.FLAG_COARSEN, bx.FLAG_SAME],
         "dst_to_dst_chld_id": [5, 0, 0], "dst_to_src_subd_id": [0, -1, 0],
         "dst_to_src_elem_id": [3, 0, 6],
         "coarse_dst_to_src_chld_id": list(range(8)),
         "coarse_dst_to_src_subd_id": [0, 0, 1, 0, 0, 1, 0, 0],
         "coarse_dst_to_src_elem_id": [0, 1, 0, 2, 4, 1, 5, 7],
         "dst_subd": [0, 0, 0], "dst_elem": [1, 2, 0]}
    bx.transfer_fields(m, src, [dst], cfg["dt"])
    got = dst.download()
    for s in src + [dst]:
        s.close()
    dev.close()
    want = oracle.transfer(m, qs, [Ns, Nt], [3], [Nd])[0]
    tol = 1e-12 + (2.0 ** -24 if dp == bx.FP32 else 0.0)
    assert np.abs(got - want).max() <= tol * np.abs(want).max()
