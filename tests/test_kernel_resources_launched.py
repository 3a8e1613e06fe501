"""Registers of the node-parallel stage kernels that launches run, read from
the compiler's resource report for gfx950 (CPU only): no scratch, and the
wavefronts per SIMD that their measured rates rest on.  The FP32 kernel of
N = 6 (six wavefronts a block, four blocks a CU) needs at most 72 vector and
96 scalar registers: past either an 18^3 stage takes 77 us instead of 58."""
import os
import re
import shutil
import subprocess

import pytest

from bfam_amd import build as B

PREC = {"fp32": "IfffLb0EEE", "fp32_rhs": "IdffLb0EEE", "fp64": "IdddLb0EEE"}
# (order, precision) -> elements per block, task split over blocks, wavefronts
# per SIMD by registers
LAUNCHED = {(3, "fp32"): (1, 1, 6), (4, "fp32"): (1, 1, 6), (5, "fp32"): (1, 1, 7),
            (6, "fp32"): (1, 0, 7), (7, "fp32"): (1, 0, 6),
            (3, "fp32_rhs"): (1, 1, 5), (4, "fp32_rhs"): (1, 1, 4), (5, "fp32_rhs"): (1, 1, 5),
            (6, "fp32_rhs"): (1, 0, 6), (7, "fp32_rhs"): (1, 0, 6),
            (3, "fp64"): (2, 1, 3), (4, "fp64"): (1, 1, 4), (5, "fp64"): (1, 1, 4),
            (6, "fp64"): (1, 0, 4), (7, "fp64"): (1, 0, 4)}


@pytest.fixture(scope="module")
def report(tmp_path_factory):
    if shutil.which("hipcc") is None:
        pytest.skip("hipcc not found")
    out = tmp_path_factory.mktemp("ru") / "stage_elastic.o"
    src = os.path.join(B.CSRC, "device", "stage_elastic.hip")
    p = subprocess.run(["hipcc"] + B.HIPFLAGS + B.INCS +
                       ["-c", src, "-o", str(out), "-Rpass-analysis=kernel-resource-usage"],
                       capture_output=True, text=True)
    assert p.returncode == 0, p.stderr[-2000:]
    rep = {}
    for blk in p.stderr.split("Function Name: ")[1:]:
        def get(key):
            return int(re.search(key + r": (\d+)", blk).group(1))

        rep[blk.split()[0]] = {"sgpr": get("TotalSGPRs"), "vgpr": get("VGPRs"),
                               "scratch": get(r"ScratchSize \[bytes/lane\]"),
                               "waves": get(r"Occupancy \[waves/SIMD\]")}
    return rep


@pytest.mark.parametrize("N,prec", sorted(LAUNCHED))
def test_launched_kernel(report, N, prec):
    epb, split, waves = LAUNCHED[(N, prec)]
    key = f"elastic_stage_kernelILi{N}ELi{epb}ENS_4Prec{PREC[prec]}Lb{split}E"
    hits = [v for k, v in report.items() if key in k]
    assert len(hits) == 1, key
    r = hits[0]
    assert r["scratch"] == 0 and r["waves"] >= waves, r
    if (N, prec) == (6, "fp32"):
        assert r["vgpr"] <= 72 and r["sgpr"] <= 96, r
