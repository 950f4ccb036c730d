"""The kernels of large FP64 domains and batches (the split ones) and the
register-tile SOR sweeps keep everything in registers and LDS, vector and
scalar, and fit the blocks per CU that their times were measured at.  Reads the
compiler's resource report that the build writes next to the library."""
import os
import re

import pytest

from conftest import ROOT

REPORT = os.path.join(ROOT, "swm_amd", "libswmgpu.resources.txt")
STEP = "_ZN3swm17step_kernel_splitIdLi1ELi%dELi32ELi8ELb1EEEvNS_3DynIT_EE"
BATCH = "_ZN3swm18batch_kernel_splitIdLi1ELi%dELi32ELi8EEEvPKNS_6MemberIT_EEPKNS_10MemberStepEPKii"
SOR = "_ZN3swm8sor_rowsI%sLi%dELi%dEEEvNS_11SorRowsArgsIT_EEPKS2_PS2_"
LDS = 160 * 1024     # of a CU
# kernel: threads of a block, blocks that a CU must hold
KERNELS = {STEP % 0: (256, 6), STEP % 1: (256, 5), STEP % 2: (256, 4),
           BATCH % 0: (256, 6), BATCH % 1: (256, 5), BATCH % 2: (256, 4)}
for t in "df":
    KERNELS.update({SOR % (t, 8, 4): (512, 1), SOR % (t, 16, 4): (1024, 1), SOR % (t, 8, 6): (512, 2)})


@pytest.fixture(scope="module")
def report():
    if not os.path.exists(REPORT):
        pytest.skip("no resource report: run __graft_entry__.build()")
    out = {}
    for block in open(REPORT).read().split("remark: Function Name: ")[1:]:
        get = lambda key: int(re.search(key + r": (\d+)", block).group(1))
        out[block.split()[0]] = {"scratch": get(r"ScratchSize \[bytes/lane\]"), "vspill": get("VGPRs Spill"),
                                 "sspill": get("SGPRs Spill"), "vgpr": get(r"\bVGPRs"),
                                 "lds": get(r"LDS Size \[bytes/block\]")}
    return out


@pytest.mark.parametrize("kernel", KERNELS)
def test_kernel_fits(report, kernel):
    threads, blocks = KERNELS[kernel]
    r = report[kernel]
    assert r["scratch"] == r["vspill"] == r["sspill"] == 0, r
    waves = 512 // (-(-r["vgpr"] // 8) * 8)      # per SIMD, by the vector registers
    assert waves * 4 * 64 >= threads * blocks and r["lds"] * blocks <= LDS, r
