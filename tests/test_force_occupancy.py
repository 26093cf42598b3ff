"""Waves per compute unit that the force kernels for MHD fields and unequal smoothing lengths leave room for, from
the registers and the LDS of the built kernels (CPU): 512 registers per lane and SIMD in steps of 8, 160 KiB of LDS
in steps of 1,280 bytes. A few registers or a few hundred bytes more cost a wave per SIMD."""
from __future__ import annotations

import os
import re
import shutil
import subprocess

import pytest

from spearhed_amd import capi

LLVM = "/opt/rocm/llvm/bin"


@pytest.fixture(scope="module")
def resources(tmp_path_factory):
    """(registers, LDS bytes, spilled registers) of each kernel by its mangled name."""
    if not os.path.exists(os.path.join(LLVM, "llvm-objdump")):
        pytest.skip("no llvm-objdump")
    if not os.path.exists(capi.LIB_PATH):
        pytest.skip("library not built")
    tmp = tmp_path_factory.mktemp("forces")
    lib = shutil.copy(capi.LIB_PATH, tmp)  # the code objects are written beside it
    subprocess.run([os.path.join(LLVM, "llvm-objdump"), "--offloading", lib], check=True, capture_output=True)
    out = {}
    for f in sorted(os.listdir(tmp)):
        if "gfx950" in f:
            notes = subprocess.run([os.path.join(LLVM, "llvm-readelf"), "--notes", str(tmp / f)], check=True,
                                   capture_output=True, text=True).stdout
            for k in notes.split("- .agpr_count:")[1:]:
                num = [int(re.search(rf"\.{key}:\s+(\d+)", k).group(1))
                       for key in ("vgpr_count", "group_segment_fixed_size", "vgpr_spill_count")]
                out[re.search(r"\.name:\s+(\S+)", k).group(1)] = num
    return out


# chunk, balance: waves per compute unit
@pytest.mark.parametrize("chunk,bal,waves", [(64, 0, 20), (64, 1, 16), (128, 0, 12), (128, 1, 10)])
def test_waves_of_the_general_h_force_pass(resources, chunk, bal, waves):
    # k_forces<chunk, *, MHD, *, bal, 27 cells, no persistent grid, not one h>
    names = [n for n in resources if re.match(rf"_ZN3sph8k_forcesILi{chunk}ELb[01]ELb1ELi\w+ELi{bal}ELi1ELb0ELb0E", n)]
    assert len(names) == 8  # two precisions; three smoothing kernels or any
    for n in names:
        regs, lds, spilled = resources[n]
        fit = min(4 * min(8, 512 // (-(-regs // 8) * 8)), 163840 // (-(-lds // 1280) * 1280))
        assert fit >= waves and spilled == 0, f"{n}: {regs} registers, {lds} bytes, {spilled} spilled: {fit} waves"
