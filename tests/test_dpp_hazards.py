"""The lane-broadcast hazard check that the build runs on its library
(laplace-fmm_amd/csrc/check_dpp.py): finds a write too close to a broadcast, also
around a loop and through EXEC, counts wait states, and finds nothing in the
built library.  Listings only; nothing here is run on a GPU."""
import importlib.util
import os
import re
import subprocess
import sys

import pytest

from conftest import ROOT

CSRC = os.path.join(ROOT, "laplace-fmm_amd", "csrc")
spec = importlib.util.spec_from_file_location("check_dpp", os.path.join(CSRC, "check_dpp.py"))
check_dpp = importlib.util.module_from_spec(spec)
spec.loader.exec_module(check_dpp)

READ = "v_fmac_f64_dpp v[0:1], v[4:5], v[6:7] row_newbcast:3 row_mask:0xf bank_mask:0xf"
OTHER = "v_add_f64 v[10:11], v[12:13], v[14:15]"


def hazards(lines):
    """lines: instructions; a branch names the line it goes to as 'op @line'."""
    out = ["0000000000001000 <k>:"]
    for i, text in enumerate(lines):
        op, _, to = text.partition(" @")
        target = " <k+0x%x>" % (8 * int(to)) if to else ""
        out.append("\t%s // %012X: 00000000%s" % (op, 0x1000 + 8 * i, target))
    return list(check_dpp.Code(out).hazards())


@pytest.mark.parametrize("write", ["v_mov_b32_e32 v5, v9", "v_mov_b64_e32 v[4:5], v[8:9]", "v_accvgpr_read_b32 v4, a3",
                                   "v_permlane32_swap_b32_e32 v9, v4"])
def test_write_just_before(write):
    assert len(hazards([write, READ])) == 1
    assert len(hazards([write, OTHER, READ])) == 1
    assert len(hazards([write, "s_nop 0", READ])) == 1
    assert hazards([write, OTHER, OTHER, READ]) == []
    assert hazards([write, "s_nop 1", READ]) == []


def test_other_registers_and_loads():
    assert hazards(["v_mov_b32_e32 v6, v9", "v_mov_b32_e32 v0, v9", READ]) == []
    assert hazards(["ds_read_b64 v[4:5], v20", "s_waitcnt lgkmcnt(0)", READ]) == []
    assert hazards(["global_load_dwordx2 v[4:5], v[20:21], off", "v_cmp_gt_i32_e32 vcc, v4, v5", READ]) == []


def test_around_a_loop():
    loop = [READ, OTHER, OTHER, "v_mov_b32_e32 v4, v9", "s_cbranch_scc1 65532 @0", "s_endpgm"]
    assert len(hazards(loop)) == 1
    assert hazards(loop[:4] + [OTHER] + loop[4:]) == []
    # what only falls through is not reached past an unconditional branch
    assert hazards(["v_mov_b32_e32 v4, v9", "s_branch 3 @3", "s_endpgm", OTHER, READ]) == []
    assert len(hazards(["s_branch 1 @2", "v_mov_b32_e32 v4, v9", READ])) == 1


def test_exec():
    assert len(hazards(["v_cmpx_gt_i32_e32 v4, v9"] + [OTHER] * 4 + [READ])) == 1
    assert hazards(["v_cmpx_gt_i32_e32 v4, v9"] + [OTHER] * 5 + [READ]) == []


@pytest.mark.skipif(not os.path.exists(check_dpp.OBJDUMP), reason="needs llvm-objdump")
def test_built_library(lfmm):
    lfmm.lib()  # builds if nothing is built
    r = subprocess.run([sys.executable, check_dpp.__file__, os.path.join(ROOT, "laplace-fmm_amd", "_build", "liblfmm.so")],
                       capture_output=True, text=True, timeout=300)
    reads, hits = map(int, re.search(r"check_dpp: (\d+) reads, (\d+) hazards", r.stdout).groups())
    assert r.returncode == 0 and reads > 50000 and hits == 0, r.stdout
