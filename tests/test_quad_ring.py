"""The build's check of the quad-union kernel's register ring (csrc/check_quad_ring.py), on assembly written here: what it
lets pass between the marked blocks and what it does not, also on a way that the text shows after the second mark."""

import os
import subprocess
import sys

import pytest

from conftest import PKG

FIRST, DRAINED, LOOP = (";;#ASMSTART\n; %s\n%s\n;;#ASMEND\n" % x for x in (
    ("ring: first requests", "global_load_dword v84, v1, s[40:41]"), ("ring: drained", "s_waitcnt vmcnt(0)"),
    ("chunks", "v_mfma_f32_4x4x1_16b_f32 v[32:35], v84, v48, v[32:35]")))
KERNEL = ("_Z26ellpack_matmul_quad_kernelILi0EEv: ; @k\n\tglobal_load_dword v90, v0, s[2:3]\n" + FIRST + "\ts_cbranch_scc1 .LBB0_2\n"
          ".LBB0_1:\n" + LOOP + "\t%(inside)s\n\ts_cbranch_scc0 .LBB0_1\n" + DRAINED + "\tv_mov_b32 v85, v1\n\tglobal_store_dword v0, v85, s[2:3]\n\ts_endpgm\n"
          ".LBB0_2:\n\t%(sunk)s\n\ts_branch .LBB0_1\n.Lfunc_end0:\n")
HARMLESS = "v_add_u32 v83, v96, v1 ; not v84"


@pytest.mark.parametrize("inside,sunk,ok", [
    (HARMLESS, "ds_write_b128 v1, v[80:83]", True), ("v_mov_b32 v1, v84", HARMLESS, False), (HARMLESS, "v_accvgpr_write_b32 a0, v95", False),
    ("v_mov_b64 v[94:95], v[2:3]", HARMLESS, False), (HARMLESS, "ds_write_b128 v1, v[81:84]", False), ("global_load_dword v1, v0, s[2:3]", HARMLESS, False),
    (HARMLESS, "scratch_store_dword off, v1, s32", False), (HARMLESS, "s_endpgm", False)])
def test_ring_check(tmp_path, inside, sunk, ok):
    path = tmp_path / "k.s"
    path.write_text(KERNEL % {"inside": inside, "sunk": sunk})
    r = subprocess.run([sys.executable, os.path.join(PKG, "csrc", "check_quad_ring.py"), str(path)], stderr=subprocess.PIPE, text=True)
    assert (r.returncode == 0) == ok, r.stderr


def test_ring_check_needs_the_kernel_and_its_marks(tmp_path):
    path = tmp_path / "k.s"
    for text in ("", KERNEL.replace("ring: drained", "drained") % {"inside": HARMLESS, "sunk": HARMLESS}):
        path.write_text(text)
        assert subprocess.run([sys.executable, os.path.join(PKG, "csrc", "check_quad_ring.py"), str(path)], stderr=subprocess.DEVNULL).returncode != 0
