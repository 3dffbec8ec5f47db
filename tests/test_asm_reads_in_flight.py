"""tinytorch_amd/csrc/check_asm_hazards.py follows the LDS reads that an asm statement leaves in flight: small listings, good and bad.  (The kernels' own
are scanned by test_asm_hazards.py.)  Runs on the CPU."""
import os
import subprocess
import sys

import pytest

CSRC = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "tinytorch_amd", "csrc")

STREAM = """kernel:
\t;;#ASMSTART
\tds_read_b128 v[224:227], v1
\tds_read_b128 v[228:231], v1 offset:16
\t;;#ASMEND
.LBB0_1:
%s
\t;;#ASMSTART
\ts_waitcnt lgkmcnt(1)
\tv_mfma_f32_32x32x16_bf16 v[0:15], v[224:227], v[96:99], v[0:15]
\tds_read_b128 v[224:227], v1
\ts_waitcnt lgkmcnt(%d)
\tv_mfma_f32_32x32x16_bf16 v[0:15], v[228:231], v[96:99], v[0:15]
\tds_read_b128 v[228:231], v1 offset:16
\t;;#ASMEND
\ts_cbranch_scc1 .LBB0_1
%s
\tv_mov_b32_e32 v224, v0
\ts_endpgm
.Lfunc_end0:
"""
WAIT = "\ts_waitcnt lgkmcnt(0)"


@pytest.mark.parametrize("between,count,behind,finding", [
    ("\tv_mov_b32_e32 v82, v83", 1, WAIT, None),
    ("\tds_write_b32 v1, v2", 1, WAIT, None),                       # one more operation: the waits only cover more
    (WAIT + "\n\tv_mov_b32_e32 v230, 0", 1, WAIT, None),
    ("\tv_mov_b32_e32 v230, 0", 1, WAIT, "v_mov_b32_e32 v230"),      # a copy or a spill of the compiler's
    ("\tscratch_store_dwordx2 off, v[226:227], off", 1, WAIT, "scratch_store"),
    ("\ts_waitcnt lgkmcnt(1)\n\tv_mov_b32_e32 v228, 0", 1, WAIT, "v_mov_b32_e32 v228"),
    ("\ts_load_dword s4, s[0:1], 0x0\n\ts_waitcnt lgkmcnt(2)\n\tv_mov_b32_e32 v224, 0", 1, WAIT, "v_mov_b32_e32 v224"),  # scalar loads do not count
    ("", 2, WAIT, "v_mfma"),                                        # a statement's own wait that covers too little
    ("", 1, "", "v_mov_b32_e32 v224"),                              # behind the loop
    ("\tds_read_b32 v3, v2\n\ts_barrier\n" + WAIT, 1, WAIT, "s_barrier"),
    ("\tds_read_b32 v3, v2\n" + WAIT + "\n\ts_barrier", 1, WAIT, None),
    ("\ts_barrier", 1, WAIT, None),                                 # the stream's own reads may cross one
])
def test_the_checker_follows_reads_in_flight(tmp_path, between, count, behind, finding):
    f = tmp_path / "stream.s"
    f.write_text(STREAM % (between, count, behind))
    r = subprocess.run([sys.executable, os.path.join(CSRC, "check_asm_hazards.py"), str(f)], capture_output=True, text=True)
    assert r.returncode == (finding is not None), r.stdout
    assert finding is None or finding in r.stdout


def test_the_checker_follows_code_that_is_out_of_line(tmp_path):
    f = tmp_path / "aside.s"
    text = "kernel:\n\t;;#ASMSTART\n\tds_read_b32 v9, v1\n\ts_cbranch_scc0 .Lm\n.Le:\n\t.subsection 1\n.Lm:\n%s\ts_branch .Le\n\t.subsection 0\n\t;;#ASMEND\n\ts_waitcnt lgkmcnt(0)\n\ts_endpgm\n.Lfunc_end0:\n"
    tool = os.path.join(CSRC, "check_asm_hazards.py")
    for body, rc in (("\tv_mov_b32_e32 v8, 0\n", 0), ("\tv_mov_b32_e32 v9, 0\n", 1)):
        f.write_text(text % body)
        assert subprocess.run([sys.executable, tool, str(f)], capture_output=True).returncode == rc
