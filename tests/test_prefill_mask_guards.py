"""The pipelined prefill launchers refuse the attnMasks that their instruction streams cannot apply: such a mask would be read as other
bytes than it holds, or left out.  CPU only (nothing is launched; hipcc builds the host program)."""
import os
import shutil
import subprocess

import pytest

from conftest import ROOT

HIPCC = os.environ.get("HIPCC", "/opt/rocm/bin/hipcc")
LIBDIR = os.path.join(ROOT, "tinytorch_amd", "lib")


@pytest.mark.skipif(not (os.path.exists(HIPCC) or shutil.which(HIPCC)), reason="hipcc not installed")
def test_masks_without_streams_are_refused(tmp_path):
    exe = str(tmp_path / "guards")
    r = subprocess.run([HIPCC, "--offload-arch=gfx950", "-O1", "-std=c++17", "-Xclang", "-target-feature", "-Xclang", "-packed-fp32-ops",
                        "-Wno-unused-command-line-argument", "-I" + os.path.join(ROOT, "tinytorch_amd", "csrc"), "-I" + os.path.join(ROOT, "include"),
                        os.path.join(ROOT, "tests", "cpp", "prefill_mask_guards.hip"), "-o", exe, "-L" + LIBDIR, "-lttsdpa", "-Wl,-rpath," + LIBDIR],
                       capture_output=True, text=True)
    assert r.returncode == 0, r.stderr[-2000:]
    env = dict(os.environ, HIP_VISIBLE_DEVICES="-1")  # a call that were not refused must not reach a device
    r = subprocess.run([exe], capture_output=True, text=True, timeout=100, env=env)
    assert r.returncode == 0, r.stdout
