"""The head_dim-128 dq kernel's loop reloads no spilled register: a reload's wait in front of a tile's requests is one for the tiles in flight
too.  Looked up in the compiler's listing, on the CPU."""
import os
import re

import pytest

from test_asm_hazards import HIPCC, listing


@pytest.mark.skipif(not os.path.exists(HIPCC), reason="hipcc not installed")
def test_no_reload_between_the_streams_of_dq(tmp_path):
    out = str(tmp_path / "d128.s")
    assert listing("sdpa_backward_d128.hip", out).returncode == 0
    kernels = re.findall(r"^(_ZN\S*backward_dq128_kernel\S*):(.*?)^\.Lfunc_end", open(out).read(), re.M | re.S)
    assert len(kernels) == 4
    for name, body in kernels:
        streams = [m for m in re.finditer(r";#ASMSTART.*?;#ASMEND", body, re.S) if m.group().count("v_mfma") >= 24]
        assert len(streams) == 4, name
        assert "scratch_" not in body[streams[0].start():streams[-1].end()], name
