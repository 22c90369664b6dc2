"""Registers of the timed one-wave kernels at beams up to 256: at most 80, six
waves per SIMD, where LDS lets a CU hold 24 queries (d 128 / degree 32, d 96 /
degree 32 and 16, padded dimension 64, padded 128 up to d 96).  With one more
a CU holds 20, and a batch between the two sizes takes a second round."""
from __future__ import annotations

import os
import re
import subprocess

import pytest

from test_kernel_resources import HIPCC, ROOT, _flags


@pytest.mark.skipif(not os.path.exists(HIPCC), reason="hipcc not installed")
def test_six_waves_per_simd(tmp_path):
    src = os.path.join(ROOT, "flashgann_amd", "csrc", "fg_shapes.hip")
    procs = []
    for shape in range(5):
        out = tmp_path / f"{shape}.s"
        procs.append((out, subprocess.Popen([HIPCC, *_flags(), f"-DFG_SHAPE={shape}", "--cuda-device-only", "-S", "-o",
                                             str(out), src], stderr=subprocess.DEVNULL)))
    seen = {}
    for out, p in procs:
        assert p.wait(timeout=900) == 0
        # <WT, DPL, DIM_T, DEG_T, COUNT, PROF, BIG, NW>
        for name, vgprs in re.findall(r"\.amdhsa_kernel (\S+ELb0ELb0ELb0ELi1EEE\S+)\n.*?\.amdhsa_next_free_vgpr (\d+)",
                                      out.read_text(), re.S):
            seen[name] = int(vgprs)
    assert len(seen) == 5 and all(v <= 80 for v in seen.values()), seen
