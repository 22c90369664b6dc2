"""Properties of the search kernels' compiled code that their speed rests on and
that no result shows."""
from __future__ import annotations

import os
import re
import subprocess

import pytest

from test_kernel_resources import HIPCC, ROOT, _flags

pytestmark = pytest.mark.skipif(not os.path.exists(HIPCC), reason="hipcc not installed")


@pytest.fixture(scope="module")
def asm(tmp_path_factory):
    """Device assembly of shape classes 0 .. 4 and 6, compiled in parallel."""
    src = os.path.join(ROOT, "flashgann_amd", "csrc", "fg_shapes.hip")
    tmp, procs = tmp_path_factory.mktemp("asm"), {}
    for shape in (6, 0, 1, 2, 3, 4):
        out = tmp / f"{shape}.s"
        procs[shape] = (out, subprocess.Popen([HIPCC, *_flags(), f"-DFG_SHAPE={shape}", "--cuda-device-only", "-S",
                                               "-o", str(out), src], stderr=subprocess.DEVNULL))
    for _, p in procs.values():
        assert p.wait(timeout=900) == 0
    return {shape: out.read_text() for shape, (out, _) in procs.items()}


def test_six_waves_per_simd(asm):
    """Registers of the timed one-wave kernels at beams up to 256: at most 80, six
    waves per SIMD, where LDS lets a CU hold 24 queries (d 128 / degree 32, d 96 /
    degree 32 and 16, padded dimension 64, padded 128 up to d 96).  With one more
    a CU holds 20, and a batch between the two sizes takes a second round."""
    seen = {}
    for shape in range(5):
        # <WT, DPL, DIM_T, DEG_T, COUNT, PROF, BIG, NW>
        for name, vgprs in re.findall(r"\.amdhsa_kernel (\S+ELb0ELb0ELb0ELi1EEE\S+)\n.*?\.amdhsa_next_free_vgpr (\d+)",
                                      asm[shape], re.S):
            seen[name] = int(vgprs)
    assert len(seen) == 5 and all(v <= 80 for v in seen.values()), seen


def test_code_loads_stay_whole(asm):
    """The wide kernels (padded dimension 512 and up) read neighbour codes 16 bytes
    at a time where the row layout allows it.  A code is 64 to 256 bytes per lane:
    read word by word, each load touches 64 cache lines for 4 bytes of each, and a
    full launch at padded dimension 512 took up to 20% longer."""
    bodies = re.findall(r"^_ZN3fgk16fg_search_kernelI\w+ELi(\d)EEEv\w+:(.*?)\.Lfunc_end", asm[6], re.S | re.M)
    assert len(bodies) == 18
    for waves, body in bodies:
        # 16- and 32-word spans (4 + 8 loads): once for a single expander, then
        # for each of a wave's four, two or one sub-rounds of several
        least = 12 * (1 + 4 // int(waves))
        assert len(re.findall(r"\bglobal_load_dwordx4\b", body)) >= least, waves
