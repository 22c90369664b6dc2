"""The wide kernels (padded dimension 512 and up) read neighbour codes 16 bytes
at a time where the row layout allows it.  A code is 64 to 256 bytes per lane:
read word by word, each load touches 64 cache lines for 4 bytes of each, and a
full launch at padded dimension 512 took up to 20% longer."""
from __future__ import annotations

import os
import re
import subprocess

import pytest

from test_kernel_resources import HIPCC, ROOT, _flags


@pytest.mark.skipif(not os.path.exists(HIPCC), reason="hipcc not installed")
def test_code_loads_stay_whole(tmp_path):
    src = os.path.join(ROOT, "flashgann_amd", "csrc", "fg_shapes.hip")
    out = tmp_path / "fg_shape6.s"
    subprocess.run([HIPCC, *_flags(), "-DFG_SHAPE=6", "--cuda-device-only", "-S", "-o", str(out), src], check=True,
                   capture_output=True, timeout=900)
    bodies = re.findall(r"^_ZN3fgk16fg_search_kernelI\w+ELi(\d)EEEv\w+:(.*?)\.Lfunc_end", out.read_text(), re.S | re.M)
    assert len(bodies) == 18
    for waves, body in bodies:
        # 16- and 32-word spans (4 + 8 loads): once for a single expander, then
        # for each of a wave's four, two or one sub-rounds of several
        least = 12 * (1 + 4 // int(waves))
        assert len(re.findall(r"\bglobal_load_dwordx4\b", body)) >= least, waves
