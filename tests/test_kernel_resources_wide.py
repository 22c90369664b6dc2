"""The kernels of padded dimension 256 use no scratch memory either (see
test_kernel_resources.py)."""
from __future__ import annotations

import os
import re
import subprocess

import pytest

from test_kernel_resources import HIPCC, ROOT, _flags


@pytest.mark.skipif(not os.path.exists(HIPCC), reason="hipcc not installed")
def test_padded_256_kernels_use_no_scratch(tmp_path):
    src = os.path.join(ROOT, "flashgann_amd", "csrc", "fg_shapes.hip")
    out = tmp_path / "fg_shape7.s"
    subprocess.run([HIPCC, *_flags(), "-DFG_SHAPE=7", "--cuda-device-only", "-S", "-o", str(out), src], check=True,
                   capture_output=True, timeout=900)
    sizes = [int(x) for x in re.findall(r"; ScratchSize: (\d+)", out.read_text())]
    assert len(sizes) == 18 and not any(sizes), sizes
