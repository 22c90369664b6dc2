"""Where a wave of the search kernel writes when it has no child to list: the
beam's pad entry, whichever side of the beam its list lies on.  The index is
checked on the host, with 64-bit addresses: on the device a difference taken
modulo 2^32 would still reach the entry, but only through 32-bit LDS
addresses."""
from __future__ import annotations

import os
import subprocess

import pytest

from test_kernel_resources import HIPCC, ROOT, _flags

PROGRAM = r"""
#include "fg_kernel.hpp"
int main() {
    alignas(16) static unsigned char smem[65536];
    int bad = 0;
    for (uint32_t beam = 1; beam <= 1024; beam += beam < 130 ? 1 : 149)
        for (uint32_t dim = 64; dim <= 2048; dim *= 4)
            for (uint32_t degree = 16; degree <= 64; degree *= 2) {
                const uint32_t pb = fgk::effective_sort_beam(beam);
                const fgk::LdsLayout L =
                    fgk::lds_layout(dim, dim, pb, fgk::visited_buckets(dim, dim, pb, beam, degree));
                const uint2 *bp = reinterpret_cast<const uint2 *>(smem + L.beam_off) + 1;
                const uint32_t *pad = reinterpret_cast<const uint32_t *>(bp + pb + 2);
                const fgk::TeamBlock *tb = reinterpret_cast<const fgk::TeamBlock *>(smem + L.total);
                const uint32_t *lists[] = {reinterpret_cast<const uint32_t *>(smem + L.scratch_off), tb->list,
                                           tb->list + 8, tb->list + 16};
                for (const uint32_t *list : lists)
                    bad += &list[fgk::list_spare(list, bp, static_cast<int>(pb))] != pad ? 1 : 0;
                bad += reinterpret_cast<const unsigned char *>(pad + 1) > smem + L.hash_off ? 1 : 0;
            }
    return bad ? 1 : 0;
}
"""


@pytest.mark.skipif(not os.path.exists(HIPCC), reason="hipcc not installed")
def test_spare_index_reaches_the_pad_entry(tmp_path):
    src = tmp_path / "words.hip"
    src.write_text(PROGRAM)
    exe = tmp_path / "words"
    subprocess.run([HIPCC, *_flags(), "-I", os.path.join(ROOT, "flashgann_amd", "csrc"), "-o", str(exe), str(src)],
                   check=True, capture_output=True, timeout=600)
    assert subprocess.run([str(exe)], timeout=60).returncode == 0
