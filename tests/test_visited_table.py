"""The visited table of each search shape, on the host: it has a slot to spare
for the most keys a search can insert, it is never smaller than it has to be
for a CU to hold its queries, and a batch that fits the device anyway has the
roomiest one."""
from __future__ import annotations

import os
import subprocess

import pytest

from test_kernel_resources import HIPCC, ROOT, _flags

PROGRAM = r"""
#include "fg_kernel.hpp"
using namespace fgk;
int main() {
    int bad = 0;
    for (uint32_t padded = 64; padded <= 2048; padded *= 2)
        for (uint32_t degree : {1u, 16u, 32u, 33u, 64u, 96u})
            for (uint32_t beam = 1; beam <= 1024; ++beam) {
                const uint32_t pb = effective_sort_beam(beam), b = visited_buckets(padded, padded, pb, beam, degree);
                const uint32_t lo = visited_buckets_min(beam, degree), hi = visited_buckets_roomy(beam, degree);
                bool ok = b >= lo && b <= hi && 4u * b > visited_keys_max(beam, degree);
                const uint32_t m1 = padded <= 128 ? 32 : padded == 256 ? 16 : 11, m2 = padded <= 128 ? 16 : padded == 256 ? 10 : 6;
                const auto one = [&](uint32_t n) { return std::min(m1, lds_groups(lds_layout(padded, padded, pb, n).total)); };
                const auto two = [&](uint32_t n) { return std::min(m2, lds_groups(lds_layout(padded, padded, pb, n).total_team)); };
                ok = ok && one(b) == one(lo) && two(b) == two(lo);
                ok = ok && (b == hi || one(b + 1) < one(lo) || two(b + 1) < two(lo));
                if (!ok) std::printf("padded %u degree %u beam %u: %u of %u .. %u\n", padded, degree, beam, b, lo, hi);
                bad += !ok;
            }
    // a whole number of workgroups leaves room for the roomiest table here
    bad += visited_buckets(600, 1024, 1024, 1024, 32) != visited_buckets_roomy(1024, 32);
    // 8,960 bytes: seven units of LDS, 18 to a CU
    bad += lds_groups(8960) != 18 || lds_groups(8961) != 16;
    return bad ? 1 : 0;
}
"""


@pytest.mark.skipif(not os.path.exists(HIPCC), reason="hipcc not installed")
def test_visited_table_sizes(tmp_path):
    src = tmp_path / "table.hip"
    src.write_text(PROGRAM)
    exe = tmp_path / "table"
    subprocess.run([HIPCC, *_flags(), "-I", os.path.join(ROOT, "flashgann_amd", "csrc"), "-o", str(exe), str(src)],
                   check=True, capture_output=True, timeout=600)
    r = subprocess.run([str(exe)], timeout=60, capture_output=True, text=True)
    assert r.returncode == 0, r.stdout[:2000]
