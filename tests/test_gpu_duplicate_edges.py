"""A repeated neighbour anywhere in the codebook is found when the index is
created: a search that took such a codebook for one without repeats would
list the repeated child twice.  The repeat sits in the entry point's row, in
the first or last row, at the ends of the row and around a wave's 64 slots;
empty slots (0xFFFFFFFF) may repeat without being one."""
from __future__ import annotations

import copy

import numpy as np
import pytest

from conftest import small_index

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("degree,pair", [(2, (0, 1)), (31, (0, 30)), (32, (30, 31)), (33, (0, 32)), (64, (0, 63)),
                                         (65, (63, 64)), (96, (31, 95)), (32, None)])
@pytest.mark.parametrize("last", [False, True])
def test_repeated_edge_is_found(gpu_available, degree, pair, last):
    from flashgann_amd import Index
    from oracle import oracle as O
    cb, q, _ = small_index(n=700, nq=12, dim=64, comps=8, degree=degree, kind="unit", config=3)
    cb = copy.copy(cb)
    cb.rows = cb.rows.copy()
    cb.entry = cb.npoints - 1 if last else 0
    lay = cb.layout
    if pair is None:  # empty slots only
        cb.neighbors()[cb.entry, 3:6] = 0xFFFFFFFF
    else:
        i, j = pair
        cb.neighbors()[cb.entry, j] = cb.neighbors()[cb.entry, i]
        words = lay.padded_dim // 32
        codes = cb.rows[:, lay.code_offset:lay.factor_offset].reshape(cb.npoints, degree, words)
        codes[cb.entry, j] = codes[cb.entry, i]
        for k in range(3):
            row = cb.rows[cb.entry, lay.factor_offset + k * degree:]
            row[j] = row[i]
    beam = 64
    ix = Index.from_codebook(cb)
    ids, _, cnt = ix.search(q, 20, beam, counters=True)
    ix.close()
    rids, rcnt = O.OracleIndex.from_codebook(cb).search(q, 20, beam)
    assert np.array_equal(ids, rids)
    assert np.array_equal(cnt, rcnt.view(np.uint32).reshape(-1, 6))
