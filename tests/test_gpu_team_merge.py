"""The team form's beam merge above 256 entries, which its two or four waves share: ids
and work counters against the oracle at beams around the segment counts where
the shares change size (an odd number of segments, one per lane, more than
128, the full 256), on integer data, whose equal distances also take the
merge through its tie replay."""
from __future__ import annotations

import numpy as np
import pytest

from conftest import small_index

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("beam", [257, 258, 320, 384, 511, 513, 777, 1023, 1024])
@pytest.mark.parametrize("dim,kind", [(128, "int"), (64, "int"), (300, "box")])
def test_team_merge_matches_oracle(gpu_available, monkeypatch, beam, dim, kind):
    from flashgann_amd import Index
    from oracle import oracle as O
    monkeypatch.setenv("FLASHGANN_TEAM", "1")
    cb, q, _ = small_index(n=2500, nq=16, dim=dim, comps=10, degree=32, kind=kind)
    ix = Index.from_codebook(cb)
    assert ix.search_waves(q.shape[0], 20, beam) == (4 if dim > 256 else 2)
    ids, _, cnt = ix.search(q, 20, beam, counters=True)
    ix.close()
    rids, rcnt = O.OracleIndex.from_codebook(cb).search(q, 20, beam)
    assert np.array_equal(ids, rids)
    assert np.array_equal(cnt, rcnt.view(np.uint32).reshape(-1, 6))
