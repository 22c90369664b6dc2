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
@pytest.mark.parametrize("dim,kind", [(128, "int"), (64, "int"), (200, "box"), (300, "box")])
@pytest.mark.parametrize("waves", [2, 4])
def test_team_merge_matches_oracle(gpu_available, monkeypatch, beam, dim, kind, waves):
    from flashgann_amd import Index
    from oracle import oracle as O
    monkeypatch.setenv("FLASHGANN_TEAM", str(waves))
    cb, q, _ = small_index(n=2500, nq=16, dim=dim, comps=10, degree=32, kind=kind)
    ix = Index.from_codebook(cb)
    assert ix.search_waves(q.shape[0], 20, beam) == waves
    ids, _, cnt = ix.search(q, 20, beam, counters=True)
    ix.close()
    rids, rcnt = O.OracleIndex.from_codebook(cb).search(q, 20, beam)
    assert np.array_equal(ids, rids)
    assert np.array_equal(cnt, rcnt.view(np.uint32).reshape(-1, 6))


@pytest.mark.parametrize("dim,degree,beam", [(128, 32, 65), (96, 32, 10), (100, 24, 200), (64, 33, 128), (200, 64, 17),
                                             (33, 1, 64), (256, 31, 256), (128, 96, 100)])
@pytest.mark.parametrize("use_ip", [False, True])
def test_four_waves_match_oracle(gpu_available, monkeypatch, dim, degree, beam, use_ip):
    """Beams up to 256 with four waves per query: the waves' shares of a round
    at partial tiles, at more tiles than one round holds and at rounds with
    fewer tasks than waves, for both metrics."""
    from flashgann_amd import Index
    from oracle import oracle as O
    monkeypatch.setenv("FLASHGANN_TEAM", "4")
    cb, q, _ = small_index(n=1200, nq=9, dim=dim, comps=5, degree=degree, kind="unit" if use_ip else "int",
                           use_ip=use_ip)
    ix = Index.from_codebook(cb)
    K = min(10, beam)
    assert ix.search_waves(q.shape[0], K, beam) == 4
    ids, _, cnt = ix.search(q, K, beam, counters=True)
    ix.close()
    rids, rcnt = O.OracleIndex.from_codebook(cb).search(q, K, beam)
    assert np.array_equal(ids, rids)
    assert np.array_equal(cnt, rcnt.view(np.uint32).reshape(-1, 6))
