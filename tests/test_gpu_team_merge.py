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
                                             (33, 1, 64), (256, 31, 256), (128, 96, 100), (300, 32, 129),
                                             (600, 24, 256), (1100, 40, 100)])
@pytest.mark.parametrize("use_ip", [False, True])
@pytest.mark.parametrize("waves", [2, 4])
def test_waves_match_oracle(gpu_available, monkeypatch, dim, degree, beam, use_ip, waves):
    """Beams up to 256 with two and four waves per query: the waves' shares of a
    round at partial tiles, at more tiles than one round holds and at rounds
    with fewer tasks than waves, for both metrics."""
    from flashgann_amd import Index
    from oracle import oracle as O
    monkeypatch.setenv("FLASHGANN_TEAM", str(waves))
    cb, q, _ = small_index(n=1200, nq=9, dim=dim, comps=5, degree=degree, kind="unit" if use_ip else "int",
                           use_ip=use_ip)
    ix = Index.from_codebook(cb, metric=1 if use_ip else 0)
    K = min(10, beam)
    assert ix.search_waves(q.shape[0], K, beam) == waves
    ids, _, cnt = ix.search(q, K, beam, counters=True)
    ix.close()
    rids, rcnt = O.OracleIndex.from_codebook(cb, use_ip=use_ip).search(q, K, beam)
    assert np.array_equal(ids, rids)
    assert np.array_equal(cnt, rcnt.view(np.uint32).reshape(-1, 6))


@pytest.mark.parametrize("dim,degree", [(128, 32), (96, 16), (40, 8), (100, 24), (200, 32), (300, 32)])
@pytest.mark.parametrize("beam", [64, 128, 300])
def test_forced_forms(gpu_available, monkeypatch, dim, degree, beam):
    """FLASHGANN_TEAM: 0 one wave, 1 and 2 two, 4 four where the geometry has
    them, at every beam and batch."""
    from flashgann_amd import Index
    cb, _, _ = small_index(n=400, nq=4, dim=dim, comps=4, degree=degree, kind="unit")
    ix = Index.from_codebook(cb)
    four = 2 if (dim, degree) == (96, 16) else 4
    for value, waves in (("0", 1), ("1", 2), ("2", 2), ("4", four)):
        monkeypatch.setenv("FLASHGANN_TEAM", value)
        assert [ix.search_waves(nq, 10, beam) for nq in (1, 64, 3000, 100000)] == [waves] * 4, value
    ix.close()
