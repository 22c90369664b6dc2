"""The builder and ground-truth paths bench.py runs on the GPU, against the
same code on the CPU and against a float64 numpy brute force."""
from __future__ import annotations

import numpy as np
import pytest

pytestmark = [pytest.mark.gpu, pytest.mark.usefixtures("search_form")]


def test_gpu_codebook_equals_cpu_codebook_on_integer_data(gpu_available):
    """On integer-valued data every distance, rotation and factor numerator
    is an exact integer in the builder's float32 / float64 arithmetic, so the
    GPU build (graph, codes, factors, entry) is byte-identical to the CPU
    build."""
    from flashgann_amd import builder, datasets
    base, _ = datasets.integer_mixture(3000, 1, 128, 16, config=1)
    signs = datasets.signs_for(128, 1)
    a = builder.build_codebook(base, 32, signs, device="cpu")
    b = builder.build_codebook(base, 32, signs, device="cuda")
    assert a.entry == b.entry
    assert np.array_equal(a.rows.view(np.uint32), b.rows.view(np.uint32))


def test_gpu_encoding_of_float_data_within_rounding(gpu_available):
    """On float data the GPU and CPU encodings of one graph agree: codes
    bit-for-bit except where a rotated residual is within rounding of zero,
    factors within float64 summation-order rounding."""
    from flashgann_amd import builder, datasets
    base, _ = datasets.normalized_mixture(2500, 1, 96, 16, config=3)
    signs = datasets.signs_for(128, 3)
    import torch
    nbrs = builder.build_graph(torch.as_tensor(base), 16)
    a = builder.codebook_from_graph(base, nbrs, signs, device="cpu")
    b = builder.codebook_from_graph(base, nbrs, signs, device="cuda")
    assert np.array_equal(a.neighbors(), b.neighbors())
    ca, cb_ = a.codes(), b.codes()
    assert (ca == cb_).mean() > 0.9999
    fa, fb = a.factors(), b.factors()
    np.testing.assert_allclose(fb, fa, rtol=1e-6, atol=1e-6)


@pytest.mark.parametrize("use_ip", [False, True])
def test_gpu_ground_truth_equals_brute_force(gpu_available, use_ip):
    """GPU ground truth (the ids bench.py scores recall against) equals a
    float64 numpy brute force with ties by id, on integer data where every
    distance is exact."""
    from flashgann_amd import builder, datasets
    base, q = datasets.integer_mixture(5000, 64, 128, 16, config=2)
    gt = builder.ground_truth(base, q, 100, device="cuda", use_ip=use_ip)
    b64, q64 = base.astype(np.float64), q.astype(np.float64)
    if use_ip:
        d = -(q64 @ b64.T)
    else:
        d = (q64 * q64).sum(1)[:, None] + (b64 * b64).sum(1)[None, :] - 2.0 * (q64 @ b64.T)
    ids = np.broadcast_to(np.arange(base.shape[0]), d.shape)
    want = np.lexsort((ids, d), axis=1)[:, :100]
    assert np.array_equal(gt, want.astype(np.int32))


def test_gpu_partitioned_knn_reduces_to_exact_knn(gpu_available):
    """On the GPU as on the CPU: every cell probed is the exact search."""
    import torch
    from flashgann_amd import builder, datasets
    base, _ = datasets.integer_mixture(6000, 1, 64, 8, config=1)
    x = torch.as_tensor(base, device="cuda")
    a_ids, a_d = builder.knn(x, 32)
    b_ids, b_d = builder.knn_partitioned(x, 32, cells=8, probes=8)
    assert torch.equal(a_ids, b_ids) and torch.equal(a_d, b_d)


def test_search_on_partitioned_gpu_build_1536(gpu_available):
    """The C5 build path at small scale: data drawn on the GPU, partitioned
    k-NN graph and encoding on the GPU, then the search (generic geometry,
    padded dimension 2048) against the oracle on the same codebook."""
    from flashgann_amd import Index, builder, datasets
    from oracle import oracle as O
    base, q = datasets.anisotropic_unit_mixture_device(6000, 12, 1536, 24, device="cuda")
    cb = builder.build_codebook(base, 32, datasets.signs_for(2048, 5), device="cuda", knn_method="partitioned")
    qn = q.cpu().numpy()
    ix = Index.from_codebook(cb)
    ids, _, cnt = ix.search(qn, 100, 256, counters=True)
    ix.close()
    rids, rcnt = O.OracleIndex.from_codebook(cb).search(qn, 100, 256)
    assert np.array_equal(ids, rids)
    assert np.array_equal(cnt, rcnt.view(np.uint32).reshape(-1, 6))
    gt = builder.ground_truth(base, q, 100, device="cuda")
    from flashgann_amd.metrics import compute_recall
    assert compute_recall(ids, gt, 100) > 0.9


@pytest.mark.parametrize("dim,degree,use_ip", [(33, 1, False), (64, 3, True), (65, 64, False), (100, 65, True),
                                               (128, 130, False), (200, 24, True), (512, 31, False), (960, 32, True),
                                               (1536, 16, False), (2048, 8, True)])
def test_gpu_encode_kernel_equals_cpu_encoding(gpu_available, dim, degree, use_ip):
    """fg_encode_rows (every register count of its transform, degrees around
    its 64-edge blocks, a last staging block that is not full) against the
    torch path on the CPU.  Integer data with empty slots, a node linked to
    itself and a repeated point: all sums are whole numbers below 2^53 in
    both, and the one division rounds once, so the rows are the same bytes."""
    import torch
    from flashgann_amd import builder, datasets
    from flashgann_amd.codebook import padded_dim_for
    n = 301
    rng = np.random.default_rng(dim + degree)
    base = rng.integers(-40, 200, size=(n, dim)).astype(np.float32)
    base[7] = base[5]
    nbrs = rng.integers(0, n, size=(n, degree))
    nbrs[rng.random((n, degree)) < 0.1] = -1
    nbrs[3, 0] = 3
    nbrs[5, -1] = 7
    signs = datasets.signs_for(padded_dim_for(dim))
    a = builder.codebook_from_graph(base, nbrs, signs, use_ip=use_ip, device="cpu", entry=0)
    b = builder.codebook_from_graph(base, nbrs, signs, use_ip=use_ip, device="cuda", entry=0)
    assert np.array_equal(a.rows.view(np.uint32), b.rows.view(np.uint32))
    x, nb = torch.as_tensor(base).cuda(), torch.as_tensor(nbrs).cuda()
    c = builder._encode_rows_gpu(x, nb, signs, a.layout, use_ip, stage_bytes=7 * a.layout.row_bytes)
    assert np.array_equal(a.rows.view(np.uint32), c.view(np.uint32))
    nb[0, 0] = n
    with pytest.raises(IndexError):
        builder._encode_rows_gpu(x, nb, signs, a.layout, use_ip)


def test_gpu_encoding_ignores_graph_rows_past_the_vectors(gpu_available):
    """A graph of more rows than vectors encodes the vectors' rows, as on the
    CPU, whatever ids the further rows hold; a shorter one is refused."""
    from flashgann_amd import builder, datasets
    from flashgann_amd.codebook import padded_dim_for
    n, dim, degree = 50, 40, 4
    rng = np.random.default_rng(2)
    base = rng.integers(0, 50, size=(n, dim)).astype(np.float32)
    nbrs = rng.integers(0, n, size=(n + 10, degree))
    nbrs[n:] = n + 3
    signs = datasets.signs_for(padded_dim_for(dim))
    a = builder.codebook_from_graph(base, nbrs, signs, device="cpu", entry=0)
    b = builder.codebook_from_graph(base, nbrs, signs, device="cuda", entry=0)
    assert np.array_equal(a.rows.view(np.uint32), b.rows.view(np.uint32))
    with pytest.raises(RuntimeError):
        builder.codebook_from_graph(base, nbrs[:n - 1], signs, device="cuda", entry=0)
