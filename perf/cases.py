"""Performance cases: the searches and codebook work a program does through
flashgann_amd's public entry points, over the sizes, shapes and options it
meets them in.

Every case is a plain dict.  `call` says which entry point a pass goes through:

  device   Index.search_device: queries and ids in device memory, the
           program's own stream (a resident index)
  host     Index.search: host queries in, host ids out
  stream   Index.search_stream: a serving loop's batches
  cold     Index.from_rows, one search, close: what a program pays that uploads
           a codebook for each search, as the drop-in search method and a
           one-shot command-line run do
  encode   builder.codebook_from_graph: vectors and a graph into a codebook

A search case's index is built once per data set and stays resident, as a
serving program keeps it; the seed draws the queries.  `cold` and `encode`
draw the data set itself from the seed.  The data sets are the mixtures of
flashgann_amd.datasets (integer-valued, unit-norm, unit-box, anisotropic
unit-norm), drawn on the GPU; the graphs are RNG-pruned exact k-NN edges
within a component plus random long links, the builder's recipe.
"""
from __future__ import annotations

import math
from collections import OrderedDict

import numpy as np
import torch

import flashgann_amd as fg
from flashgann_amd import builder, datasets
from flashgann_amd.codebook import Layout, padded_dim_for

DEV = "cuda"
INDEX_SEED = 20240601  # the resident data sets
MAX_RESIDENT = 6       # indexes kept for the search cases


# ------------------------------------------------------------------ the cases

def _case(name, call, data, components, per_component, dim, degree, metric, nq, K, beam, batch=0, streams=0):
    c = dict(call=call, data=data, components=components, per_component=per_component, dim=dim, degree=degree,
             metric=metric, nq=nq, K=K, beam=beam, batch=batch, streams=streams)
    return dict(name=name, **c) if name else c


def listed():
    return [
        # one interactive query against a million points, host in, host out:
        # the smallest call, latency of one search and of the call around it
        _case("one_query_host", "host", "int", 1024, 977, 128, 32, "l2", 1, 10, 64),
        # a micro-batch of a request handler
        _case("micro_batch_d96", "device", "unit", 300, 1000, 96, 32, "l2", 64, 10, 128),
        # a serving loop's small batches on two streams (100k x 128, K 10)
        _case("serve_batches_d128", "stream", "int", 64, 1563, 128, 32, "l2", 8000, 10, 128, batch=1000, streams=2),
        # the benchmark's workload: 10k queries, K 100, recall 0.99
        _case("batch_10k_d128", "device", "int", 1024, 977, 128, 32, "l2", 10000, 100, 256),
        # lower-degree graph, high recall
        _case("batch_10k_d96_deg16", "device", "unit", 1024, 977, 96, 16, "l2", 10000, 100, 512),
        # the widest beam (recall 0.9999)
        _case("beam_1024_d128", "device", "int", 1024, 977, 128, 32, "l2", 2000, 100, 1024),
        # long vectors, a batch that does not fill the device
        _case("batch_1k_d960", "device", "box", 100, 1000, 960, 32, "l2", 1000, 100, 384),
        # embedding vectors, the largest call
        _case("batch_10k_d1536", "device", "aniso", 100, 1000, 1536, 32, "l2", 10000, 100, 640),
        # odd sizes: no dimension, degree, K, beam or batch is a power of two
        _case("ragged_d100_deg24", "device", "unit", 211, 947, 100, 24, "l2", 3001, 37, 200),
        # inner product on 200-d text-to-image sized vectors
        _case("ip_d200", "device", "unit", 250, 800, 200, 32, "ip", 777, 10, 300),
        # upload, search once, release
        _case("cold_search_d128", "cold", "int", 100, 1000, 128, 32, "l2", 1000, 10, 128),
        # a codebook from vectors and their graph
        _case("encode_d128", "encode", "int", 50, 1000, 128, 32, "l2", 0, 0, 0),
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    call = rng.choices(("device", "host", "stream", "cold", "encode"), (60, 14, 10, 8, 8))[0]
    if rng.random() < 0.6:
        dim = rng.choice((64, 96, 100, 128, 200, 256, 384, 512, 768, 960))
    else:
        dim = _log_int(rng, 33, 1100)
    data = "aniso" if dim > 1000 else rng.choice(("int", "unit", "unit", "box"))
    degree = rng.choice((16, 24, 31, 32, 32, 32, 48, 64))
    metric = "ip" if data == "unit" and rng.random() < 0.4 else "l2"
    lay = Layout.make(dim, degree)
    # a codebook of at most 400 MB (a tenth of that for encode: its arithmetic is wide)
    most = min(150_000, (4e8 if call != "encode" else 6e7) / lay.row_bytes)
    per = rng.randint(400, 1000)
    components = max(4, int(rng.uniform(0.4, 1.0) * most) // per)
    if call == "encode":
        return _case("", call, data, components, per, dim, degree, metric, 0, 0, 0)
    beam = _log_int(rng, 10, 1024)
    K = min(beam, _log_int(rng, 1, 100))
    nq = _log_int(rng, 1, 10000 if call in ("device", "host") else 3000)
    # no more than the largest listed case
    nq = max(1, min(nq, int(6e10 / (beam * _bytes_per_expansion(dim, degree)))))
    batch, streams = (max(1, nq // rng.randint(2, 9)), rng.randint(1, 4)) if call == "stream" else (0, 0)
    return _case("", call, data, components, per, dim, degree, metric, nq, K, beam, batch, streams)


# ------------------------------------------------------------------ data sets

def _generator(seed):
    g = torch.Generator(device=DEV)
    g.manual_seed(seed)
    return g


def _means(c, g):
    shape = (c["components"], c["dim"])
    if c["data"] == "int":
        return torch.rand(shape, generator=g, device=DEV) * 100.0
    if c["data"] == "box":
        return torch.rand(shape, generator=g, device=DEV)
    return torch.randn(shape, generator=g, device=DEV)


def _points(c, means, g, comp):
    """One point of each listed component."""
    z = torch.randn((comp.shape[0], c["dim"]), generator=g, device=DEV)
    mu = means[comp]
    if c["data"] == "int":
        return (mu + 10.0 * z).round_().clamp_(min=0.0)
    if c["data"] == "box":
        return (mu + 0.1 * z).clamp_(0.0, 1.0)
    if c["data"] == "aniso":
        # each component has its own spread in each dimension
        scale = 0.05 + 0.45 * torch.frac(mu.abs() * 997.0)
        x = mu + scale * z
    else:
        x = mu + 0.3 * z
    return x / torch.linalg.vector_norm(x, dim=1, keepdim=True)


def _queries(c, means, seed):
    g = _generator(seed * 2 + 1)
    comp = torch.randint(0, c["components"], (c["nq"],), generator=g, device=DEV)
    return _points(c, means, g, comp)


def _local_edges(x, degree):
    """x: (components, m, dim).  RNG-pruned exact k-NN edges within each
    component, at most degree - degree // 4 of 2 * degree candidates: places
    within the component (components, m, keep), -1 where the rule kept fewer."""
    nc, m, _ = x.shape
    kc = min(2 * degree, m - 1)
    keep = min(kc, degree - degree // 4)
    out = torch.full((nc, m, keep), -1, dtype=torch.int64, device=DEV)
    step = max(1, (1 << 27) // (m * kc * kc))
    for s in range(0, nc, step):
        xb = x[s:s + step]
        n2 = (xb * xb).sum(-1)
        d = n2[:, :, None] + n2[:, None, :] - 2.0 * torch.bmm(xb, xb.transpose(1, 2).contiguous())
        d.clamp_(min=0.0)
        torch.diagonal(d, dim1=1, dim2=2).fill_(float("inf"))
        du, cand = torch.topk(d, kc, dim=2, largest=False, sorted=True)
        flat = cand[:, :, :, None] * m + cand[:, :, None, :]
        pd = torch.gather(d.reshape(d.shape[0], m * m), 1, flat.reshape(d.shape[0], -1)).view(flat.shape)
        del flat, d
        kept = torch.zeros(cand.shape, dtype=torch.bool, device=DEV)
        count = torch.zeros(cand.shape[:2], dtype=torch.int64, device=DEV)
        for i in range(kc):
            ok = count < keep
            if i:
                ok &= ~((pd[:, :, i, :i] < du[:, :, i:i + 1]) & kept[:, :, :i]).any(2)
            kept[:, :, i] = ok
            count += ok
        place = torch.where(kept, torch.arange(kc, device=DEV), kc)
        order = torch.sort(place, dim=2).values[:, :, :keep]
        got = torch.gather(cand, 2, order.clamp(max=kc - 1))
        out[s:s + step] = torch.where(order < kc, got, torch.full_like(got, -1))
    return out


def _data_set(c, seed):
    """(means, vectors (n, dim), neighbour ids (n, degree)) on the GPU: the
    points of each component spread over the ids, every neighbour list
    without repeats."""
    g = _generator(seed)
    means = _means(c, g)
    nc, m, degree = c["components"], c["per_component"], c["degree"]
    n = nc * m
    comp = torch.arange(nc, device=DEV).repeat_interleave(m)
    x = _points(c, means, g, comp)
    local = _local_edges(x.view(nc, m, -1), degree)
    first = (torch.arange(nc, device=DEV) * m)[:, None, None]
    local = torch.where(local >= 0, local + first, local).view(n, -1)
    nbrs = torch.full((n, degree), -1, dtype=torch.int64, device=DEV)
    nbrs[:, :local.shape[1]] = local
    own = torch.arange(n, device=DEV)[:, None]
    free = nbrs < 0
    bad = free
    for _ in range(64):  # random links in the free slots, drawn again where one repeats
        nbrs = torch.where(bad, torch.randint(0, n, (n, degree), generator=g, device=DEV), nbrs)
        o = torch.sort(nbrs, dim=1, stable=True)
        rep = torch.zeros_like(free)
        rep[:, 1:] = o.values[:, 1:] == o.values[:, :-1]
        again = torch.zeros_like(free).scatter_(1, o.indices, rep) | (nbrs == own)
        # a repeat can fall on a local edge: the row's free slots are then drawn again
        bad = (again | again.any(1, keepdim=True)) & free
        if not bool(bad.any()):
            break
    perm = torch.randperm(n, generator=g, device=DEV)  # place -> id
    vec = torch.empty_like(x)
    vec[perm] = x
    ids = torch.empty_like(nbrs)
    ids[perm] = perm[nbrs]
    return means, vec, ids


def _rotation(signs):
    """H_B diag(signs), float64."""
    b = signs.shape[0]
    h = torch.ones((1, 1), dtype=torch.float64, device=DEV)
    while h.shape[0] < b:
        h = torch.cat((torch.cat((h, h), 1), torch.cat((h, -h), 1)), 0)
    return h * torch.as_tensor(signs, dtype=torch.float64, device=DEV)[None, :]


def _edge_codes(c, vec, ids, signs, s, e, p):
    """Codes (e - s, degree, B / 8) uint8 and float64 factors (e - s, 3,
    degree) of the edges of nodes s .. e - 1."""
    b, dim = p.shape[0], c["dim"]
    centre = torch.zeros((e - s, b), dtype=torch.float64, device=DEV)
    centre[:, :dim] = vec[s:e]
    r = torch.zeros((e - s, ids.shape[1], b), dtype=torch.float64, device=DEV)
    r[:, :, :dim] = vec[ids[s:e]]
    r[:, :, :dim] -= centre[:, None, :dim]
    y = r @ p.T
    nr = (r * r).sum(-1)
    del r
    sabs = y.abs().sum(-1)
    bits = y > 0
    del y
    f = torch.where(sabs > 0, (-1.0 if c["metric"] == "ip" else -2.0) * nr / sabs, torch.zeros_like(nr))
    ssum = 2.0 * bits.sum(-1) - b
    if c["metric"] == "ip":
        tx = torch.zeros_like(f)
    else:
        sgn = bits.to(torch.float64).mul_(2.0).sub_(1.0)
        spc = torch.bmm(sgn, (centre @ p.T)[:, :, None])[:, :, 0]
        del sgn
        tx = torch.where(sabs > 0, nr - f * spc, torch.zeros_like(nr))
    weight = torch.tensor([8, 4, 2, 1, 128, 64, 32, 16], dtype=torch.uint8, device=DEV)
    codes = (bits.view(*bits.shape[:2], b // 8, 8) * weight).sum(-1, dtype=torch.uint8)
    return codes, torch.stack((tx, f, f * ssum), 1)


def _codebook_rows(c, vec, ids, signs):
    """Host codebook rows in the reference layout."""
    lay = Layout.make(c["dim"], c["degree"])
    n = vec.shape[0]
    p = _rotation(signs)
    rows = torch.empty((n, lay.row_offset), dtype=torch.float32, device=DEV)
    rows[:, :c["dim"]] = vec
    rows[:, lay.neighbor_offset:] = ids.to(torch.int32).view(torch.float32)
    step = max(1, (1 << 28) // (c["degree"] * lay.padded_dim))
    for s in range(0, n, step):
        e = min(n, s + step)
        codes, factors = _edge_codes(c, vec, ids, signs, s, e, p)
        rows[s:e, lay.code_offset:lay.factor_offset] = codes.view(e - s, -1).view(torch.float32)
        rows[s:e, lay.factor_offset:lay.neighbor_offset] = factors.to(torch.float32).view(e - s, -1)
    return rows.cpu().numpy()


def _entry(vec):
    """The id of the point nearest the mean."""
    mu = vec.to(torch.float64).mean(0)
    return int(torch.argmin((vec.to(torch.float64) - mu).square().sum(1)).item())


def _signs(c):
    return datasets.signs_for(padded_dim_for(c["dim"]))


def _metric(c):
    return fg.METRIC_IP if c["metric"] == "ip" else fg.METRIC_L2


_resident: "OrderedDict[tuple, tuple]" = OrderedDict()


def _index(c):
    """(index, means) of the case's resident data set."""
    key = tuple(c[k] for k in ("data", "components", "per_component", "dim", "degree", "metric"))
    if key not in _resident:
        while len(_resident) >= MAX_RESIDENT:
            _resident.popitem(last=False)
        means, vec, ids = _data_set(c, INDEX_SEED)
        rows = _codebook_rows(c, vec, ids, _signs(c))
        index = fg.Index.from_rows(rows, _signs(c), c["dim"], c["degree"], _entry(vec), _metric(c))
        del vec, ids, rows
        torch.cuda.empty_cache()
        _resident[key] = (index, means)
    _resident.move_to_end(key)
    return _resident[key]


# ------------------------------------------------------------------ measuring

def prepare(case, seed):
    c = dict(case)
    if c["call"] == "encode":
        _, vec, ids = _data_set(c, seed)
        return dict(case=c, vectors=vec, graph=ids, signs=_signs(c), entry=_entry(vec))
    if c["call"] == "cold":
        means, vec, ids = _data_set(c, seed)
        return dict(case=c, rows=_codebook_rows(c, vec, ids, _signs(c)), signs=_signs(c), entry=_entry(vec),
                    queries=_queries(c, means, seed).cpu().numpy())
    index, means = _index(c)
    q = _queries(c, means, seed)
    if c["call"] == "host":
        return dict(case=c, index=index, queries=q.cpu().numpy())
    return dict(case=c, index=index, queries=q, ids=torch.empty((c["nq"], c["K"]), dtype=torch.int32, device=DEV))


def run(state):
    c = state["case"]
    if c["call"] == "encode":
        cb = builder.codebook_from_graph(state["vectors"], state["graph"], state["signs"],
                                         use_ip=c["metric"] == "ip", device=DEV, entry=state["entry"])
        return dict(vectors=cb.vectors(), codes=cb.codes(), factors=cb.factors(), neighbors=cb.neighbors())
    if c["call"] == "cold":
        index = fg.Index.from_rows(state["rows"], state["signs"], c["dim"], c["degree"], state["entry"], _metric(c))
        ids, _, _ = index.search(state["queries"], c["K"], c["beam"])
        index.close()
        return ids
    index = state["index"]
    if c["call"] == "host":
        ids, _, _ = index.search(state["queries"], c["K"], c["beam"])
        return ids
    stream = torch.cuda.current_stream().cuda_stream
    q, ids = state["queries"], state["ids"]
    if c["call"] == "stream":
        index.search_stream(q.data_ptr(), c["nq"], c["K"], c["beam"], ids.data_ptr(), c["batch"], c["streams"], stream)
    else:
        index.search_device(q.data_ptr(), c["nq"], c["K"], c["beam"], ids.data_ptr(), 0, stream)
    return ids


def _bytes_per_expansion(dim, degree):
    """Neighbour ids, codes and factors of one node, and its vector."""
    return degree * (4 + padded_dim_for(dim) // 8 + 12) + 4 * dim


def work(case):
    """A search ends when every beam entry is expanded, so it reads at least
    `beam` nodes' neighbour blocks and vectors; each query is read and its ids
    written once.  `cold` also moves the codebook in; `encode` reads each
    edge's vector and writes the rows."""
    c = case
    n = c["components"] * c["per_component"]
    b = padded_dim_for(c["dim"])
    row = Layout.make(c["dim"], c["degree"]).row_bytes
    if c["call"] == "encode":
        edges = n * c["degree"]
        return {"bytes": n * c["dim"] * 4 + edges * 8 + n * row,
                "flops": edges * (b * math.log2(b) + 6.0 * b)}
    beam = min(c["beam"], n)
    moved = c["nq"] * (4 * c["dim"] + 4 * c["K"] + beam * _bytes_per_expansion(c["dim"], c["degree"]))
    flops = c["nq"] * beam * (3.0 * c["dim"] + c["degree"] * (2.0 * b + 8.0))
    return {"bytes": moved + (n * row if c["call"] == "cold" else 0), "flops": flops}


def tolerance(case):
    """Searches return ids, which are the same for any correct build: the
    order of every sum in the search is part of its definition.  An encoded
    codebook's factors are float32 of float64 sums, so another summation
    order moves one by a rounding step at most (2^-24 relative, measured
    2.5e-8 over all against float64), and a code bit only where a rotated
    residual is within float64 rounding of zero."""
    if case["call"] == "encode":
        return {"rel": 1e-7, "max": 5e-7, "differ": 1e-7}
    return "exact"


def exact(case, seed):
    """The encoded codebook's vectors and factors in float64 (ids and code
    bits, and the ids of a search, are whole numbers)."""
    c = dict(case)
    if c["call"] != "encode":
        return None
    _, vec, ids = _data_set(c, seed)
    signs = _signs(c)
    p = _rotation(signs)
    n = vec.shape[0]
    step = max(1, (1 << 27) // (c["degree"] * p.shape[0]))
    factors = torch.cat([_edge_codes(c, vec, ids, signs, s, min(n, s + step), p)[1] for s in range(0, n, step)])
    return dict(vectors=vec.to(torch.float64), codes=None, factors=factors, neighbors=None)
