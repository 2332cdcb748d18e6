"""The work that users of jasper_amd have it do, as cases that can be timed.

A case names a kind of call, its sizes and the data it runs on:

  search   Graph.search over a plain graph (exact distances)
  lsh, pq, rabitq
           the estimated searches of a directional graph
  build    Graph.build, then a batch of searches in what it built
  update   a live index: build, append, delete, consolidate, search
  knn      bruteforce_knn (ground truth, exact answers)
  rotate   the prerotation of a set of rows
  encode   rabitq_quantize, one-bit codes of a set of rows

The data are those of jasper_amd.datasets, made on the GPU: "clustered"
(integers, as u8 datasets stored in fp16), "gaussian", "sphere" (unit rows,
for inner products) and "sparse" (non-negative rows with zeros). Sizes follow
the repository's configurations and the ranges around them.
"""

from __future__ import annotations

import math

import torch

import jasper_amd
from jasper_amd import Graph, datasets

# A construction's own search beam, and the share of an expanded node's
# neighbours that a search has not met before (about 0.4 on the 1M x 128
# graph at beam widths of 44 to 64); work() prices a traversal with them.
BUILD_BEAM = 64
NEW_SHARE = 0.4


def listed():
    return [
        # One user's query to a server that holds a 1M-row index: the call's
        # own latency, launch included.
        {"name": "search-one", "kind": "search", "data": "clustered", "metric": "l2", "rows": 1_000_000, "dim": 128,
         "degree": 64, "queries": 1, "k": 10, "beam": 64},
        # The headline: 10k queries over 1M integer rows at the beam width
        # that reaches recall@10 >= 0.95 there.
        {"name": "search-batch", "kind": "search", "data": "clustered", "metric": "l2", "rows": 1_000_000, "dim": 128,
         "degree": 64, "queries": 10_000, "k": 10, "beam": 44},
        # Embeddings compared by inner product: rows that are no integers.
        {"name": "search-ip", "kind": "search", "data": "sphere", "metric": "ip", "rows": 1_000_000, "dim": 96,
         "degree": 64, "queries": 10_000, "k": 10, "beam": 64},
        # Long rows (image descriptors), a moderate batch, high recall.
        {"name": "search-long", "kind": "search", "data": "sparse", "metric": "l2", "rows": 100_000, "dim": 960,
         "degree": 64, "queries": 1_000, "k": 10, "beam": 128},
        # The LSH estimator of the large configuration (16 ranks, distinct
        # results), where a wide beam has to make up for the estimate.
        {"name": "search-lsh", "kind": "lsh", "data": "clustered", "metric": "l2", "rows": 1_000_000, "dim": 128,
         "degree": 64, "queries": 10_000, "k": 10, "beam": 256, "k_ranks": 16, "pq_m": 0, "unique": True},
        # Product quantization of long rows, one subspace per 8 dims.
        {"name": "search-pq", "kind": "pq", "data": "sparse", "metric": "l2", "rows": 100_000, "dim": 960,
         "degree": 64, "queries": 1_000, "k": 10, "beam": 128, "k_ranks": 16, "pq_m": 120, "unique": False},
        # An index of 1M integer rows from scratch, and its first queries.
        {"name": "build-batch", "kind": "build", "data": "clustered", "metric": "l2", "rows": 1_000_000, "dim": 128,
         "degree": 64, "queries": 10_000, "k": 10, "beam": 64, "artifacts": "none", "k_ranks": 4},
        # A live index of real-valued rows of a ragged size: a tenth more
        # rows arrive, a tenth is deleted, the graph is repaired.
        {"name": "update-ragged", "kind": "update", "data": "gaussian", "metric": "l2", "rows": 150_001, "dim": 100,
         "degree": 32, "queries": 1_000, "k": 10, "beam": 64, "more": 15_003, "less": 15_001},
        # Ground truth of the headline's queries.
        {"name": "knn-batch", "kind": "knn", "data": "clustered", "metric": "l2", "rows": 1_000_000, "dim": 128,
         "queries": 10_000, "k": 10},
        # Ground truth of long rows, at the utility's default k.
        {"name": "knn-long", "kind": "knn", "data": "sparse", "metric": "l2", "rows": 1_000_000, "dim": 960,
         "queries": 1_000, "k": 100},
        # The prerotation that a directional index of long rows begins with.
        {"name": "rotate-long", "kind": "rotate", "data": "sparse", "metric": "l2", "rows": 1_000_000, "dim": 960},
        # One-bit codes of 1M rows around their centroid.
        {"name": "encode-batch", "kind": "encode", "data": "clustered", "metric": "l2", "rows": 1_000_000, "dim": 128,
         "half": True},
    ]


def _log(rng, lo, hi):
    """A whole number between lo and hi, even over its logarithm."""
    return max(lo, min(hi, round(math.exp(rng.uniform(math.log(lo), math.log(hi))))))


def draw(rng):
    kind = rng.choice(("search", "search", "search", "lsh", "pq", "rabitq", "build", "update", "knn", "knn",
                       "rotate", "encode"))
    data, metric = rng.choice((("clustered", "l2"), ("clustered", "l2"), ("gaussian", "l2"), ("sphere", "ip"),
                               ("sparse", "l2")))
    dim = rng.choice((32, 64, 96, 96, 100, 128, 128, 128, 200, 256, 384, 768, 960, rng.randint(17, 960)))
    if kind in ("rabitq", "encode"):
        dim = rng.choice((32, 64, 96, 100, 128, 128, 200, 256, rng.randint(17, 256)))
    if kind == "update":
        dim = rng.choice((50, 64, 96, 100, 128, 128, 200))
    if kind == "pq" and dim % 8:
        dim = 8 * (dim // 8)
    case = {"kind": kind, "data": data, "metric": metric, "dim": dim}
    most = min(1_000_000, 128_000_000 // dim)
    if kind == "rotate":
        case["rows"] = _log(rng, 10_000, 1_000_000)
    elif kind == "encode":
        case["rows"] = _log(rng, 10_000, most)
        case["half"] = rng.random() < 0.75
    elif kind == "knn":
        case["rows"] = _log(rng, 20_000, 1_000_000)
        case["queries"] = _log(rng, 100, min(10_000, 960_000 // dim))
        case["k"] = rng.choice((1, 10, 10, 32, 100))
    else:
        case["rows"] = _log(rng, 20_000, most if kind in ("search", "build") else min(most, 300_000))
        case["degree"] = rng.choice((32, 64, 64) if kind in ("lsh", "pq", "rabitq") else (16, 32, 64, 64))
        case["queries"] = _log(rng, 1, 10_000)
        case["k"] = rng.choice((1, 10, 10, 10, 32))
        case["beam"] = _log(rng, 32, 256)
    if kind in ("lsh", "pq", "rabitq"):
        case["k_ranks"] = rng.choice((4, 16))
        case["pq_m"] = 0
        case["unique"] = rng.random() < 0.5
    if kind == "pq":
        case["pq_m"] = rng.choice([m for m in (4, 8, 16, dim // 8) if dim % m == 0 and dim // m <= 64])
    if kind == "build":
        case["k_ranks"] = rng.choice((4, 16))
        case["artifacts"] = rng.choice(("none", "none", "lsh")) if case["degree"] >= 32 else "none"
    if kind == "update":
        case["rows"] = min(case["rows"], 150_000)
        case["more"] = max(1, round(case["rows"] * rng.uniform(0.01, 0.1)))
        case["less"] = max(1, round(case["rows"] * rng.uniform(0.01, 0.1)))
    return case


def _rows(case, count, seed):
    """Rows [count, dim] of the case's data in fp16, on the GPU."""
    data, dim = case["data"], case["dim"]
    if data == "clustered":
        return datasets.clustered_device(count, dim, seed, "cuda", n_clusters=max(10, case["rows"] // 1000))
    if data == "sparse":
        return datasets.sparse_abs_device(count, dim, seed, "cuda")
    gen = torch.Generator(device="cuda")
    gen.manual_seed(seed)
    x = torch.randn((count, dim), generator=gen, device="cuda")
    if data == "sphere":
        x /= x.norm(dim=1, keepdim=True)
    return x.to(torch.float16)


def _rotation(dim, seed):
    """An orthogonal matrix, column-major fp32 as rabitq_quantize takes it."""
    gen = torch.Generator().manual_seed(seed)
    q, _ = torch.linalg.qr(torch.randn((dim, dim), generator=gen, dtype=torch.float64))
    return q.to(torch.float32).cuda()


def prepare(case, seed):
    kind, dim = case["kind"], case["dim"]
    base = _rows(case, case["rows"], 4 * seed)
    state = {"case": dict(case)}
    if "queries" in case:
        state["queries"] = _rows(case, case["queries"], 4 * seed + 1)
    if kind in ("search", "lsh", "pq", "rabitq"):
        # the program keeps the index; the rows it was built from may go
        more = {}
        if kind == "lsh":
            more = {"build_lsh": True, "k_ranks": case["k_ranks"]}
        elif kind == "pq":
            more = {"build_pq": True, "k_ranks": case["k_ranks"], "pq_m": case["pq_m"]}
        elif kind == "rabitq":
            more = {"build_rabitq": True, "k_ranks": case["k_ranks"]}
        state["graph"] = Graph.build(base, n_neighbors=case["degree"], distance=case["metric"], **more)
        return state
    state["base"] = base
    if kind == "update":
        state["more"] = _rows(case, case["more"], 4 * seed + 2)
        gen = torch.Generator().manual_seed(seed)
        state["less"] = torch.randperm(case["rows"], generator=gen)[:case["less"]].to(torch.int32).sort().values
    elif kind == "encode":
        state["base"] = base if case["half"] else base.float()
        state["rotation"] = _rotation(dim, seed)
        state["centroid"] = base.float().mean(dim=0)
    return state


def run(state):
    case = state["case"]
    kind = case["kind"]
    if kind == "search":
        return state["graph"].search(state["queries"], k=case["k"], beam_width=case["beam"])
    if kind == "lsh":
        return state["graph"].directional_search(state["queries"], k=case["k"], beam_width=case["beam"],
                                                 unique=case["unique"])
    if kind == "pq":
        return state["graph"].pq_search(state["queries"], k=case["k"], beam_width=case["beam"], unique=case["unique"])
    if kind == "rabitq":
        return state["graph"].rabitq_search(state["queries"], k=case["k"], beam_width=case["beam"],
                                            unique=case["unique"])
    if kind == "build":
        lsh = case["artifacts"] == "lsh"
        graph = Graph.build(state["base"], n_neighbors=case["degree"], distance=case["metric"], build_lsh=lsh,
                            k_ranks=case["k_ranks"])
        search = graph.directional_search if lsh else graph.search
        return search(state["queries"], k=case["k"], beam_width=case["beam"])
    if kind == "update":
        graph = Graph.build(state["base"], n_neighbors=case["degree"], distance=case["metric"])
        ids = graph.append(state["more"])
        graph.mark_deleted(state["less"])
        graph.consolidate()
        found, dist = graph.search(state["queries"], k=case["k"], beam_width=case["beam"])
        return ids, found, dist
    if kind == "knn":
        return jasper_amd.bruteforce_knn(state["base"], state["queries"], case["k"], case["metric"])
    if kind == "rotate":
        return jasper_amd.rotate(state["base"])
    codes = jasper_amd.rabitq_quantize(state["base"], rotation=state["rotation"], centroid=state["centroid"],
                                       distance=case["metric"])
    return codes.codes, codes.f_add, codes.f_rescale


def _traversal(case, queries, beam, per_edge):
    """Bytes and operations of a beam search: as many nodes expanded as the
    beam holds, each with its row of neighbours and, for each neighbour that
    is new, what the search scores it by (per_edge bytes, or its vector)."""
    dim, degree = case["dim"], case["degree"]
    if per_edge is None:
        node, ops = 4 * degree + NEW_SHARE * degree * 2 * dim, NEW_SHARE * degree * 3 * dim
    else:
        node, ops = 4 * degree + degree * per_edge + 2 * dim, degree * per_edge + 3 * dim
    return queries * (beam * node + 2 * dim), queries * beam * ops


def work(case):
    kind, dim, rows = case["kind"], case["dim"], case["rows"]
    if kind == "rotate":
        return {"bytes": 4 * rows * dim + 2 * dim * dim, "flops": 2 * rows * dim * dim}
    if kind == "encode":
        code = 4 * ((dim + 31) // 32)
        return {"bytes": rows * ((2 if case["half"] else 4) * dim + code + 8) + 4 * dim * dim,
                "flops": 2 * rows * dim * dim}
    queries, k = case["queries"], case["k"]
    out = 8 * queries * k
    if kind == "knn":
        return {"bytes": 2 * dim * (rows + queries) + out, "flops": 2 * rows * queries * dim}
    per_edge = None
    if kind == "lsh" or case.get("artifacts") == "lsh":
        per_edge = case["k_ranks"] * (1 if dim <= 128 else 2) + 2
    elif kind == "pq":
        per_edge = case["pq_m"]
    elif kind == "rabitq":
        per_edge = 4 * ((dim + 31) // 32) + 8
    size, ops = _traversal(case, queries, case["beam"], per_edge)
    if kind in ("build", "update"):
        # each row that is wired in: a search for its candidates, then the
        # two prunes' candidate rows; its vector read, its edges written
        wired = rows + case.get("more", 0) + case.get("less", 0)
        b, f = _traversal(case, wired, BUILD_BEAM, None)
        row = 2 * (BUILD_BEAM + case["degree"]) * 2 * dim + 6 * case["degree"]
        size, ops = size + b + wired * row, ops + f + wired * BUILD_BEAM * case["degree"] * 2 * dim
    return {"bytes": size + out, "flops": ops}


def tolerance(case):
    kind = case["kind"]
    if kind == "rotate":
        # fp32 sums of exact products, rounded once to fp16: another order of
        # the sums moves some results by one fp16 step
        return {"rel": 1e-4, "max": 2e-3}
    if kind == "encode":
        # fp32 rotation and sums; f_add is a difference of larger sums, and a
        # residual that is zero to fp32 may come out with either sign (f_add
        # is 2.6e-4 off its 64-bit value on the listed case)
        return {"rel": 1e-3, "differ": 1e-4}
    if kind == "knn" and (case["data"] != "clustered" or case["dim"] > 256):
        if case["metric"] == "ip":
            # the product is rounded to fp16, so neighbours tie often and a
            # last bit decides between them
            return {"rel": 2e-4, "differ": 2e-2}
        # distances 1.2e-6 off their 64-bit values on the listed case
        return {"rel": 5e-6, "differ": 2e-2}
    # Integer rows of up to 256 dims have exact distances. The searches and constructions order
    # their candidates by (distance, id) with every rounding laid down, so
    # their answers are the same bits for every correct implementation.
    return "exact"


def exact(case, seed):
    kind = case["kind"]
    if kind == "knn":
        base = _rows(case, case["rows"], 4 * seed).double()
        queries = _rows(case, case["queries"], 4 * seed + 1).double()
        norms = base.square().sum(dim=1)
        found = []
        step = max(1, 250_000_000 // case["rows"])
        for q in queries.split(step):
            dist = q @ base.T
            if case["metric"] == "l2":
                dist = dist.mul_(-2).add_(norms).add_(q.square().sum(dim=1, keepdim=True)).clamp_(min=0)
            else:
                dist = dist.neg_()
            found.append(torch.topk(dist, min(case["k"], case["rows"]), dim=1, largest=False, sorted=True).values)
        return None, torch.cat(found)
    if kind == "encode":
        base = _rows(case, case["rows"], 4 * seed)
        centroid = base.float().mean(dim=0).double()
        p = _rotation(case["dim"], seed).double()  # row i is column i of the column-major matrix
        x = base.double()
        r = x @ p.T - p.T @ centroid  # rows by P^T, the centroid by P, as the quantizer defines it
        c = p.T @ centroid
        half = torch.where(r >= 0, 0.5, -0.5)
        norm = r.norm(dim=1)
        unit = r.abs().sum(dim=1) / norm
        rb, cb, rc = (r * half).sum(dim=1), (half * c).sum(dim=1), r @ c
        if case["metric"] == "l2":
            f_add = norm.square() + 2 * norm.square() * cb / rb
            f_rescale = -2 * norm / (0.5 * unit)
        else:
            f_add = 1 - rc + norm.square() * cb / rb
            f_rescale = -norm / (0.5 * unit)
        return None, f_add, f_rescale
    # The rotation's matrix is the library's own sequence, and what a graph
    # search finds depends on the graph: neither has a value apart from it.
    return None
