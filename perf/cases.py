"""Timing cases of the spatial index: what a program does with it, from one
small lookup to a 10M-box join, through the public Python entry points.

  points      Query(kContains) of points: point location
  contains    Query(kContains) of envelopes: data boxes around each envelope
  within      Query(kWithin): data boxes inside each envelope
  intersects  Query(kIntersects): data boxes meeting each envelope (the join)
  lines       QueryLines(kIntersects): data boxes each segment meets
  build       Clear, Insert and Build of a whole index, a point lookup, an Insert
              of 1% more boxes and the lookup again (it walks the small tree of
              recent inserts too)
  refresh     Delete and Update on a resident index (refit), then a point lookup
  serve       rts_serve_run over a mixed trace of requests, all arrived

Queries count (SharedValue) or collect (Queue). The queue has no order of its
own, so collecting cases put its pairs in (query, box) order with sort_pairs
and into a table of fixed size, as a program does that joins the pairs on.

Every coordinate is made on the GPU from the seed. `uniform`: corners
U[0, 1)^2, sides U[0, side]. `mixture`: centres from 16 Gaussians (sigma 0.02,
means U[0.1, 0.9]^2), log-normal sides with median `side`, queries from the
same mixture. Results are whole numbers and exact: there is nothing for a
wider type to say about them.
"""
import math

import torch

import rtspatial_amd as R
from rtspatial_amd import _native as N
from rtspatial_amd import serve

P = R.Predicate
PRED = {"points": P.kContains, "contains": P.kContains, "within": P.kWithin,
        "intersects": P.kIntersects, "lines": P.kIntersects}


def listed():
    return [
        # The smallest call: a thousand lookups in a thousand boxes, all launch latency.
        dict(name="points_1k", kind="points", boxes=1000, queries=1000, dist="uniform",
             side=0.05, qside=0.0, coord="f32", handler="count"),
        # Point location of one batch in a small map.
        dict(name="points_100k", kind="points", boxes=100_000, queries=100_000, dist="uniform",
             side=0.01, qside=0.0, coord="f32", handler="count"),
        # The lookup of a large resident index, collected; the mutable index's query.
        dict(name="points_10m", kind="points", boxes=10_000_000, queries=1_000_000,
             dist="uniform", side=1e-3, qside=0.0, coord="f32", handler="collect"),
        # Which regions cover each small envelope (the reference's kContains).
        dict(name="contains_1m", kind="contains", boxes=1_000_000, queries=200_003,
             dist="uniform", side=0.01, qside=1e-3, coord="f32", handler="collect"),
        # Window queries with some twenty results each.
        dict(name="within_1m", kind="within", boxes=1_000_000, queries=1_000_000,
             dist="uniform", side=1e-3, qside=0.01, coord="f32", handler="collect"),
        # The skewed join, as a selectivity count.
        dict(name="join_10m_count", kind="intersects", boxes=10_000_000, queries=1_000_000,
             dist="mixture", side=1e-4, qside=5e-3, coord="f32", handler="count"),
        # The skewed join, collected: a thousand results for each query.
        dict(name="join_1m", kind="intersects", boxes=1_000_003, queries=20_000,
             dist="mixture", side=1e-4, qside=5e-3, coord="f32", handler="collect"),
        # The same in double coordinates.
        dict(name="join_1m_f64", kind="intersects", boxes=1_000_000, queries=10_000,
             dist="mixture", side=1e-4, qside=5e-3, coord="f64", handler="collect"),
        # Road segments against boxes.
        dict(name="lines_1m", kind="lines", boxes=1_000_000, queries=100_000, dist="mixture",
             side=1e-4, qside=5e-3, coord="f32", handler="collect"),
        # A whole index from its boxes, at a size that fills no tile.
        dict(name="build_10m", kind="build", boxes=9_999_991, queries=10_000, dist="uniform",
             side=1e-3, qside=0.0, coord="f32", handler="collect"),
        # A round of the mutable index without inserts.
        dict(name="refresh_10m", kind="refresh", boxes=10_000_000, queries=100_000,
             dist="uniform", side=1e-3, qside=0.0, coord="f32", handler="collect"),
        # The served stream at saturation: many uneven requests on one index.
        dict(name="serve_1m", kind="serve", boxes=1_000_000, queries=64, dist="mixture",
             side=1e-4, qside=5e-3, coord="f32", handler="count"),
    ]


def _log_int(rng, lo, hi):
    return max(lo, min(hi, int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))))


def draw(rng):
    kind = rng.choice(["points", "points", "contains", "within", "intersects", "intersects",
                       "lines", "build", "refresh", "serve"])
    handler = rng.choice(["count", "collect"])
    coord = "f64" if rng.random() < 0.2 else "f32"
    boxes = _log_int(rng, 1000, 10_000_000)
    queries = _log_int(rng, 100, 1_000_000)
    dist, side, qside = rng.choice(["uniform", "mixture"]), 1e-3, 0.0
    if kind == "points":
        side = math.sqrt(10.0 / boxes) if dist == "uniform" else 1e-3  # a few results each
    elif kind == "contains":
        dist, side, qside = "uniform", math.sqrt(80.0 / boxes), math.sqrt(1.0 / boxes)
    elif kind == "within":
        dist, side, qside = "uniform", math.sqrt(1.0 / boxes), math.sqrt(80.0 / boxes)
    elif kind in ("intersects", "lines"):
        dist, side, qside = "mixture", 1e-4, 5e-3
        if handler == "collect":  # bounded results: some 2e7 pairs
            queries = min(queries, max(100, int(2e10 / boxes)))
    elif kind in ("build", "refresh"):
        dist, side, queries = "uniform", math.sqrt(10.0 / boxes), min(queries, 100_000)
    else:
        handler, coord, dist, side, qside = "count", "f32", "mixture", 1e-4, 5e-3
        boxes, queries = min(boxes, 1_000_000), rng.randrange(8, 65)
    return dict(kind=kind, boxes=boxes, queries=queries, dist=dist, side=side, qside=qside,
                coord=coord, handler=handler)


# ------------------------------------------------------------------ inputs ----
def _dtype(case):
    return torch.float64 if case["coord"] == "f64" else torch.float32


def _boxes(case, g, n, side, means):
    dt = _dtype(case)
    if case["dist"] == "uniform":
        lo = torch.rand(n, 2, generator=g, device="cuda", dtype=dt)
        hi = lo + torch.rand(n, 2, generator=g, device="cuda", dtype=dt) * side
        return torch.cat([lo, hi.clamp_(max=1.0)], 1)
    comp = torch.randint(means.shape[0], (n,), generator=g, device="cuda")
    c = means[comp] + 0.02 * torch.randn(n, 2, generator=g, device="cuda", dtype=dt)
    c.clamp_(0.0, 1.0)
    half = 0.5 * torch.exp(math.log(max(side, 1e-30))
                           + torch.randn(n, 2, generator=g, device="cuda", dtype=dt))
    return torch.cat([c - half, c + half], 1)


def _queries(case, g, n, means):
    kind = case["kind"]
    if kind in ("points", "build", "refresh"):
        if case["dist"] == "uniform":
            return torch.rand(n, 2, generator=g, device="cuda", dtype=_dtype(case))
        return _boxes(case, g, n, 1e-4, means)[:, :2].contiguous()
    q = _boxes(case, g, n, case["qside"], means)
    if kind == "lines":  # either diagonal of the envelope
        flip = torch.rand(n, generator=g, device="cuda") < 0.5
        y0, y1 = torch.where(flip, q[:, 3], q[:, 1]), torch.where(flip, q[:, 1], q[:, 3])
        q = torch.stack([q[:, 0], y0, q[:, 2], y1], 1).contiguous()
    return q


def _generator(seed):
    g = torch.Generator(device="cuda")
    g.manual_seed(int(seed))
    return g


def _bits(n):
    return max(1, (max(n, 2) - 1).bit_length())


def prepare(case, seed):
    g = _generator(seed)
    kind, n, m = case["kind"], case["boxes"], case["queries"]
    s = dict(case=case)
    means = 0.1 + 0.8 * torch.rand(16, 2, generator=g, device="cuda", dtype=_dtype(case))
    boxes = _boxes(case, g, n, case["side"], means)
    ix = R.SpatialIndex(_dtype(case))
    # The reference only refits; under the default policy every few rounds of
    # updates become a rebuild, which the build case times.
    policy = N.RTS_REBUILD_NEVER if kind == "refresh" else N.RTS_REBUILD_SAH
    ix.Init(R.Config(rebuild_policy=policy))
    s["ix"] = ix
    if kind == "serve":
        ix.Insert(boxes)
        ix.Build()
        s["requests"] = _trace(case, g, m, means, seed)
        return s
    s["q"] = _queries(case, g, m, means)
    s["counter"] = R.SharedValue()
    if case["handler"] == "collect":
        s["queue"] = R.Queue(_rows(case))
    if kind == "build":
        s["boxes"] = boxes
        s["more"] = _boxes(case, g, max(1, n // 100), case["side"], means)
        return s
    ix.Insert(boxes)
    ix.Build()
    if kind == "refresh":
        pick = torch.randperm(n, generator=g, device="cuda")
        gone, moved = pick[:max(1, n // 1000)].sort()[0], pick[-max(1, n // 500):].sort()[0]
        shift = (torch.rand(moved.shape[0], 2, generator=g, device="cuda", dtype=boxes.dtype)
                 - 0.5) * case["side"]
        s["gone"] = gone.contiguous()
        s["moved"] = R.pack_updates(moved, boxes[moved] + torch.cat([shift, shift], 1),
                                    coord_t=boxes.dtype)
    return s


def _trace(case, g, m, means, seed):
    """A saturated mixed trace: 40% point, 30% within and 30% intersects
    requests, sizes log-uniform in [1, 20000]."""
    cpu = torch.Generator().manual_seed(int(seed))
    kinds = torch.rand(m, generator=cpu).tolist()
    sizes = torch.exp(torch.rand(m, generator=cpu) * math.log(2e4)).round().long().tolist()
    out = []
    for u, k in zip(kinds, sizes):
        q = _boxes(case, g, max(1, k), case["qside"], means)
        if u < 0.4:
            out.append(serve.Request(q[:, :2].contiguous(), P.kContains))
        else:
            out.append(serve.Request(q, P.kWithin if u < 0.7 else P.kIntersects))
    return out


# --------------------------------------------------------------------- run ----
def _query(s, arg):
    kind = s["case"]["kind"]
    if kind == "lines":
        s["ix"].QueryLines(P.kIntersects, s["q"], arg)
    else:
        s["ix"].Query(PRED.get(kind, P.kContains), s["q"], arg)


def _count(s):
    s["counter"].set(0)
    _query(s, s["counter"])
    return s["counter"].tensor.clone()


def _collect(s):
    """The pairs in (query, box) order: a table of query ids and one of box
    ids, -1 past the results."""
    case = s["case"]
    s["queue"].Clear()
    _query(s, s["queue"])
    pairs = s["queue"].pairs()
    k = pairs.shape[0]
    out = torch.full((2, _rows(case)), -1, dtype=torch.int32, device="cuda")
    if k:
        geom, query = pairs[:, 0].contiguous(), pairs[:, 1].contiguous()
        geom, query = R.sort_pairs(geom, query, key_bits=_bits(case["boxes"] + case["boxes"] // 50))
        query, geom = R.sort_pairs(query, geom, key_bits=_bits(case["queries"]))
        out[0, :k] = query
        out[1, :k] = geom
    return out


def _answer(s):
    return _collect(s) if s["case"]["handler"] == "collect" else _count(s)


def run(s):
    case = s["case"]
    kind = case["kind"]
    ix = s["ix"]
    if kind == "serve":
        # 3 batches in flight, each with room for 64M result pairs
        results, _ = serve.run(ix, s["requests"], arena_pairs=1 << 26, max_batch_queries=1 << 19,
                               chunk_queries=1 << 16, hash_results=1)
        signed = [r["hash"] - (1 << 64) if r["hash"] >> 63 else r["hash"] for r in results]
        return (torch.tensor([r["count"] for r in results], dtype=torch.int64),
                torch.tensor(signed, dtype=torch.int64))
    if kind == "build":
        ix.Clear()
        ix.Insert(s["boxes"])
        ix.Build()
        before = _answer(s)
        ix.Insert(s["more"])
        return before, _answer(s)
    if kind == "refresh":
        ix.Delete(s["gone"])
        ix.Update(s["moved"])
    return _answer(s)


# -------------------------------------------------------------------- work ----
def _rows(case):
    """Rows of a collecting case's queue and table: room for four times the
    expected pairs (the mixture's overlap varies with its means)."""
    return int(4 * _results(case)) + 4096


def _results(case):
    """Expected result pairs of the case's queries."""
    n, m, kind = case["boxes"], case["queries"], case["kind"]
    if kind in ("points", "build", "refresh"):
        if case["dist"] == "uniform":
            return m * n * 0.25 * case["side"] ** 2
        return m * n * 9.0 * 2.7 * case["side"] ** 2
    if kind == "contains":
        return m * n * (0.5 * max(case["side"] - case["qside"], 0.0)) ** 2
    if kind == "within":
        return m * n * (0.5 * max(case["qside"] - case["side"], 0.0)) ** 2
    return m * n * (4e-5 if kind == "lines" else 1e-3)


def work(case):
    """Bytes a pass cannot do without: its inputs and outputs once and, for
    queries, the boxes they report read once each (at most all of them)."""
    n, m, kind = case["boxes"], case["queries"], case["kind"]
    w = 2 if case["coord"] == "f64" else 1
    if kind == "serve":  # mean size 2e4 / ln 2e4; results dropped, but found
        q = m * 2e4 / math.log(2e4)
        return {"bytes": q * 13.0 + 16.0 * n + 0.6 * q * n * 1e-3 * 8, "flops": 0}
    qb = (8 if kind in ("points", "build", "refresh") else 16) * w
    hits = _results(case)
    b = m * qb + 16.0 * w * min(float(n), hits + m)
    if kind == "build":  # boxes in, boxes in tree order out, their ids; two lookups
        b = 2 * b + 1.01 * n * (16.0 * w + 16.0 + 4.0)
    elif kind == "refresh":  # every box in tree order read to bound it again
        b += n * 16.0 + (n // 1000) * 8 + (n // 500) * (8 + 16 * w)
    if case["handler"] == "collect":
        b += 8.0 * hits
    return {"bytes": b, "flops": 0}


def exact(case, seed):
    """Every output is a whole number and exact already."""
    return None
