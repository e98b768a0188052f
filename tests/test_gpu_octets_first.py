"""Calls large enough for octets to take the queries first (from 24,576 queries
on 256 CUs, 16 to a ticket from 131,072), of light and heavy queries together,
where the float tests of a single tree do not reach: double queries, a tree of
recent inserts beside the main one (the second walk takes the first's lists,
tickets and logs), and served requests that are walked by launches of their own
(octets without a log)."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

torch = pytest.importorskip("torch")
if not torch.cuda.is_available():
    pytest.skip("no GPU", allow_module_level=True)

import rtspatial_amd as R  # noqa: E402
from rtspatial_amd import _native as N  # noqa: E402
from rtspatial_amd import serve as S  # noqa: E402
from gpu_util import canon, collect, count, dev, log, make_index  # noqa: E402

P = R.Predicate
NB = 20_000


def _boxes(rng, dtype):
    lo = rng.random((NB, 2))
    b = np.concatenate([lo, lo + rng.random((NB, 2)) * 2.0 / np.sqrt(NB)], 1).astype(dtype)
    return np.ascontiguousarray(b)


def _queries(rng, b, nq, heavy):
    """Small windows, a third of them within 1e-13 of a box's corners, and a
    share of windows of thousands of boxes."""
    c = rng.random((nq, 2))
    h = rng.random((nq, 2)) * 1.5 / np.sqrt(NB)
    big = rng.random(nq) < heavy
    h[big] = 0.02 if heavy >= 0.5 else rng.random((int(big.sum()), 1)) * 0.1
    q = np.concatenate([c - h, c + h], 1)
    tie = (rng.random(nq) < 1 / 3) & ~big
    src = b[rng.integers(0, NB, int(tie.sum()))].astype(np.float64)
    q[tie] = src + rng.choice([-1e-13, 0.0, 1e-13], size=src.shape)
    return np.ascontiguousarray(q.astype(b.dtype))


def _want(oracle, pred, b, q, alive=None, lines=False):
    f = oracle.bf_pairs64 if b.dtype == np.float64 else oracle.bf_pairs
    return f(int(pred), b, q, alive=alive, lines=lines)


def _check(ix, pred, q, want):
    assert count(ix, pred, q) == want.shape[0]
    got, k = collect(ix, pred, q, capacity=want.shape[0] + 1)
    assert k == want.shape[0] and np.array_equal(got, want)


@pytest.mark.parametrize("heavy", [0.02, 0.9])
@pytest.mark.parametrize("nq", [24_576, 131_077])
def test_double_queries(oracle, nq, heavy):
    log(f"octets first, double, nq={nq} heavy={heavy}")
    rng = np.random.default_rng(nq + int(100 * heavy))
    b = _boxes(rng, np.float64)
    q = _queries(rng, b, nq, heavy)
    ix = make_index(b, traversal=N.RTS_TRAVERSAL_WAVE)
    for pred in (P.kIntersects, P.kWithin):
        _check(ix, pred, q, _want(oracle, pred, b, q))
    ix.Sync()


@pytest.mark.parametrize("dtype", [np.float32, np.float64])
@pytest.mark.parametrize("nq", [24_576, 131_077])
def test_with_a_tree_of_recent_inserts(oracle, nq, dtype):
    log(f"octets first, two trees, nq={nq} {np.dtype(dtype).name}")
    rng = np.random.default_rng(nq)
    b = _boxes(rng, dtype)
    q = _queries(rng, b, nq, 0.02)
    alive = np.ones(NB, np.uint8)
    ix = make_index(b[:-3000], traversal=N.RTS_TRAVERSAL_WAVE, insert_delta_pct=20)
    ix.Build()
    ix.Insert(dev(b[-3000:]))
    dead = rng.choice(NB, 500, replace=False).astype(np.int64)
    ix.Delete(dev(dead))
    alive[dead] = 0
    for pred in (P.kIntersects, P.kWithin):
        _check(ix, pred, q, _want(oracle, pred, b, q, alive))
    assert ix.stats()["delta_boxes"] == 3000
    ix.Sync()


@pytest.mark.parametrize("dtype", [np.float32, np.float64])
def test_served_requests_with_launches_of_their_own(oracle, dtype):
    log(f"octets first, served, {np.dtype(dtype).name}")
    rng = np.random.default_rng(9)
    b = _boxes(rng, dtype)
    host = []
    for nq, pred, lines in ((30_000, P.kIntersects, True), (26_001, P.kIntersects, False),
                            (24_577, P.kWithin, False), (40_000, P.kContains, False)):
        q = _queries(rng, b, nq, 0.01)
        if lines:  # short segments, and long ones that meet many boxes
            q[::200, 2:] = 1 - q[::200, :2]
        host.append((np.ascontiguousarray(q[:, :2]) if pred == P.kContains else q, pred, lines))
    want = [_want(oracle, p, b, q, lines=s) for q, p, s in host]
    reqs = [S.Request(queries=dev(q), predicate=p, collect=w.shape[0] + 8, segments=s)
            for (q, p, s), w in zip(host, want)]
    ix = make_index(b)
    res, st = S.run(ix, reqs, slots=2, max_batch_queries=1 << 17, arena_pairs=1 << 25)
    assert st["requests"] == len(reqs)
    for i, (rr, w) in enumerate(zip(res, want)):
        assert rr["count"] == w.shape[0] and w.shape[0] > 0, i
        assert np.array_equal(canon(rr["pairs"]), w), i
