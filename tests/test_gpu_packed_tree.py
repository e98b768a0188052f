"""The packed tree at the sizes where its levels, octets and workgroups fill or
just do not: every predicate under both walks, counted and collected, equals
the oracle, with whole blocks and whole subtrees deleted, inverted boxes and
queries that are infinite, empty or NaN."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

torch = pytest.importorskip("torch")
if not torch.cuda.is_available():
    pytest.skip("no GPU", allow_module_level=True)

import rtspatial_amd as R  # noqa: E402
from rtspatial_amd import _native as N  # noqa: E402
from gpu_util import canon, collect, count, dev, log, make_index  # noqa: E402

P = R.Predicate
SIZES = [1, 2, 7, 8, 9, 63, 64, 65, 511, 512, 513, 4095, 4096, 4097, 32767, 32769, 262145]


def _boxes(rng, n):
    lo = rng.random((n, 2)).astype(np.float32)
    side = (rng.random((n, 2)) * 2.0 / np.sqrt(n)).astype(np.float32)
    b = np.concatenate([lo, lo + side], 1)
    b[::17] = b[::17][:, [2, 3, 0, 1]]  # corners swapped: matches what its coordinates say
    return np.ascontiguousarray(b)


def _queries(rng, n):
    c = rng.random((40, 2)).astype(np.float32)
    h = (rng.random((40, 2)) * 3.0 / np.sqrt(n)).astype(np.float32)
    inf, nan = np.float32(np.inf), np.float32(np.nan)
    extra = np.float32([[-1, -1, 2, 2], [-inf, -inf, inf, inf], [0.25, 0.25, 0.75, 0.75],
                        [0.5, 0.5, 0.5, 0.5], [nan, 0, 1, 1], [0.9, 0.9, 0.1, 0.1],
                        [inf, inf, inf, inf], [-inf, -inf, 0.5, 0.5]])
    return np.ascontiguousarray(np.concatenate([np.concatenate([c - h, c + h], 1), extra]))


@pytest.mark.parametrize("mode", [N.RTS_TRAVERSAL_THREAD, N.RTS_TRAVERSAL_WAVE])
@pytest.mark.parametrize("n", SIZES)
def test_edges_of_levels_and_blocks(oracle, n, mode):
    log(f"packed tree n={n} traversal={mode}")
    rng = np.random.default_rng(n)
    b, q = _boxes(rng, n), _queries(rng, n)
    alive = np.ones(n, np.uint8)
    ix = make_index(b, traversal=mode)
    for step in range(2):
        for pred, qq in ((P.kIntersects, q), (P.kWithin, q), (P.kContains, q),
                         (P.kContains, np.ascontiguousarray(q[:, :2]))):
            points = qq.shape[1] == 2
            want = oracle.bf_pairs(int(pred), b, qq, alive=alive)
            got, k = collect(ix, pred, qq)
            assert k == want.shape[0] and np.array_equal(got, want), (step, int(pred), points)
            assert count(ix, pred, qq) == want.shape[0], (step, int(pred), points)
        # Everything in one part of the scene dies (its nodes have no live
        # leaf), and a few boxes elsewhere (nodes inside a query that are not
        # whole); then the tree is bounded again in place.
        dead = np.flatnonzero((b[:, 0] < 0.4) | (np.arange(n) % 29 == 3)).astype(np.int64)
        if dead.size:
            ix.Delete(dev(dead))
            alive[dead] = 0
    ix.Sync()


@pytest.mark.parametrize("n", [9, 513, 40_000])
def test_every_box_deleted(n):
    log(f"packed tree, all of {n} boxes deleted")
    rng = np.random.default_rng(n)
    ix = make_index(_boxes(rng, n))
    q = _queries(rng, n)
    assert count(ix, P.kIntersects, q) > 0
    ix.Delete(dev(np.arange(n, dtype=np.int64)))
    for pred in (P.kIntersects, P.kWithin, P.kContains):
        assert count(ix, pred, q) == 0
    ix.Build()
    new = np.float32([[0.1, 0.1, 0.2, 0.2], [0.5, 0.5, 0.6, 0.6], [0.9, 0.2, 0.95, 0.3]])
    ix.Update((dev(np.arange(3, dtype=np.int64)), dev(new)))
    assert count(ix, P.kWithin, np.float32([[-9, -9, 9, 9]])) == 3
    ix.Sync()


@pytest.mark.parametrize("nq", [24_575, 24_576, 131_071, 131_077])
@pytest.mark.parametrize("heavy", [0.0, 0.02, 0.9])
def test_light_and_heavy_queries_together(oracle, nq, heavy):
    # Around the sizes at which octets take the queries first (8, then 16 to a
    # ticket), with none, few or most of them too heavy for an octet: windows
    # of thousands of boxes, and thin ones that meet many blocks.
    log(f"light and heavy queries nq={nq} heavy={heavy}")
    rng = np.random.default_rng(nq + int(heavy * 100))
    n = 60_000
    b = _boxes(rng, n)
    c = rng.random((nq, 2)).astype(np.float32)
    h = (rng.random((nq, 2)) * 2.0 / np.sqrt(n)).astype(np.float32)
    big = rng.random(nq) < heavy
    if heavy < 0.5:
        h[big] = (rng.random((int(big.sum()), 2)) * 0.06).astype(np.float32)
        h[big[:] & (np.arange(nq) % 2 == 0), 1] = 1e-4  # thin
    else:
        h[big] = np.float32(0.02)
    q = np.ascontiguousarray(np.concatenate([c - h, c + h], 1))
    tree = oracle.RTree(b)
    ix = make_index(b, traversal=N.RTS_TRAVERSAL_WAVE)
    for pred in (P.kIntersects, P.kWithin):
        want = tree.pairs(int(pred), q)
        assert count(ix, pred, q) == want.shape[0]
        got, k = collect(ix, pred, q, capacity=want.shape[0] + 1)
        assert k == want.shape[0] and np.array_equal(got, want)
    ix.Sync()


def test_large_windows_outgrow_their_log(oracle):
    # Some 5000 partly covered blocks per query: more than a query's log holds.
    log("windows that outgrow their logs")
    rng = np.random.default_rng(77)
    n = 2_000_000
    b = _boxes(rng, n)
    b[:, 2:] = b[:, :2]  # points, so that a thin window meets no whole node
    q = np.float32([[-1, y, 2, y + 0.004] for y in (0.1, 0.35, 0.6, 0.85)] + [[-1, -1, 2, 2]])
    tree = oracle.RTree(b)
    ix = make_index(b)
    want = tree.pairs(oracle.INTERSECTS, q)
    got, k = collect(ix, P.kIntersects, q, capacity=want.shape[0] + 1)
    assert k == want.shape[0] and np.array_equal(got, want)
    ix.Sync()


@pytest.mark.parametrize("nq,giants", [(1, [0]), (5, [4]), (3000, [0, 1499, 1500, 2999]),
                                       (40_000, [7, 39_999]), (40_000, [])])
def test_write_windows(oracle, nq, giants):
    # Waves write windows of the output: queries of 1e5 results that take many
    # windows, long stretches of queries without results, and the rest of a few
    # results; each query's pairs together, in query order; into a queue with
    # room for all and for some.
    log(f"write windows nq={nq} giants={giants}")
    rng = np.random.default_rng(nq)
    n = 120_000
    b = _boxes(rng, n)
    c = rng.random((nq, 2)).astype(np.float32)
    c[nq // 3: nq // 2] += 5  # off the boxes
    h = np.full((nq, 2), 1.5 / np.sqrt(n), np.float32)
    h[giants] = 0.45
    c[giants] = 0.5
    q = np.ascontiguousarray(np.concatenate([c - h, c + h], 1))
    want = oracle.RTree(b).pairs(oracle.INTERSECTS, q)
    ix = make_index(b)
    queue = R.Queue(want.shape[0] + 8)
    ix.Query(P.kIntersects, dev(q), queue)
    assert queue.size() == want.shape[0]
    assert np.array_equal(canon(queue.pairs()), want)
    ids = queue.pairs()[:, 1].cpu().numpy()
    assert (np.diff(ids.astype(np.int64)) >= 0).all()
    some = R.Queue(want.shape[0] // 2 + 1)
    ix.Query(P.kIntersects, dev(q), some)
    assert some.size() == want.shape[0]
    # The slots of the first half of the results, each written once.
    assert np.array_equal(some.pairs()[:, 1].cpu().numpy(), ids[:some.capacity()])
    a, b = canon(some.pairs()).astype(np.uint64), want.astype(np.uint64)
    a, b = a[:, 0] << np.uint64(32) | a[:, 1], b[:, 0] << np.uint64(32) | b[:, 1]
    assert np.unique(a).size == a.size and np.isin(a, b).all()
    ix.Sync()
