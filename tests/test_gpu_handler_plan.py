"""Plans of calls with caller-compiled handlers and of the library's own calls
are apart: handlers walk the binary tree, a query per lane or wavefront, the
library's calls the packed tree."""
import ctypes

import numpy as np
import pytest

pytestmark = pytest.mark.gpu

torch = pytest.importorskip("torch")
if not torch.cuda.is_available():
    pytest.skip("no GPU", allow_module_level=True)

import rtspatial_amd as R  # noqa: E402
from rtspatial_amd import _native as N  # noqa: E402
from gpu_util import collect, count, dev, log, make_index  # noqa: E402
from test_gpu_handlers import THREAD, WAVE, X, run_summary  # noqa: E402,F401

P = R.Predicate
POINTS, ENVELOPES, LINES = N.RTS_QUERY_POINTS, N.RTS_QUERY_ENVELOPES, N.RTS_QUERY_LINES


def _plan(ix, pred, kind, n):
    p = N.rts_query_plan()
    N.check(N.lib().rts_index_query_plan(ix._handle(), int(pred), kind, n, ctypes.byref(p)))
    return p.traversal, p.sort_queries == 1, p.leaf_size


def _scene(n, nq, seed):
    rng = np.random.default_rng(seed)
    lo = rng.random((n, 2)).astype(np.float32)
    side = (rng.random((n, 2)) * 3.0 / np.sqrt(n)).astype(np.float32)
    return np.concatenate([lo, lo + side], 1), rng.random((nq, 2)).astype(np.float32)


def test_default_plans_of_handlers_calls():
    log("handlers' default plans")
    ix = make_index(_scene(100, 1, 1)[0], leaf_size=4)
    for pred, kind in ((P.kContains, POINTS), (P.kContains, ENVELOPES)):
        assert _plan(ix, pred, kind, (1 << 19) - 1) == (THREAD, False, 4)
        assert _plan(ix, pred, kind, 1 << 19) == (THREAD, True, 4)  # lanes share descents
    for pred, kind in ((P.kIntersects, ENVELOPES), (P.kWithin, ENVELOPES), (P.kIntersects, LINES)):
        assert _plan(ix, pred, kind, 65_535) == (WAVE, False, 4)
        assert _plan(ix, pred, kind, 65_536) == (WAVE, True, 4)
    forced = make_index(_scene(100, 1, 1)[0], traversal=WAVE, sort_queries=2)
    assert _plan(forced, P.kContains, POINTS, 1 << 20) == (WAVE, False, 8)


@pytest.mark.parametrize("collecting", [False, True])
def test_tuned_plans_are_apart_and_exact(X, oracle, collecting):
    b, q = _scene(150_000, 600_000, 2)
    log(f"tuned plans of both kinds collect={collecting}")
    ix = make_index(b)
    ix.Build()
    ix.Sync()
    before = ix.memory()["bvh"]
    r = ix.Autotune(P.kContains, dev(q[:70_000]), collect=collecting, sample=8192,
                    leaf_sizes=(16,), reps=2)
    trav, _, leaf = _plan(ix, P.kContains, POINTS, 1000)
    assert leaf == r["leaf_size"] and leaf in (8, 16) and trav in (THREAD, WAVE)
    # The tree made for the handlers' timing is gone.
    assert ix.memory()["bvh"] == before
    # Ordering 70k points costs more than their whole walk by octets; having
    # lost there it is not used at any size, as without a tuning.
    dq = dev(q)
    if r["traversal"] == THREAD and r["sort_queries"] == 2:
        R.profile_enable(True)
        R.profile_read()
        assert count(ix, P.kContains, dq) > 0
        assert R.profile_read()["query_order"][0] == 0
        R.profile_enable(False)
    tot, want, _ = oracle.RTree(b).checksums(oracle.CONTAINS, q)
    got, k = collect(ix, P.kContains, dq)
    assert k == tot and np.array_equal(np.bincount(got[:, 0], minlength=q.shape[0]), want)
    c, _, _, d = run_summary(X, ix, P.kContains, dq, 0)  # a handler's own plan
    assert np.array_equal(c, want) and np.array_equal(d, want)
