"""Served requests on an index without boxes: one that never held any, and one
cleared after a run with results, whose scratch the next run is given again.
Every request kind answers with no results: tiles (float envelopes and points)
and requests walked by launches of their own (segments, and every request on a
double index)."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

torch = pytest.importorskip("torch")
if not torch.cuda.is_available():
    pytest.skip("no GPU", allow_module_level=True)

import rtspatial_amd as R  # noqa: E402
from rtspatial_amd import serve as S  # noqa: E402
from gpu_util import dev, log  # noqa: E402

P = R.Predicate


@pytest.mark.parametrize("mode", ["batched", "plain"])
@pytest.mark.parametrize("cleared", [False, True])
@pytest.mark.parametrize("dtype", [np.float32, np.float64])
def test_requests_on_an_index_without_boxes(dtype, cleared, mode):
    log(f"serve without boxes dtype={np.dtype(dtype).name} cleared={cleared} mode={mode}")
    rng = np.random.default_rng(8)
    lo = rng.random((5000, 2)).astype(dtype)
    boxes = np.concatenate([lo, lo + dtype(0.02)], 1)
    ix = R.SpatialIndex(torch.float64 if dtype == np.float64 else torch.float32)
    ix.Init(R.Config())
    q4, q2 = dev(boxes[:700]), dev(np.ascontiguousarray(boxes[:300, :2]))
    reqs = [S.Request(queries=q4, predicate=P.kIntersects, collect=64),
            S.Request(queries=q4, predicate=P.kIntersects, collect=64, segments=True),
            S.Request(queries=q2, predicate=P.kContains, collect=64),
            S.Request(queries=q4, predicate=P.kWithin, collect=64),
            S.Request(queries=q4, predicate=P.kContains, collect=64, segments=True)]
    kw = dict(mode=mode, hash_results=1, slots=1, max_batch_queries=4096, arena_pairs=1 << 20)
    if cleared:
        # The run's counts and pairs stay behind in its scratch.
        ix.Insert(dev(boxes))
        res, _ = S.run(ix, reqs, **kw)
        assert min(res[0]["count"], res[1]["count"], res[2]["count"]) > 0
        ix.Clear()
    res, st = S.run(ix, reqs, **kw)
    assert st["requests"] == len(reqs) and st["results"] == 0 and st["relaunches"] == 0
    for i, r in enumerate(res):
        assert r["count"] == 0 and r["hash"] == 0 and not r["truncated"], i
        assert r["pairs"].shape[0] == 0, i
