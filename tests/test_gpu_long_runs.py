"""Long runs of leaves in a query's log, written as whole lines of the output
from the first line that starts inside the run: at every place of a run's start
in its line, in a queue whose data starts anywhere, and in one that ends inside
a run."""
import ctypes

import numpy as np
import pytest

pytestmark = pytest.mark.gpu

torch = pytest.importorskip("torch")
if not torch.cuda.is_available():
    pytest.skip("no GPU", allow_module_level=True)

import rtspatial_amd as R  # noqa: E402
from rtspatial_amd import _native as N  # noqa: E402
from gpu_util import canon, dev, log, make_index  # noqa: E402

P = R.Predicate
NB = 6_000


def _scene():
    rng = np.random.default_rng(31)
    p = rng.random((NB, 2)).astype(np.float32)
    b = np.concatenate([p, p], 1)
    q = [[-1, -1, 2, 2]]
    for k in range(17):  # a query of k results moves the next one by k pairs
        x = b[k]
        q += [[x[0], x[1], x[0], x[1]]] * (k % 3) + [[-1, -1, 2, 2], [0.1 + k * 0.01, -1, 0.9, 2]]
    return b, np.float32(q)


@pytest.mark.parametrize("shift", [0, 1, 2, 15, 16, 17])
def test_runs_into_a_queue_that_starts_anywhere(oracle, shift):
    log(f"long runs, queue data at pair {shift}")
    b, q = _scene()
    want = oracle.bf_pairs(oracle.WITHIN, b, q)
    ix = make_index(b, traversal=N.RTS_TRAVERSAL_WAVE)
    n = want.shape[0]
    for cap in (n, n - 1, n - 700, n // 2 + 3):
        data = torch.full((n + 64, 2), -9, dtype=torch.int32, device="cuda")
        counter = torch.zeros(1, dtype=torch.int64, device="cuda")
        words = torch.tensor([data.data_ptr() + 8 * shift, cap, counter.data_ptr()],
                             dtype=torch.int64, device="cuda")
        dq = dev(q)
        N.check(N.lib().rts_index_query_envelopes(
            ix._handle(), int(P.kWithin), dq.data_ptr(), q.shape[0], N.RTS_HANDLER_COLLECT,
            words.data_ptr(), ctypes.c_void_p(torch.cuda.current_stream().cuda_stream)), "query")
        ix.Sync()
        assert int(counter.item()) == n
        assert (data[:shift] == -9).all() and (data[shift + cap:] == -9).all(), cap
        got = canon(data[shift:shift + cap])
        if cap == n:
            assert np.array_equal(got, want)
        else:  # the first pairs in query order, each once
            key = lambda a: a[:, 0].astype(np.uint64) << np.uint64(32) | a[:, 1].astype(np.uint64)
            assert np.unique(key(got)).size == cap and np.isin(key(got), key(want)).all(), cap
