"""The tree that caller-compiled handlers walk is made when a view of it is
asked for. The view is complete for work on the stream it was asked for on,
whatever other stream its tree was queued on, and one taken while a graph is
being captured leaves nothing of the tree to the graph's replays."""
import ctypes

import numpy as np
import pytest

pytestmark = pytest.mark.gpu

torch = pytest.importorskip("torch")
if not torch.cuda.is_available():
    pytest.skip("no GPU", allow_module_level=True)

import rtspatial_amd as R  # noqa: E402
from gpu_util import dev, log, make_index  # noqa: E402
from test_gpu_graph import CAPTURE_THREAD_LOCAL, _check, _hip  # noqa: E402
from test_gpu_handlers import THREAD, WAVE, X  # noqa: E402,F401

P = R.Predicate


def _scene(n, nq, seed):
    rng = np.random.default_rng(seed)
    lo = rng.random((n, 2)).astype(np.float32)
    side = (rng.random((n, 2)) * 3.0 / np.sqrt(n)).astype(np.float32)
    return rng, np.concatenate([lo, lo + side], 1), rng.random((nq, 2)).astype(np.float32)


def _counts(oracle, b, q, alive):
    return oracle.RTree(b, alive=alive).checksums(oracle.CONTAINS, q)[1]


def _run(X, ix, q, out, trav, stream):
    rc = X.rtsx_count(ix._handle(), int(P.kContains), q.data_ptr(), q.shape[0], 1, 0, trav,
                      out.data_ptr(), ctypes.c_void_p(stream.cuda_stream))
    assert rc == 0, X.rtsx_last_error()


def _delete_some(rng, ix, alive):
    dead = rng.choice(alive.size, alive.size // 50, replace=False).astype(np.int64)
    ix.Delete(dev(dead))
    alive[dead] = 0
    ix.Build()
    ix.Sync()


def test_views_on_several_streams_at_once(X, oracle):
    rng, b, q = _scene(4_000_000, 20_000, 61)
    log("handler views on three streams at once, 4M boxes")
    alive = np.ones(b.shape[0], np.uint8)
    ix = make_index(b)
    ix.Build()
    ix.Sync()
    dq = dev(q)
    streams = [torch.cuda.Stream() for _ in range(3)]
    for step in range(2):
        want = _counts(oracle, b, q, alive)
        outs = [torch.full((q.shape[0],), -7, dtype=torch.int64, device="cuda") for _ in streams]
        torch.cuda.synchronize()
        for s, out in zip(streams, outs):  # the first queues the tree, the others follow at once
            _run(X, ix, dq, out, THREAD, s)
        torch.cuda.synchronize()
        for out in outs:
            assert np.array_equal(out.cpu().numpy().view(np.uint64), want), step
        ix.Sync()
        _delete_some(rng, ix, alive)  # the next view bounds the tree again


def test_view_taken_under_capture(X, oracle):
    hip = _hip()
    R.profile_enable(False)
    rng, b, q = _scene(200_000, 5_000, 62)
    log("handler views taken under capture")
    alive = np.ones(b.shape[0], np.uint8)
    ix = make_index(b)
    ix.Build()
    ix.Sync()
    dq = dev(q)
    s = torch.cuda.Stream()
    h = ctypes.c_void_p(s.cuda_stream)
    out = torch.full((q.shape[0],), -7, dtype=torch.int64, device="cuda")
    eager = torch.full_like(out, -7)
    for step in range(2):  # the tree is first built under capture, then bounded again
        want = _counts(oracle, b, q, alive)
        torch.cuda.synchronize()
        graph, exe = ctypes.c_void_p(), ctypes.c_void_p()
        _check(hip.hipStreamBeginCapture(h, CAPTURE_THREAD_LOCAL), "hipStreamBeginCapture")
        try:
            _run(X, ix, dq, out, THREAD, s)
        finally:
            _check(hip.hipStreamEndCapture(h, ctypes.byref(graph)), "hipStreamEndCapture")
        # Before any replay: eager calls see a whole tree.
        _run(X, ix, dq, eager, WAVE, torch.cuda.current_stream())
        torch.cuda.synchronize()
        assert np.array_equal(eager.cpu().numpy().view(np.uint64), want), step
        _check(hip.hipGraphInstantiate(ctypes.byref(exe), graph, None, None, ctypes.c_size_t(0)),
               "hipGraphInstantiate")
        try:
            for rep in range(3):
                out.fill_(-7)
                torch.cuda.synchronize()
                _check(hip.hipGraphLaunch(exe, h), "hipGraphLaunch")
                s.synchronize()
                assert np.array_equal(out.cpu().numpy().view(np.uint64), want), (step, rep)
                _run(X, ix, dq, eager, THREAD, s)
                s.synchronize()
                assert np.array_equal(eager.cpu().numpy().view(np.uint64), want), (step, rep)
        finally:
            hip.hipGraphExecDestroy(exe)
            hip.hipGraphDestroy(graph)
        _delete_some(rng, ix, alive)
