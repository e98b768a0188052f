"""Scratch kept between calls: calls of many sizes on several streams and
threads at once share the kept blocks and stay exact, and destroying the last
index gives the blocks back."""
import threading

import numpy as np
import pytest

pytestmark = pytest.mark.gpu

torch = pytest.importorskip("torch")
if not torch.cuda.is_available():
    pytest.skip("no GPU", allow_module_level=True)

import rtspatial_amd as R  # noqa: E402
from gpu_util import canon, dev, log, make_index  # noqa: E402

P = R.Predicate


def test_streams_and_threads_share_scratch(oracle):
    log("workspace: 4 threads x 12 calls on streams of their own")
    from rtspatial_amd import workloads as W
    b, q = W.config2(50_000, 70_000)
    ix = make_index(b)
    ix.Build()
    ix.Sync()
    tree = oracle.RTree(b)
    sizes = [1, 70, 900, 5_000, 20_000, 70_000]
    want = {n: tree.pairs(oracle.INTERSECTS, q[:n]) for n in sizes}
    dq = dev(q)
    torch.cuda.synchronize()
    errors = []

    def work(t):
        try:
            s = torch.cuda.Stream()
            for k in range(12):
                n = sizes[(k + t) % len(sizes)]
                with torch.cuda.stream(s):
                    queue = R.Queue(want[n].shape[0] + 8)
                    ix.Query(P.kIntersects, dq[:n], queue, stream=s)
                    got = queue.pairs(s)
                assert np.array_equal(canon(got), want[n]), (t, k, n)
        except Exception as e:  # reported by the main thread
            errors.append(repr(e))

    threads = [threading.Thread(target=work, args=(t,)) for t in range(4)]
    for t in threads:
        t.start()
    for t in threads:
        t.join()
    assert not errors, errors
    ix.Sync()


def test_last_index_gives_scratch_back():
    log("workspace: given back with the last index")
    import gc
    gc.collect()
    rng = np.random.default_rng(5)
    boxes = rng.random((1000, 2)).astype(np.float32)
    boxes = np.concatenate([boxes, boxes + np.float32(0.01)], 1)
    ix = make_index(boxes)
    q = dev(np.repeat(boxes, 400, 0))  # 400k queries: some 1.6 GB of range logs
    queue = R.Queue(8_000_000)
    ix.Query(P.kIntersects, q, queue)
    torch.cuda.synchronize()
    before = torch.cuda.mem_get_info()[0]
    del ix
    gc.collect()
    torch.cuda.synchronize()
    assert torch.cuda.mem_get_info()[0] - before > (1 << 30)
