"""Scratch kept between calls gives way: to the index's own arrays when the
device is full, and to the rest of the program on request."""
import gc

import numpy as np
import pytest

pytestmark = pytest.mark.gpu

torch = pytest.importorskip("torch")
if not torch.cuda.is_available():
    pytest.skip("no GPU", allow_module_level=True)

import rtspatial_amd as R  # noqa: E402
from rtspatial_amd import serve as S  # noqa: E402
from gpu_util import count, dev, log, make_index  # noqa: E402

P = R.Predicate
GIB = 1 << 30


def _free():
    torch.cuda.synchronize()
    return torch.cuda.mem_get_info()[0]


def _served(boxes):
    """An index that has served requests: the slot's scratch (some 14 GiB) is kept."""
    ix = make_index(boxes)
    ix.Build()
    ix.Sync()
    before = _free()
    res, _ = S.run(ix, [S.Request(queries=dev(boxes))], slots=1)
    assert res[0]["count"] >= boxes.shape[0]
    held = before - _free()
    assert held > 8 * GIB, held
    return ix, held


def _boxes():
    lo = np.random.default_rng(6).random((1000, 2)).astype(np.float32)
    return np.concatenate([lo, lo + np.float32(0.01)], 1)


def test_scratch_is_released_on_request():
    log("scratch released on request")
    gc.collect()
    boxes = _boxes()
    ix, held = _served(boxes)
    before = _free()
    R.release_scratch()
    assert _free() - before > held - GIB
    assert count(ix, P.kIntersects, boxes) >= 1000  # and leased again
    ix.Sync()


def test_index_grows_into_kept_scratch():
    log("an index grows on a full device")
    gc.collect()
    torch.cuda.empty_cache()
    ix, _ = _served(_boxes())
    n = 60_000_000  # some 4 GB of arrays
    lo = torch.rand((n, 2), device="cuda")
    b = torch.cat([lo, lo + 1e-5], 1).contiguous()
    del lo
    torch.cuda.empty_cache()
    rest = torch.empty(_free() - 2 * GIB, dtype=torch.uint8, device="cuda")
    try:
        ix.Insert(b)
        ix.Build()
        ix.Sync()
    finally:
        del rest
        torch.cuda.empty_cache()
    q = np.float32([[-1, -1, 3, 3]])
    assert count(ix, P.kWithin, q) == n + 1000
    ix.Sync()


def test_failed_growth_leaves_a_usable_index():
    log("an index whose growth failed is cleared and used again")
    gc.collect()
    torch.cuda.empty_cache()
    boxes = _boxes()
    ix = make_index(np.concatenate([boxes] * 3))
    assert count(ix, P.kIntersects, boxes) >= 3000
    n = 60_000_000
    lo = torch.rand((n, 2), device="cuda")
    b = torch.cat([lo, lo + 1e-5], 1).contiguous()
    del lo
    torch.cuda.empty_cache()
    ix.Insert(b)  # (its copy by id; the trees take another 2.4 GB)
    R.release_scratch()
    rest = torch.empty(_free() - GIB, dtype=torch.uint8, device="cuda")
    try:
        with pytest.raises(R.RtsError, match="out of memory"):
            ix.Build()
    finally:
        del rest
        torch.cuda.empty_cache()
    # Fewer boxes than the arrays held before the growth.
    ix.Clear()
    ix.Insert(dev(boxes))
    assert count(ix, P.kIntersects, boxes) >= 1000
    ix.Sync()
