"""The radix sort at the edges of its tiles and digits: key widths around the
digit and pass limits, sizes around a tile and around the large-tile limit,
keys with bits above the sorted ones, values given or numbered, input in
place and in pinned memory. The order is the stable order of the low bits."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

torch = pytest.importorskip("torch")
if not torch.cuda.is_available():
    pytest.skip("no GPU", allow_module_level=True)

import rtspatial_amd as R  # noqa: E402
from rtspatial_amd import _native as N  # noqa: E402
from gpu_util import dev, log  # noqa: E402


def _want(keys, bits):
    low = keys.astype(np.uint64) & np.uint64((1 << bits) - 1)
    return np.argsort(low, kind="stable")


@pytest.mark.parametrize("bits", [1, 7, 8, 9, 10, 11, 18, 20, 21, 30, 31, 32])
@pytest.mark.parametrize("n", [1, 2, 63, 2047, 2048, 2049, 50_000, (1 << 19) - 1, 1 << 19,
                               (1 << 19) + 8193])
def test_sort_edges(n, bits):
    if n > 100_000 and bits not in (9, 10, 20, 30, 32):
        pytest.skip("large sizes: one width per digit size")
    log(f"sort n={n} bits={bits}")
    rng = np.random.default_rng(n * 37 + bits)
    keys = rng.integers(0, 1 << 32, size=n, dtype=np.uint64).astype(np.uint32)  # high bits set
    if n > 100:
        keys[n // 2:] = keys[0]  # long runs of one digit
    vals = rng.integers(0, 1 << 32, size=n, dtype=np.uint64).astype(np.uint32)
    order = _want(keys, bits)
    dk, dv = dev(keys.view(np.int32)), dev(vals.view(np.int32))
    k, v = R.sort_pairs(dk, dv, key_bits=bits)
    assert np.array_equal(k.cpu().numpy().view(np.uint32), keys[order])
    assert np.array_equal(v.cpu().numpy().view(np.uint32), vals[order])
    assert np.array_equal(dk.cpu().numpy().view(np.uint32), keys)  # the input is left alone
    k, v = R.sort_pairs(dk, None, key_bits=bits)
    assert np.array_equal(v.cpu().numpy().view(np.uint32), order.astype(np.uint32))


@pytest.mark.parametrize("bits", [10, 20])  # an odd and an even number of passes
def test_sort_in_place_and_from_pinned_memory(bits):
    log(f"sort in place and from pinned memory, bits={bits}")
    rng = np.random.default_rng(bits)
    keys = rng.integers(0, 1 << bits, size=70_001, dtype=np.uint64).astype(np.uint32)
    order = _want(keys, bits)
    s = torch.cuda.current_stream().cuda_stream
    k = dev(keys.view(np.int32))
    v = dev(np.arange(keys.size, dtype=np.int32))
    N.check(N.lib().rts_sort_pairs(k.data_ptr(), v.data_ptr(), k.data_ptr(), v.data_ptr(),
                                   keys.size, bits, s), "in place")
    assert np.array_equal(k.cpu().numpy().view(np.uint32), keys[order])
    assert np.array_equal(v.cpu().numpy(), order.astype(np.int32))
    pk = torch.from_numpy(keys.view(np.int32).copy()).pin_memory()
    ko, vo = torch.empty_like(k), torch.empty_like(v)
    N.check(N.lib().rts_sort_pairs(pk.data_ptr(), None, ko.data_ptr(), vo.data_ptr(), keys.size,
                                   bits, s), "pinned")
    assert np.array_equal(ko.cpu().numpy().view(np.uint32), keys[order])
    assert np.array_equal(vo.cpu().numpy(), order.astype(np.int32))
