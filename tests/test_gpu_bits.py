"""dpc_bytes_to_bits_indexed where its waves' windows end: slot counts around one
wave's and one workgroup's share, maps that ascend, descend, jump between two
places, spread far apart or have no order, indices at and beyond n_bits, and bits
that were set before.  Against a bit-by-bit reference in numpy."""
import numpy as np
import pytest

from pipeline_amd import _lib
from pipeline_amd import device as dev

pytestmark = pytest.mark.gpu


def index_map(kind, n, rng):
    if kind == "none":
        return None
    if kind == "ascending":
        return np.cumsum(rng.integers(1, 4, n)).astype(np.uint32)
    if kind == "descending":
        return np.arange(n)[::-1].astype(np.uint32)
    if kind == "two places":
        return np.where(np.arange(n) % 512 < 300, np.arange(n) + 50_000, np.arange(n)).astype(np.uint32)
    if kind == "far apart":
        return (np.arange(n, dtype=np.uint64) * 997 % 3_000_017).astype(np.uint32)
    return rng.permutation(n).astype(np.uint32)


@pytest.mark.parametrize("kind", ["none", "ascending", "descending", "two places", "far apart", "random"])
@pytest.mark.parametrize("n", [1, 63, 511, 512, 513, 2_047, 2_048, 2_049, 70_001])
def test_bits(n, kind):
    rng = np.random.default_rng(n)
    lib = _lib.load()
    index = index_map(kind, n, rng)
    at = np.arange(n) if index is None else index.astype(np.int64)
    for share, cut in ((0.02, 0), (0.7, 1), (1.0, n // 3)):
        n_bits = max(int(at.max()) + 1 - cut, 1)
        data = (rng.random(n) < share).astype(np.uint8) * rng.integers(1, 256, n).astype(np.uint8)
        words = (n_bits + 31) // 32
        before = np.zeros(words, np.uint32)
        before[:: 5] = 0x80000001
        want = np.unpackbits(before.view(np.uint8), bitorder="little")
        hit = at[data != 0]
        want[hit[hit < n_bits]] = 1
        d_bytes, d_bits = dev.DeviceArray.from_host(data), dev.DeviceArray.from_host(before)
        d_index = None if index is None else dev.DeviceArray.from_host(index)
        _lib.check(lib.dpc_bytes_to_bits_indexed(d_bytes.ptr, None if index is None else d_index.ptr, n, d_bits.ptr, n_bits,
                                                 None))
        got = np.unpackbits(d_bits.download().view(np.uint8), bitorder="little")
        assert np.array_equal(got, want)
        for d in (d_bytes, d_bits, d_index):
            if d is not None:
                d.free()
