"""dpc_bytes_to_bits_indexed over maps that do not ascend: descending, in clusters whose
order changes within a wave, shuffled within a window and over all, at the ends of a
wave's window.  Against numpy, and a descending map in about an ascending one's time."""
import numpy as np
import pytest

from pipeline_amd import _lib
from pipeline_amd import device as dev

pytestmark = pytest.mark.gpu


def maps(n, rng):
    yield "descending", np.arange(n)[::-1]
    yield "two clusters, the high one first", np.where(np.arange(n) % 512 < 450, np.arange(n) + 100_000, np.arange(n))
    yield "two clusters, the low one first", np.where(np.arange(n) % 512 < 60, np.arange(n), np.arange(n) + 100_000)
    yield "shuffled within 4096", np.concatenate([a + rng.permutation(min(4096, n - a)) for a in range(0, n, 4096)])
    yield "a window's ends", np.where(np.arange(n) % 64 == 1, np.arange(n) + 8_191, np.arange(n) * 0 + np.arange(n) // 64 * 64 + np.arange(n) % 64 // 2 * 2)
    yield "random", rng.permutation(n)


@pytest.mark.parametrize("n", [64, 513, 5_000, 70_001])
def test_orders(n):
    rng = np.random.default_rng(n)
    lib = _lib.load()
    for kind, index in maps(n, rng):
        for share in (0.05, 1.0):
            data = (rng.random(n) < share).astype(np.uint8)
            n_bits = int(index.max()) + 1
            want = np.zeros((n_bits + 63) // 64 * 64, np.uint8)
            want[index[data != 0]] = 1
            d_bytes, d_index = dev.DeviceArray.from_host(data), dev.DeviceArray.from_host(np.ascontiguousarray(index, np.uint32))
            d_bits = dev.DeviceArray(want.size // 32, np.uint32)
            d_bits.fill_u32(0)
            _lib.check(lib.dpc_bytes_to_bits_indexed(d_bytes.ptr, d_index.ptr, n, d_bits.ptr, n_bits, None))
            got = np.unpackbits(d_bits.download().view(np.uint8), bitorder="little")
            assert np.array_equal(got, want), kind
            for d in (d_bytes, d_index, d_bits):
                d.free()


def test_descending_takes_an_ascending_maps_time():
    """Both gather a wave's 512 bits in one window; bit by bit the descending one took
    four and a half times as long."""
    n, lib, stream = 200_003, _lib.load(), dev.Stream()
    data, bits = dev.DeviceArray.from_host(np.ones(n, np.uint8)), dev.DeviceArray((n + 31) // 32, np.uint32)
    best = []
    for index in (np.arange(n), np.arange(n)[::-1]):
        d_index = dev.DeviceArray.from_host(np.ascontiguousarray(index, np.uint32))
        times = []
        for _ in range(20):
            a, b = dev.Event(), dev.Event()
            a.record(stream.handle)
            for _ in range(20):
                _lib.check(lib.dpc_bytes_to_bits_indexed(data.ptr, d_index.ptr, n, bits.ptr, n, stream.handle))
            b.record(stream.handle)
            stream.sync()
            times.append(a.elapsed_ms(b))
            a.destroy()
            b.destroy()
        best.append(min(times))
        d_index.free()
    for d in (data, bits, stream):
        d.destroy() if d is stream else d.free()
    assert best[1] < 2.0 * best[0]
