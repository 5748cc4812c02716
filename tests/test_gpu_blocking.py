"""Short blocking copies, which report their own end: what they moved is where it belongs when the call returns."""

import numpy as np
import pytest

from memfabric_hybrid_amd import bm, native
from tests import gpu_util

pytestmark = pytest.mark.gpu

ROOM = 4 << 20


@pytest.fixture(scope="module")
def pool(lib):
    assert bm.initialize("tcp://127.0.0.1:0", 1, 0) == 0, native.last_error()
    handle = bm.create(1, 2 * ROOM, 2 * ROOM)
    yield handle
    handle.destroy()
    bm.uninitialize()


def _read(lib, addr, nbytes):
    out = np.empty(nbytes, dtype=np.uint8)
    assert lib.mfrt_memcpy(out.ctypes.data, addr, nbytes) == 0
    return out


# one workgroup, its edges; the first of several; the last copy with a word of its own on each route, the first without
SIZES = [1, 15, 16, 17, 4095, 16383, 16384, 16385, 65537, 131072, 131073, (1 << 20) - 1, 1 << 20, (1 << 20) + 1]


@pytest.mark.parametrize("route", ["hbm", "to_host", "from_host"])
def test_single_copies(lib, pool, route):
    dev, host = pool.peer_rank_ptr(0, bm.BmMemType.DEVICE), pool.peer_rank_ptr(0, bm.BmMemType.HOST)
    source, target = (host if route == "from_host" else dev), (host if route == "to_host" else dev) + ROOM
    rng = np.random.default_rng(5)
    data = rng.integers(0, 256, ROOM, dtype=np.uint8)
    assert lib.mfrt_memcpy(source, data.ctypes.data, ROOM) == 0
    for round_ in range(3):
        for size in SIZES:
            s, d = (0, 0) if round_ == 0 else (int(rng.integers(0, 300)), int(rng.integers(16, 300)))
            assert lib.mfrt_memset(target, 0xA5, size + 512) == 0
            assert pool.copy_data(source + s, target + d, size, bm.BmCopyType.G2G) == 0, native.last_error()
            got = gpu_util.host_view(target, size + 512).copy() if route == "to_host" else _read(lib, target, size + 512)
            assert np.array_equal(got[d:d + size], data[s:s + size]), (size, s, d)
            assert np.all(got[:d] == 0xA5) and np.all(got[d + size:] == 0xA5), (size, s, d)


@pytest.mark.parametrize("route", ["hbm", "to_host", "from_host"])
@pytest.mark.parametrize("count, most", [(2, 40000), (31, 4097), (128, 1000), (128, 8200), (129, 4000)])
def test_batches_one_behind_the_other(lib, pool, route, count, most):
    """Each batch reads what the one before it wrote."""
    dev, host = pool.peer_rank_ptr(0, bm.BmMemType.DEVICE), pool.peer_rank_ptr(0, bm.BmMemType.HOST)
    a, b = {"hbm": (dev, dev + ROOM), "to_host": (dev, host), "from_host": (host, dev)}[route]
    rng = np.random.default_rng(count)
    image = {a: rng.integers(0, 256, ROOM, dtype=np.uint8), b: rng.integers(0, 256, ROOM, dtype=np.uint8)}
    for addr, data in image.items():
        assert lib.mfrt_memcpy(addr, data.ctypes.data, ROOM) == 0
    for _ in range(20):
        sizes = rng.integers(1, most, count)
        slot = ROOM // count
        source, target = rng.permutation(count) * slot, rng.permutation(count) * slot + rng.integers(0, slot - most, count)
        for frm, to in ((a, b), (b, a)):
            assert pool.copy_data_batch(frm + source, to + target, sizes, count, bm.BmCopyType.G2G) == 0, native.last_error()
            for s, d, n in zip(source, target, sizes):
                image[to][d:d + n] = image[frm][s:s + n]
    for addr, data in image.items():
        assert np.array_equal(_read(lib, addr, ROOM), data)
