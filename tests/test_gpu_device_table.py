"""Tables in device memory whose segments are unlike the first ones, which decide how a table is shared out: lengths on both
sides of what a segment's own workgroups copy and of a listed piece, and lists that run over; on every route, and twice in a row,
so that a list left behind by the first call shows."""
import numpy as np
import pytest

from memfabric_hybrid_amd import native
from tests import gpu_util
from tests.test_gpu_xcopy import _random_bytes

pytestmark = pytest.mark.gpu

CHUNK = 4096
PIECE = 64 << 10
OWN = 4 * CHUNK                       # of a segment, where the first segments have one chunk


@pytest.fixture(scope="module")
def gpu(lib):
    assert lib.hybm_init(0, 0) == 0, native.last_error()
    yield lib
    lib.hybm_uninit()


class Pinned(gpu_util.PinnedBuffer):
    def upload(self, array):
        self.array[:] = array

    def download(self):
        return self.array.copy()


def _lengths(kind):
    edges = [1, 15, 16, 17, CHUNK - 1, CHUNK, CHUNK + 1, OWN - 1, OWN, OWN + 1, OWN + 16, OWN + PIECE - 1, OWN + PIECE, OWN + PIECE + 1,
             OWN + 3 * PIECE + 7, 0, 0, 3 << 20]
    if kind == "short first":
        return [0, 1, 100, 4000, 0, 7, 64, 16] + edges
    if kind == "long first":                                     # 64 parts, the most, and 1 MiB of every segment
        own = 64 * OWN
        return [0, 2 << 20] + edges + [own - 1, own, own + 1, own + PIECE + 1, 6 << 20]
    if kind == "few":                                            # fewer segments than the sample
        return [0, 5 << 20, 33]
    if kind == "one":
        return [9 << 20]
    return [5] * 8 + [OWN + 16 + i % 32 for i in range(11000)]   # "list": more pieces than the static list has room for


@pytest.mark.parametrize("kind,route,static", [
    ("short first", native.ROUTE_HBM, False), ("long first", native.ROUTE_HBM, False), ("few", native.ROUTE_HBM, False),
    ("one", native.ROUTE_HBM, False), ("short first", native.ROUTE_TO_HOST, False), ("long first", native.ROUTE_FROM_HOST, False),
    ("long first", native.ROUTE_HBM, True), ("list", native.ROUTE_HBM, True),
])
def test_table_unlike_its_first_segments(gpu, oracle, kind, route, static):
    lens = np.array(_lengths(kind), dtype=np.uint64)
    rng = np.random.default_rng(len(lens))
    steps = (lens + np.uint64(127)) // np.uint64(64) * np.uint64(64)
    at = np.concatenate(([0], np.cumsum(steps)[:-1])).astype(np.uint64)
    size = int(steps.sum()) + 64
    src = at + rng.integers(0, 16, len(lens)).astype(np.uint64)
    dst = at + rng.integers(0, 16, len(lens)).astype(np.uint64)
    sources = [_random_bytes(oracle, size, 7), _random_bytes(oracle, size, 8)]
    before = _random_bytes(oracle, size, 9)
    make = [Pinned if route == r else gpu_util.DeviceBuffer for r in (native.ROUTE_FROM_HOST, native.ROUTE_TO_HOST)]
    a, b = make[0](gpu, size), make[1](gpu, size)
    table = gpu_util.DeviceBuffer(gpu, len(lens) * 24)
    entry = gpu.mf_xcopy_device_table_static if static else gpu.mf_xcopy_device_table
    try:
        table.upload(np.stack([a.ptr + src, b.ptr + dst, lens], axis=1).astype(np.uint64).view(np.uint8).reshape(-1))
        for source in sources:
            a.upload(source)
            b.upload(before)
            assert entry(table.ptr, len(lens), route, None) == 0, native.last_error()
            assert gpu.mfrt_device_sync() == 0
            expect = before.copy()
            gpu_util.oracle_batch(oracle, source, expect, src, dst, lens)
            assert np.array_equal(b.download(), expect)
    finally:
        a.free()
        b.free()
        table.free()
