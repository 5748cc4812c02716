"""Batches and device-resident tables captured into a HIP graph.  A graph keeps the arguments of its launches, not what
they point to: a batch must travel in the arguments, whatever its size, and a replay must not share the list of long
segments with a plain call.  Every replay is compared with the oracle, after plain calls of other batches that go through
all the library's descriptor slots."""
import threading

import numpy as np
import pytest

from memfabric_hybrid_amd import native
from tests import gpu_util

pytestmark = pytest.mark.gpu

POOL = 128 << 20
HALF = POOL // 2


@pytest.fixture(scope="module")
def gpu(lib):
    assert lib.hybm_init(0, 0) == 0, native.last_error()
    yield lib
    lib.hybm_uninit()


def _batch(kind, seed):
    """Offsets and lengths; destinations in the upper half, no two of them overlapping."""
    rng = np.random.default_rng(seed)
    if kind == "few, apart modulo 16":                       # 30 MB in three segments: stores held in waves of 16 KiB
        lens = np.array([10 << 20, (10 << 20) - 4099, 9 << 20])
    elif kind == "128 ragged, apart":
        lens = rng.integers(200000, 400000, 128)
    elif kind == "129 pages":
        lens = np.full(129, 8192)
    elif kind == "300 ragged":
        lens = rng.integers(0, 150000, 300)
    elif kind == "20000 short":                              # a table beyond one of the lists for recorded calls
        lens = np.concatenate([rng.integers(0, 800, 19000), rng.integers(16385, 17000, 1000)])
    elif kind == "5000 pages":                               # in windows, but for a few
        lens = np.full(5000, 8192)
        lens[1000:5000:500] = 8191
    elif kind == "4000 short":
        lens = rng.integers(0, 3000, 4000)
    else:                                                    # a table: one segment far beyond the others
        lens = np.concatenate([rng.integers(1, 9000, 200), [20 << 20], rng.integers(1, 9000, 200)])
    steps = (lens + 127) // 64 * 64
    at = np.cumsum(steps) - steps
    src = at + (5 if "apart" in kind else 0) + rng.integers(0, 2, len(lens)) * 16
    order = rng.permutation(len(lens))
    place = np.empty(len(lens), dtype=np.int64)
    place[order] = np.cumsum(steps[order]) - steps[order]
    dst = HALF + place
    assert (src + lens).max() <= HALF and (dst + lens).max() <= POOL
    return src.astype(np.uint64), dst.astype(np.uint64), lens.astype(np.uint64)


@pytest.mark.parametrize("form, kind", [("batch", "few, apart modulo 16"), ("batch", "128 ragged, apart"), ("batch", "129 pages"),
                                        ("batch", "300 ragged"), ("batch", "4000 short"), ("table", "300 ragged"), ("table", "one long"),
                                        ("table", "20000 short"), ("table", "5000 pages")])
def test_captured_and_replayed_between_plain_calls(gpu, oracle, form, kind):
    torch = pytest.importorskip("torch")
    assert torch.cuda.is_available()
    pool = gpu_util.DeviceBuffer(gpu, POOL)
    other = gpu_util.DeviceBuffer(gpu, POOL)
    table = gpu_util.DeviceBuffer(gpu, 24 * 20000)
    stream = torch.cuda.Stream()
    raw = stream.cuda_stream
    src, dst, lens = _batch(kind, 1)
    n = len(lens)
    plain = _batch("300 ragged", 2)
    plain = [native.u64_array(a) for a in (other.ptr + plain[0], other.ptr + plain[1], plain[2])]
    args = [native.u64_array(a) for a in (pool.ptr + src, pool.ptr + dst, lens)]
    table.upload(np.stack([pool.ptr + src, pool.ptr + dst, lens], axis=1).astype(np.uint64).view(np.uint8).reshape(-1))

    def call():
        if form == "table":
            return gpu.mf_xcopy_device_table(table.ptr, n, native.ROUTE_HBM, raw)
        return gpu.mf_xcopy_batch(*args, n, native.ROUTE_HBM, raw)

    try:
        assert call() == 0, native.last_error()
        torch.cuda.synchronize()
        graph = torch.cuda.CUDAGraph()
        with torch.cuda.graph(graph, stream=stream):
            ret = call()
        assert ret == 0, native.last_error()
        for replay in range(3):
            init = np.empty(POOL, dtype=np.uint8)
            oracle.orc_fill_random(init.ctypes.data, POOL, 700 + replay)
            pool.upload(init)
            for _ in range(9):                               # every slot of the thread's ring, on this stream and on the thread's own
                assert gpu.mf_xcopy_batch(*plain, 300, native.ROUTE_HBM, raw) == 0, native.last_error()
            for _ in range(9):
                assert gpu.mf_xcopy_batch(*plain, 300, native.ROUTE_HBM, None) == 0, native.last_error()
            assert gpu.mfrt_device_sync() == 0
            graph.replay()
            torch.cuda.synchronize()
            expect = init.copy()
            gpu_util.oracle_batch(oracle, init, expect, src, dst, lens)
            assert np.array_equal(pool.download(), expect), f"replay {replay} differs"
        del graph
    finally:
        pool.free()
        other.free()
        table.free()


@pytest.mark.parametrize("change", ["a second thread copies", "the table grows"])
def test_table_captured_after_a_plain_call_of_another_route(gpu, oracle, change):
    """The plain call before the capture goes out in one launch, the captured one in two, which need a list."""
    torch = pytest.importorskip("torch")
    pool = gpu_util.DeviceBuffer(gpu, POOL)
    src, dst, lens = _batch("20000 short", 3)
    table = gpu_util.DeviceBuffer(gpu, 24 * len(lens))
    stream = torch.cuda.Stream()
    raw = stream.cuda_stream
    warm = 1000
    n = warm if change == "a second thread copies" else len(lens)
    table.upload(np.stack([pool.ptr + src, pool.ptr + dst, lens], axis=1).astype(np.uint64).view(np.uint8).reshape(-1))
    ready, done = threading.Event(), threading.Event()

    def beside():
        assert gpu.mf_xcopy_thread_stream()
        ready.set()
        done.wait(60)

    second = threading.Thread(target=beside)
    graph = torch.cuda.CUDAGraph()
    try:
        gpu.hybm_uninit()                                    # a thread that has no lists from calls before
        assert gpu.hybm_init(0, 0) == 0, native.last_error()
        launches = gpu.mf_xcopy_launch_count()
        assert gpu.mf_xcopy_device_table(table.ptr, warm, native.ROUTE_HBM, raw) == 0, native.last_error()
        assert gpu.mf_xcopy_launch_count() - launches == 1
        torch.cuda.synchronize()
        if change == "a second thread copies":
            second.start()
            assert ready.wait(60)
        launches = gpu.mf_xcopy_launch_count()
        with torch.cuda.graph(graph, stream=stream):
            ret = gpu.mf_xcopy_device_table(table.ptr, n, native.ROUTE_HBM, raw)
        assert ret == 0, native.last_error()
        assert gpu.mf_xcopy_launch_count() - launches == (2 if n == warm else 4)
        for replay in range(3):
            init = np.empty(POOL, dtype=np.uint8)
            oracle.orc_fill_random(init.ctypes.data, POOL, 800 + replay)
            pool.upload(init)
            assert gpu.mf_xcopy_device_table(table.ptr, n, native.ROUTE_HBM, raw) == 0, native.last_error()
            torch.cuda.synchronize()
            pool.upload(init)
            graph.replay()
            torch.cuda.synchronize()
            expect = init.copy()
            gpu_util.oracle_batch(oracle, init, expect, src[:n], dst[:n], lens[:n])
            assert np.array_equal(pool.download(), expect), f"replay {replay} differs"
    finally:
        done.set()
        if second.is_alive():
            second.join()
        del graph
        pool.free()
        table.free()
