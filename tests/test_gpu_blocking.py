"""Short blocking copies, which report their own end: what they moved is where it belongs when the call returns."""

import ctypes
import threading
import time

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


HALF_MIB = 512 << 10


@pytest.mark.parametrize("way", ["load", "save"])
@pytest.mark.parametrize("sizes", [
    [HALF_MIB], [HALF_MIB + 1], [2 * HALF_MIB - 1], [3 * HALF_MIB + 4097, 0, 5],      # one round, its edge, the first of several
    [1000] * 700, [4000, 0, 60001] * 40,                                              # more segments in a round than a launch takes as arguments
    [HALF_MIB - 100, 300, 70000, HALF_MIB],                                           # a segment that would leave a sliver in a round
    [(37 << 20) + 13], [(9 << 20) + 1, 3, (31 << 20) + 70],                           # more rounds than there are slots
], ids=lambda s: f"{len(s)}x{s[0]}")
def test_staged_copies_of_pageable_memory(lib, pool, way, sizes):
    """Ordinary host memory through the staging ring: rounds that grow or shrink, cut inside segments, reuse their slots."""
    room = sum(sizes) + 64 * len(sizes) + 4096
    big = bm.create(2, 0, (room + (2 << 20)) // (2 << 20) * (2 << 20))
    try:
        dev = big.peer_rank_ptr(0)
        rng = np.random.default_rng(len(sizes))
        inside = np.cumsum([0] + [n + int(rng.integers(1, 64)) for n in sizes[:-1]])
        flat = rng.integers(0, 256, sum(sizes), dtype=np.uint8)
        outside = flat.ctypes.data + np.cumsum([0] + sizes[:-1])
        image = rng.integers(0, 256, room, dtype=np.uint8)
        assert lib.mfrt_memcpy(dev, image.ctypes.data, room) == 0
        source, target = (outside, dev + inside) if way == "load" else (dev + inside, outside)
        kind = bm.BmCopyType.H2G if way == "load" else bm.BmCopyType.G2H
        before = flat.copy()
        for _ in range(2):
            assert big.copy_data_batch(source.tolist(), target.tolist(), sizes, len(sizes), kind) == 0, native.last_error()
        at = 0
        for offset, n in zip(inside, sizes):
            if way == "load":
                image[offset:offset + n] = before[at:at + n]
            else:
                before[at:at + n] = image[offset:offset + n]
            at += n
        assert np.array_equal(flat, before)
        assert np.array_equal(_read(lib, dev, room), image)
    finally:
        big.destroy()


LEAST_ROUND = 576 << 10


@pytest.mark.parametrize("way", ["load", "save"])
@pytest.mark.parametrize("sizes", [
    [LEAST_ROUND], [LEAST_ROUND + 1], [3 * LEAST_ROUND // 2], [3 * LEAST_ROUND // 2 + 1],   # one round, as much as one takes, the first of two
    [5 * LEAST_ROUND // 2, 1], [130001] * 7, [LEAST_ROUND - 1, 1, 2 * LEAST_ROUND],         # the second's end, padded parts
    [1] * 9000, [(8 << 20) + 64, (4 << 20) - 1],                                            # padding alone, the longest rounds
], ids=lambda s: f"{len(s)}x{s[0]}")
def test_staged_copies_at_the_edges_of_rounds(lib, pool, way, sizes):
    test_staged_copies_of_pageable_memory(lib, pool, way, sizes)


@pytest.mark.parametrize("way", ["load", "save"])
@pytest.mark.parametrize("sizes", [
    [3 * LEAST_ROUND // 2], [3 * LEAST_ROUND // 2 + 1, 0], [16384] * 55, [16383] * 56,                # the least that streams, segments too short for it
    [65536 - 64] * 14, [65536, 65535, 65537, 1, 131072, 130900] * 3,                                # a chunk or nearly one a segment
    [65536 + 40960 - 128, 65536 + 40960, 65536 + 40961, 65536 + 41088, 196608 + 1, 3 * 65536 - 1] * 3, [65536 + 130] * 16,   # a tail that is shared out and one that is not
    [8 << 20], [(8 << 20) + 1], [(12 << 20) - 1], [12 << 20], [(33 << 20) + 1, 100000],             # back in rounds, past the caches, more chunks than slots
], ids=lambda s: f"{len(s)}x{s[0]}")
def test_copies_while_the_ring_is_filled_or_emptied(lib, pool, way, sizes):
    test_staged_copies_of_pageable_memory(lib, pool, way, sizes)


def test_chunks_that_the_host_never_fills(lib, pool):
    """The launch leaves when its wait is over, and what it would have written is as it was; what was filled is copied."""
    chunk, slots, room = 64 << 10, 4, 4096
    memory = pool.peer_rank_ptr(0)
    before = _read(lib, memory, 3 * chunk)
    host = lib.mfrt_alloc_host(slots * chunk + room)
    try:
        view = np.ctypeslib.as_array((ctypes.c_uint8 * (slots * chunk + room)).from_address(host))
        view[:] = 7
        words = view[slots * chunk:].view(np.uint64)
        words[:] = 0
        listed, host_words, gpu_words = slots * chunk, slots * chunk + 1024, slots * chunk + 2048
        for c in range(2):
            words[2 * c], words[2 * c + 1] = memory + c * chunk, 1000
        words[1024 // 8] = 11                                                         # chunk 0 is filled, chunk 1 is not
        err = lib.mfk_stream_chunks(0, ctypes.c_void_p(host), ctypes.c_void_p(host + listed), ctypes.c_void_p(host + host_words),
                                    ctypes.c_void_p(host + gpu_words), ctypes.c_uint64(10), 2, slots, 2, None)
        assert err == 0 and lib.mfrt_device_sync() == 0
        assert words[2048 // 8] == 11 and words[2048 // 8 + 8] == 0
        before[:1000] = 7
        assert np.array_equal(_read(lib, memory, 3 * chunk), before)
        assert lib.mfk_stream_chunks(0, ctypes.c_void_p(host), None, ctypes.c_void_p(host), ctypes.c_void_p(host), ctypes.c_uint64(0), 1, slots, 2, None) != 0
    finally:
        del view, words
        lib.mfrt_free_host(host)


@pytest.mark.parametrize("way, sizes", [
    ("load", [3 * LEAST_ROUND // 2 + 1]), ("load", [25600] * 37), ("load", [4 << 20]), ("load", [(4 << 20) + 1]), ("load", [50000, 300001, 70000] * 9),
    ("load", [(40 << 20) + 77]), ("save", [3 * LEAST_ROUND // 2 + 1]), ("save", [25600] * 37), ("save", [(4 << 20) + 1]), ("save", [8 << 20]),
    ("save", [40000] * 100),
], ids=lambda v: v if isinstance(v, str) else f"{len(v)}x{v[0]}")
def test_copies_are_made_beside_the_cpu(lib, pool, way, sizes):
    """In launches of 64 chunks and no others: a copy whose launches cannot be made, or leave, has the same bytes and more launches."""
    room = sum(sizes) + 256 * len(sizes)
    big = bm.create(2, 0, (room + (2 << 20)) // (2 << 20) * (2 << 20))
    try:
        inside = big.peer_rank_ptr(0) + np.cumsum([0] + [(n + 255) // 128 * 128 for n in sizes[:-1]])
        flat = np.random.default_rng(3).integers(0, 256, sum(sizes), dtype=np.uint8)
        outside = flat.ctypes.data + np.cumsum([0] + sizes[:-1])
        expect = flat.copy()
        load, save = bm.BmCopyType.H2G, bm.BmCopyType.G2H
        assert big.copy_data_batch(outside.tolist(), inside.tolist(), sizes, len(sizes), load) == 0, native.last_error()
        chunks = sum((n + 65535) // 65536 for n in sizes)
        for _ in range(3):
            if way == "save":
                flat[:] = 0
            launches = lib.mf_xcopy_launch_count()
            source, target = (outside, inside) if way == "load" else (inside, outside)
            assert big.copy_data_batch(source.tolist(), target.tolist(), sizes, len(sizes), load if way == "load" else save) == 0, native.last_error()
            assert lib.mf_xcopy_launch_count() - launches == (chunks + 63) // 64
        if way == "load":
            flat[:] = 0
            assert big.copy_data_batch(inside.tolist(), outside.tolist(), sizes, len(sizes), save) == 0, native.last_error()
        assert np.array_equal(flat, expect)
    finally:
        big.destroy()


@pytest.mark.parametrize("way, nbytes", [("load", 1 << 20), ("load", 40 << 20), ("save", 1 << 20), ("save", 8 << 20)])
def test_copies_behind_other_work(lib, pool, way, nbytes):
    """Several milliseconds of it on the same stream: the caller has gone over from polling to waiting when the launch begins."""
    other = 128 << 20
    big = bm.create(2, 0, 2 * other + (64 << 20))
    try:
        dev = big.peer_rank_ptr(0)
        at = dev + 2 * other + 77
        flat = np.random.default_rng(nbytes).integers(0, 256, nbytes, dtype=np.uint8)
        expect = flat.copy()
        load, save = bm.BmCopyType.H2G, bm.BmCopyType.G2H
        if way == "save":
            assert big.copy_data(flat.ctypes.data, at, nbytes, load) == 0, native.last_error()
            flat[:] = 0
        for _ in range(100):
            assert big.copy_data(dev, dev + other, other, bm.BmCopyType.G2G, native.ASYNC_COPY_FLAG) == 0, native.last_error()
        launches = lib.mf_xcopy_launch_count()
        source, target = (flat.ctypes.data, at) if way == "load" else (at, flat.ctypes.data)
        assert big.copy_data(source, target, nbytes, load if way == "load" else save) == 0, native.last_error()
        assert lib.mf_xcopy_launch_count() - launches == (nbytes // 65536 + 64) // 64          # one chunk more than whole ones: they begin off a line
        assert np.array_equal(flat if way == "save" else _read(lib, at, nbytes), expect)
    finally:
        assert lib.mfrt_device_sync() == 0
        big.destroy()


def test_threads_that_stream_at_once(lib, pool):
    """One of them has the helpers, the others copy alone."""
    count, room = 4, 12 << 20
    big = bm.create(2, 0, count * room + (2 << 20))
    errors = []

    def run(k):
        try:
            rng = np.random.default_rng(k)
            at = big.peer_rank_ptr(0) + k * room
            for nbytes in (1 << 20, (9 << 20) + 5, 3000001, 8 << 20):
                flat = rng.integers(0, 256, nbytes, dtype=np.uint8)
                back = np.zeros_like(flat)
                for _ in range(5):
                    assert big.copy_data(flat.ctypes.data, at + k, nbytes, bm.BmCopyType.H2G) == 0, native.last_error()
                    assert big.copy_data(at + k, back.ctypes.data, nbytes, bm.BmCopyType.G2H) == 0, native.last_error()
                    assert np.array_equal(flat, back)
                    back[:] = 0
        except BaseException as e:   # noqa: BLE001 - handed to the test's own thread
            errors.append(e)

    threads = [threading.Thread(target=run, args=(k,)) for k in range(count)]
    try:
        for t in threads:
            t.start()
        for t in threads:
            t.join()
        assert not errors, errors[0]
    finally:
        big.destroy()


class _Ring:
    """The area that a launch of chunks and the CPU share, of `slots` slots and `count` chunks at `addresses` of `lengths` bytes."""

    def __init__(self, lib, slots, addresses, lengths, base):
        self.lib, self.slots, self.count, self.base = lib, slots, len(addresses), base
        self.listed = slots << 16
        self.words_at = [self.listed + 16 * self.count + 64, 0]
        self.words_at[0] = self.words_at[0] // 64 * 64
        self.words_at[1] = self.words_at[0] + 64 * slots
        size = self.words_at[1] + 64 * slots
        self.host = lib.mfrt_alloc_host(size)
        self.bytes = np.ctypeslib.as_array((ctypes.c_uint8 * size).from_address(self.host))
        self.bytes[:] = 0
        pairs = self.bytes[self.listed:self.listed + 16 * self.count].view(np.uint64)
        pairs[0::2], pairs[1::2] = addresses, lengths
        self.filled, self.done = (self.bytes[at:at + 64 * slots].view(np.uint64)[::8] for at in self.words_at)
        self.places = [(c % slots << 16) + addresses[c] % 128 for c in range(self.count)]

    def launch(self, beside, to_host, first, count, limit=1000):
        slot = first % self.slots
        call = self.lib.mfk_stream_chunks_beside if beside else self.lib.mfk_stream_chunks
        return call(int(to_host), ctypes.c_void_p(self.host + (slot << 16)), ctypes.c_void_p(self.host + self.listed + 16 * first),
                    ctypes.c_void_p(self.host + self.words_at[0] + 64 * slot), ctypes.c_void_p(self.host + self.words_at[1] + 64 * slot),
                    ctypes.c_uint64(self.base + first), count, self.slots - slot, limit, ctypes.c_void_p(self.lib.mf_xcopy_thread_stream()))

    def wait(self, c):
        end = time.monotonic() + 5
        while int(self.done[c % self.slots]) != self.base + c + 1:
            assert time.monotonic() < end

    def close(self):
        assert self.lib.mfrt_device_sync() == 0
        del self.bytes, self.filled, self.done
        self.lib.mfrt_free_host(self.host)


CHUNK_LENGTHS = [1, 15, 16, 17, 127, 128, 4096, 8191, 40000, 65409, 65408, 30001]


@pytest.mark.parametrize("base", [0, (1 << 40) - 3])
def test_chunks_to_the_host(lib, pool, base):
    """Two launches, the second beside the first: every byte of a chunk lies in its slot as far behind a line as in HBM, and no other is written."""
    memory = pool.peer_rank_ptr(0)
    slots = 2 * len(CHUNK_LENGTHS)
    lengths = CHUNK_LENGTHS + CHUNK_LENGTHS[::-1]
    starts = [(c << 17) + (127 if n == 65409 else c * 37 % 128) for c, n in enumerate(lengths)]
    image = np.random.default_rng(5).integers(1, 256, slots << 17, dtype=np.uint8)
    assert lib.mfrt_memcpy(memory, image.ctypes.data, image.size) == 0
    ring = _Ring(lib, slots, [memory + a for a in starts], lengths, base)
    try:
        half = len(CHUNK_LENGTHS)
        assert ring.launch(False, True, 0, slots + 1) != 0                 # more chunks than slots: nobody would empty them
        assert ring.launch(False, True, 0, half) == 0 and ring.launch(True, True, half, half) == 0
        assert lib.mfrt_device_sync() == 0
        expect = np.zeros(slots << 16, dtype=np.uint8)
        for c, (a, n) in enumerate(zip(starts, lengths)):
            expect[ring.places[c]:ring.places[c] + n] = image[a:a + n]
            assert int(ring.done[c]) == base + c + 1
        assert np.array_equal(ring.bytes[:slots << 16], expect)
    finally:
        ring.close()


def test_chunks_from_the_host_round_the_ring(lib, pool):
    """Five times as many chunks as slots, in launches beside one another, while the CPU fills what has been emptied."""
    memory = pool.peer_rank_ptr(0)
    slots, times = len(CHUNK_LENGTHS), 5
    lengths = CHUNK_LENGTHS * times
    starts = [(c << 16) + (127 if n == 65409 else c * 53 % 128) for c, n in enumerate(lengths)]
    before = _read(lib, memory, len(lengths) << 16)
    data = np.random.default_rng(6).integers(0, 256, before.size, dtype=np.uint8)
    ring = _Ring(lib, slots, [memory + a for a in starts], lengths, 77)
    try:
        for c, (a, n) in enumerate(zip(starts, lengths)):
            if c % slots == 0:
                assert ring.launch(c != 0, False, c, slots) == 0
            if c >= slots:
                ring.wait(c - slots)
            ring.bytes[ring.places[c]:ring.places[c] + n] = data[a:a + n]
            before[a:a + n] = data[a:a + n]
            ring.filled[c % slots] = 77 + c + 1
        for c in range(len(lengths) - slots, len(lengths)):
            ring.wait(c)
        assert lib.mfrt_device_sync() == 0
        assert np.array_equal(_read(lib, memory, before.size), before)
    finally:
        ring.close()


@pytest.mark.parametrize("count, most, launches", [(513, 131072, 1), (1400, 65536, 2), (1601, 131072, 3)])
def test_long_batch_in_launches_that_planning_overlaps(lib, pool, count, most, launches):
    """Every byte is there when the call returns, whichever of its launches moved it."""
    rng = np.random.default_rng(count)
    lens = rng.integers(most * 15 // 16, most, count) // 16 * 16 - rng.integers(0, 2, count)
    steps = (lens + 127) // 128 * 128
    order = rng.permutation(count)
    at = np.cumsum(steps) - steps
    place = np.empty(count, dtype=np.int64)
    place[order] = np.cumsum(steps[order]) - steps[order]
    size = int(steps.sum())
    room = (size + (2 << 20) - 1) // (2 << 20) * (2 << 20)
    other = bm.create(2, 0, 2 * room)
    try:
        source = other.peer_rank_ptr(0, bm.BmMemType.DEVICE)
        data = rng.integers(0, 256, size, dtype=np.uint8)
        assert lib.mfrt_memcpy(source, data.ctypes.data, size) == 0
        assert lib.mfrt_memset(source + room, 0, room) == 0
        before = lib.mf_xcopy_launch_count()
        assert other.copy_data_batch((source + at).tolist(), (source + room + place).tolist(), lens.tolist(), count,
                                     bm.BmCopyType.G2G) == 0, native.last_error()
        assert lib.mf_xcopy_launch_count() - before == launches
        got = _read(lib, source + room, size)
    finally:
        other.destroy()
    expect = np.zeros(size, dtype=np.uint8)
    for s, d, n in zip(at, place, lens):
        expect[d:d + n] = data[s:s + n]
    assert np.array_equal(got, expect)


@pytest.mark.parametrize("threads", [1, 3])
def test_copies_whose_workgroups_count_in_two_steps(lib, pool, threads):
    """65 workgroups and more, in turn with fewer, and batches, each thread with counters of its own: 1 MiB and 16 bytes, the last
    sizes that report their own end and the first beyond."""
    mib = 1 << 20
    room = 9 * mib
    handle = bm.create(2, 0, 2 * room * threads)
    dev = handle.peer_rank_ptr(0, bm.BmMemType.DEVICE)
    failures = []

    def work(t):
        try:
            rng = np.random.default_rng(t)
            source, target = dev + 2 * room * t, dev + 2 * room * t + room
            data = rng.integers(0, 256, room, dtype=np.uint8)
            assert lib.mfrt_memcpy(source, data.ctypes.data, room) == 0
            for size in [mib, mib + 16, 4 * mib, 33, 8 * mib, 8 * mib + 1, 2 * mib - 5, mib + 1] * 2:
                s, d = int(rng.integers(0, 200)), int(rng.integers(0, 200))
                assert lib.mfrt_memset(target, 0xA5, size + 512) == 0
                assert handle.copy_data(source + s, target + d, size, bm.BmCopyType.G2G) == 0, native.last_error()
                got = _read(lib, target, size + 512)
                assert np.array_equal(got[d:d + size], data[s:s + size]) and np.all(got[d + size:] == 0xA5), (size, s, d)
            for count, each in [(128, 32768), (100, 41000), (2, 2 * mib), (2, 2 * mib + 8), (64, 16385), (129, 32513), (129, 32514), (2048, 2000), (2049, 2000),
                                (300, 4096), (700, 4099)]:
                assert lib.mfrt_memset(target, 0xA5, room) == 0
                at = rng.permutation(count) * (each + 7)
                to = rng.permutation(count) * (each + 9)
                assert handle.copy_data_batch(source + at, target + to, np.full(count, each), count, bm.BmCopyType.G2G) == 0, native.last_error()
                want = np.full(room, 0xA5, dtype=np.uint8)
                for a, b in zip(at, to):
                    want[b:b + each] = data[a:a + each]
                assert np.array_equal(_read(lib, target, room), want), (count, each)
        except Exception as e:  # noqa: BLE001 - reported by the test's own thread
            failures.append(repr(e))

    workers = [threading.Thread(target=work, args=(t,)) for t in range(threads)]
    for w in workers:
        w.start()
    for w in workers:
        w.join()
    handle.destroy()
    assert not failures, failures
