"""Batches of more than 128 segments between HBM addresses: every way a source and a destination can differ modulo 16, lengths at
the edges of the pieces they are cut into, and sizes that take each of the launch's shapes, with stores held and not."""
import time

import numpy as np
import pytest

from memfabric_hybrid_amd import native
from tests import gpu_util
from tests.test_gpu_xcopy import _random_bytes

pytestmark = pytest.mark.gpu

EDGES = [1, 15, 16, 17, 31, 33, 4079, 4080, 4096, 4097, 4111, 8192, 8193, 16383, 16384, 16385, 16399, 0, 0, 65537]


@pytest.fixture(scope="module")
def gpu(lib):
    assert lib.hybm_init(0, 0) == 0, native.last_error()
    yield lib
    lib.hybm_uninit()


def _lengths(kind, rng):
    if kind == "every shift":                                    # 256 pairs of source and destination bytes, one wave each
        return np.concatenate([rng.integers(1, 4000, 256), np.tile(EDGES, 16)])
    if kind == "held 4 KiB":                                     # 6 MB and more: stores held
        return np.concatenate([rng.integers(1, 70000, 200), EDGES])
    if kind == "held 16 KiB":                                    # 24 to 64 MiB of long segments
        return np.concatenate([rng.integers(1, 200000, 400), EDGES])
    if kind == "one wave":                                       # beyond 24 MiB the usual segment decides
        return np.concatenate([rng.integers(1, 9000, 7000), EDGES])
    if kind == "held 8 KiB":                                     # no segment longer, 4096 pieces at the most
        return np.concatenate([rng.integers(7000, 8065, 2900), [1, 0, 8064, 8065, 17, 4096]])
    if kind == "held, nearly full":
        return np.concatenate([rng.integers(111000, 131000, 760), EDGES])
    if kind == "windows":                                        # nearly full pieces, more than are held; two rounds and a fraction of 4096
        return np.concatenate([rng.integers(111000, 131000, 1100), EDGES])
    if kind == "windows, three rounds":
        return np.concatenate([np.full(8193, 16384), [16384 + 15, 16383, 1, 0]])
    if kind == "held, all that are resident":                    # 7168 pieces of 16 KiB at the most hold their stores
        return np.concatenate([np.full(7168 - len(EDGES), 16256), np.minimum(EDGES, 16256)])
    if kind == "one too many to hold":
        return np.concatenate([np.full(7169 - len(EDGES), 16256), np.minimum(np.maximum(EDGES, 1), 16256)])
    if kind == "more than are held":
        return np.concatenate([rng.integers(1, 90000, 2700), EDGES])
    if kind == "three times what is held":
        return np.concatenate([rng.integers(50000, 110000, 3000), EDGES])
    if kind == "three times what is held, part-filled":
        return np.concatenate([rng.integers(33000, 40000, 5000), EDGES])
    if kind == "four times what is held":
        return np.concatenate([rng.integers(50000, 110000, 4400), EDGES])
    if kind == "two waves":
        return np.concatenate([rng.integers(1, 20000, 3000), EDGES])
    return np.concatenate([rng.integers(1, 90000, 2000), EDGES])   # "four waves"


@pytest.mark.parametrize("kind", ["every shift", "held 4 KiB", "held 16 KiB", "held 8 KiB", "one wave", "two waves", "four waves", "windows",
                                  "held, nearly full", "windows, three rounds", "held, all that are resident", "one too many to hold", "more than are held",
                                  "three times what is held", "three times what is held, part-filled", "four times what is held"])
@pytest.mark.parametrize("odd", [True, False])
def test_batch_in_pieces(gpu, oracle, kind, odd):
    rng = np.random.default_rng(len(kind) + odd)
    lens = _lengths(kind, rng).astype(np.uint64)
    n = len(lens)
    steps = (lens + np.uint64(159)) // np.uint64(128) * np.uint64(128)
    at = np.concatenate(([0], np.cumsum(steps)[:-1])).astype(np.uint64)
    size = int(steps.sum()) + 128
    pairs = np.arange(n, dtype=np.uint64)
    src = at + (pairs % np.uint64(16) if odd else np.uint64(0))
    dst = at + (pairs // np.uint64(16) % np.uint64(16) if odd else np.uint64(0))
    order = rng.permutation(n)
    src, dst, lens = src[order], dst[order], lens[order]
    source = _random_bytes(oracle, size, 3)
    before = _random_bytes(oracle, size, 4)
    a, b = gpu_util.DeviceBuffer(gpu, size), gpu_util.DeviceBuffer(gpu, size)
    try:
        a.upload(source)
        b.upload(before)
        launches = gpu.mf_xcopy_launch_count()
        gpu_util.xcopy(gpu, a.ptr + src, b.ptr + dst, lens, native.ROUTE_HBM)
        expect = {"more than are held": 2}       # nearly full pieces on lines go in windows; short segments at odd bytes in one launch that holds nothing
        expect.update({"windows": 2, "three times what is held": 3, "four times what is held": 4} if odd else {"three times what is held, part-filled": 3})
        assert gpu.mf_xcopy_launch_count() - launches == expect.get(kind, 1)
        got = b.download()
    finally:
        a.free()
        b.free()
    gpu_util.oracle_batch(oracle, source, before, src, dst, lens)
    assert np.array_equal(got, before)


@pytest.mark.parametrize("count,size", [(1700, 65536), (1000, 131072), (1030, 110720), (16384, 16384), (7169, 16384), (8193, 32768)])
@pytest.mark.parametrize("where", ["in order", "read in order", "scattered"])
def test_lists_of_blocks_in_windows(gpu, count, size, where):
    """Blocks of one length, written one behind the other, read so, or neither, at the rates that each of them is given."""
    torch = pytest.importorskip("torch")
    rng = np.random.default_rng(count)
    at = (np.arange(count) if where == "read in order" else rng.permutation(2 * count)[:count]).astype(np.int64)
    place = (np.arange(count) if where == "in order" else rng.permutation(count)).astype(np.int64)
    source = torch.randint(-2**63, 2**63 - 1, (2 * count * size // 8,), dtype=torch.int64, device="cuda").view(torch.uint8)
    target = torch.zeros(count * size, dtype=torch.uint8, device="cuda")
    torch.cuda.synchronize()
    lens = np.full(count, size, dtype=np.uint64)
    gpu_util.xcopy(gpu, (source.data_ptr() + at * size).astype(np.uint64), (target.data_ptr() + place * size).astype(np.uint64), lens, native.ROUTE_HBM)
    assert torch.equal(target.view(count, size)[torch.from_numpy(place).cuda()], source.view(2 * count, size)[torch.from_numpy(at).cuda()])


@pytest.mark.parametrize("form", ["4 KiB", "8 KiB", "held 16 KiB", "four waves"])
@pytest.mark.parametrize("shift", [0, 5, 16])
def test_pieces_that_begin_inside_a_line(gpu, form, shift):
    """Destinations at every unit of a cache line and beside it, and lengths that end a piece at its last unit, before and behind it.
    shift: what the source is off the destination's place in its line."""
    torch = pytest.importorskip("torch")
    rng = np.random.default_rng(7)
    offsets = np.array([o + b for o in range(0, 128, 16) for b in (0, 1, 8, 15)], dtype=np.int64)
    most = {"4 KiB": 4096, "8 KiB": 8192, "held 16 KiB": 16384, "four waves": 16384}[form]
    ends = [most - 1, most, most + 1, 2 * most + 33]
    short = [] if form in ("8 KiB", "four waves") else [1, 16, 100, 128, 144]
    lens = np.concatenate([np.concatenate((most - offsets + e, np.full(len(offsets), most + e))) for e in (-16, -1, 0, 1)] +
                          [np.full(2 * len(offsets), e) for e in ends + short]).astype(np.int64)
    at = np.tile(offsets, len(lens) // len(offsets))
    times = {"4 KiB": 1, "8 KiB": 12, "held 16 KiB": 3, "four waves": 20}[form]
    lens, at = np.tile(lens, times), np.tile(at, times)
    order = rng.permutation(len(lens))
    lens, at = lens[order], at[order]
    steps = (at + shift + lens + 383) // 128 * 128
    begin = np.cumsum(steps) - steps
    size = int(steps.sum())
    source = torch.randint(0, 256, (size,), dtype=torch.uint8, device="cuda")
    target = torch.randint(0, 256, (size,), dtype=torch.uint8, device="cuda")
    expect = target.clone()
    for b, o, n in zip((begin + at).tolist(), (begin + at + shift).tolist(), lens.tolist()):
        expect[b:b + n] = source[o:o + n]
    torch.cuda.synchronize()
    gpu_util.xcopy(gpu, (source.data_ptr() + begin + at + shift).astype(np.uint64), (target.data_ptr() + begin + at).astype(np.uint64),
                   lens.astype(np.uint64), native.ROUTE_HBM)
    assert torch.equal(target, expect)


@pytest.mark.parametrize("count,least,most", [(8000, 30000, 45000), (6700, 1, 131073), (4800, 93000, 98305)])
def test_ragged_lists_at_odd_addresses_in_windows(gpu, count, least, most):
    """Three held launches' worth of short segments, more than four of others: one launch each, pieces of every fill at every byte."""
    torch = pytest.importorskip("torch")
    rng = np.random.default_rng(count)
    lens = rng.integers(least, most, count)
    steps = lens + rng.integers(0, 300, count)
    begin = np.cumsum(steps) - steps
    order = rng.permutation(count)
    size = int(steps.sum()) + 512
    source = torch.randint(-2**63, 2**63 - 1, ((size + 7) // 8,), dtype=torch.int64, device="cuda").view(torch.uint8)
    target = torch.zeros_like(source)
    other = rng.permutation(count)                       # sources in another order, so neither side has one
    src = np.empty(count, dtype=np.int64)
    src[other] = np.cumsum(steps[other]) - steps[other]
    expect = target.clone()
    for b, o, n in zip(begin.tolist(), src.tolist(), lens.tolist()):
        expect[b:b + n] = source[o:o + n]
    torch.cuda.synchronize()
    launches = gpu.mf_xcopy_launch_count()
    gpu_util.xcopy(gpu, (source.data_ptr() + src[order]).astype(np.uint64), (target.data_ptr() + begin[order]).astype(np.uint64),
                   lens[order].astype(np.uint64), native.ROUTE_HBM)
    assert gpu.mf_xcopy_launch_count() - launches == 1
    assert torch.equal(target, expect)


# Batches whose chunks are cut on the destinations' lines and go in windows: one segment just above what is held, at and beyond 128 MiB; chunks that
# are not whole, segments shorter than one, than a unit, than a line.
@pytest.mark.parametrize("lens", [[(112 << 20) + 1], [(112 << 20) - 127], [(128 << 20) + 77], [300000001], [(64 << 20) + 1 - 16500, 16500],
                                  [700001] * 127 + [5], [1 << 20] * 66 + [16384, 16383, 16385, 1, 15, 16, 17, 127, 128, 129, 0, 0, 33000] * 4], ids=str)
@pytest.mark.parametrize("shift", [(0, 0), (0, 16), (64, 48), (3, 19), (0, 1), (1, 0), (4, 0), (127, 120), (5, 11), "each another"], ids=str)
def test_batches_cut_on_lines_in_windows(gpu, lens, shift):
    torch = pytest.importorskip("torch")
    rng = np.random.default_rng(len(lens))
    lens = np.array(lens, dtype=np.int64)
    steps = (lens + 511) // 256 * 256
    order = rng.permutation(len(lens))
    at = np.cumsum(steps) - steps
    place = np.empty_like(at)
    place[order] = np.cumsum(steps[order]) - steps[order]
    if shift == "each another":
        at, place = at + rng.integers(0, 128, len(lens)), place + rng.integers(0, 128, len(lens))
    else:
        at, place = at + shift[0], place + shift[1]
    room = int(steps.sum()) + 256
    source = torch.randint(-2**63, 2**63 - 1, (room // 8,), dtype=torch.int64, device="cuda").view(torch.uint8)
    before = torch.randint(-2**63, 2**63 - 1, (room // 8,), dtype=torch.int64, device="cuda").view(torch.uint8)
    target, expect = before.clone(), before.clone()
    for s, d, l in zip(at.tolist(), place.tolist(), lens.tolist()):
        expect[d:d + l] = source[s:s + l]
    torch.cuda.synchronize()
    launches = gpu.mf_xcopy_launch_count()
    gpu_util.xcopy(gpu, (source.data_ptr() + at).astype(np.uint64), (target.data_ptr() + place).astype(np.uint64), lens.astype(np.uint64), native.ROUTE_HBM)
    assert gpu.mf_xcopy_launch_count() - launches == 1
    assert torch.equal(target, expect)


# Windows where a round of the waves ends: one of 6144 chunks of 16 KiB, two, and a chunk, a unit or a byte more or less.
@pytest.mark.parametrize("n", [2 * 6144 * 16384 + more for more in (-16385, -1, 0, 1, 16, 16384, 16389)] + [6144 * 16384 * 3 // 2 + 5])
@pytest.mark.parametrize("shift", [(0, 0), (16, 48), (3, 9)], ids=str)
def test_windows_where_a_round_ends(gpu, n, shift):
    torch = pytest.importorskip("torch")
    source = torch.randint(-2**63, 2**63 - 1, (n // 8 + 32,), dtype=torch.int64, device="cuda").view(torch.uint8)
    target = torch.zeros_like(source)
    torch.cuda.synchronize()
    gpu_util.xcopy(gpu, np.array([source.data_ptr() + shift[0]], dtype=np.uint64), np.array([target.data_ptr() + shift[1]], dtype=np.uint64),
                   np.array([n], dtype=np.uint64), native.ROUTE_HBM)
    assert torch.equal(target[shift[1]:shift[1] + n], source[shift[0]:shift[0] + n])
    assert not target[:shift[1]].any() and not target[shift[1] + n:].any()


@pytest.mark.parametrize("each", [512, 40000])
@pytest.mark.parametrize("order", ["own", "a caller's", "own and a caller's", "own, blocking between", "own, a long copy in front",
                                   "a caller's, a long copy in front"])
def test_slots_whose_followers_say_that_they_are_free(gpu, order, each):
    """More batches in flight than there are slots, none of them waited for: what each was told must stay in its slot until it has run."""
    rng = np.random.default_rng(each)
    batches, n = 40, 260
    room = n * (each + 64)
    a, b = gpu_util.DeviceBuffer(gpu, room), gpu_util.DeviceBuffer(gpu, batches * room)
    long_from, long_to = gpu_util.DeviceBuffer(gpu, 256 << 20), gpu_util.DeviceBuffer(gpu, 256 << 20)
    other = gpu.mfrt_stream_create()
    try:
        data = rng.integers(0, 256, room, dtype=np.uint8)
        a.upload(data)
        b.fill(0xA5)
        want = np.full(batches * room, 0xA5, dtype=np.uint8)
        if order.endswith("a long copy in front"):
            for _ in range(20):
                gpu_util.xcopy(gpu, [long_from.ptr], [long_to.ptr], [256 << 20], native.ROUTE_HBM, other if order[0] == "a" else None, sync=False)
        for k in range(batches):
            lens = rng.integers(1, each, n).astype(np.uint64)
            src = rng.integers(0, room - each, n).astype(np.uint64)
            dst = rng.permutation(n).astype(np.uint64) * np.uint64(each + 64) + np.uint64(k * room)
            for s, d, l in zip(src.tolist(), dst.tolist(), lens.tolist()):
                want[d:d + l] = data[s:s + l]
            stream = other if order.startswith("a caller's") or (order == "own and a caller's" and k % 5 > 2) else None
            gpu_util.xcopy(gpu, a.ptr + src, b.ptr + dst, lens, native.ROUTE_HBM, stream, sync=False)
            if order == "own, blocking between" and k % 9 == 4:
                assert gpu.mfrt_stream_sync(gpu.mf_xcopy_thread_stream()) == 0
        assert gpu.mfrt_device_sync() == 0
        assert np.array_equal(b.download(), want)
    finally:
        gpu.mfrt_stream_destroy(other)
        for buffer in (a, b, long_from, long_to):
            buffer.free()


@pytest.mark.parametrize("order", ["a caller's", "own", "own, followed by a caller's"])
def test_slots_whose_launches_do_not_start_for_a_while(gpu, order):
    """A third of a second of copies to the host in front: a call that needs a slot again looks for its word longer than it is polled for,
    and where no launch follows on the own stream it waits for an event."""
    rng = np.random.default_rng(len(order))
    batches, n, each, long = 12, 260, 20000, 256 << 20
    room = n * (each + 64)
    a, b = gpu_util.DeviceBuffer(gpu, room), gpu_util.DeviceBuffer(gpu, batches * room)
    long_from, long_to = gpu_util.DeviceBuffer(gpu, long), gpu_util.PinnedBuffer(gpu, long)
    other = gpu.mfrt_stream_create()
    try:
        data = rng.integers(0, 256, room, dtype=np.uint8)
        a.upload(data)
        b.fill(0xA5)
        want = np.full(batches * room, 0xA5, dtype=np.uint8)
        plans = []
        for k in range(batches):
            lens = rng.integers(1, each, n).astype(np.uint64)
            src = rng.integers(0, room - each, n).astype(np.uint64)
            dst = rng.permutation(n).astype(np.uint64) * np.uint64(each + 64) + np.uint64(k * room)
            for s, d, l in zip(src.tolist(), dst.tolist(), lens.tolist()):
                want[d:d + l] = data[s:s + l]
            plans.append([native.u64_array(v) for v in (a.ptr + src, b.ptr + dst, lens)])
        assert gpu.mfrt_device_sync() == 0
        first = other if order == "a caller's" else None
        for _ in range(75):                                  # 4.7 ms each
            gpu_util.xcopy(gpu, [long_from.ptr], [long_to.ptr], [long], native.ROUTE_TO_HOST, first, sync=False)
        began = time.monotonic()
        for k, plan in enumerate(plans):
            stream = other if order == "a caller's" or (k > 0 and order != "own") else None
            assert gpu.mf_xcopy_batch(*plan, n, native.ROUTE_HBM, stream) == 0, native.last_error()
        assert time.monotonic() - began > 0.25
        assert gpu.mfrt_device_sync() == 0
        assert np.array_equal(b.download(), want)
    finally:
        gpu.mfrt_device_sync()
        gpu.mfrt_stream_destroy(other)
        for buffer in (a, b, long_from, long_to):
            buffer.free()


# Lists in windows of pieces that are not full, and as many as a round of 6144 waves has, a group of 64 more or less.
@pytest.mark.parametrize("count, size", [(3072, 32896), (7232, 16400), (12288, 16384), (12287, 16384), (12352, 16384), (8000, 24576), (8000, 24001), (4000, 40000),
                                         (3700, 49153), (2400, 50048), (2200, 65535), (1500, 100352)])
@pytest.mark.parametrize("where", ["gathered", "scattered"])
def test_lists_of_part_filled_pieces_in_windows(gpu, count, size, where):
    torch = pytest.importorskip("torch")
    step = (size + 127) // 128 * 128
    rng = np.random.default_rng(count)
    at = rng.permutation(count).astype(np.int64) * step
    place = np.arange(count, dtype=np.int64) * step
    if where == "scattered":
        at, place = place, at
    source = torch.randint(-2**63, 2**63 - 1, (count * step // 8,), dtype=torch.int64, device="cuda").view(torch.uint8)
    target = torch.full_like(source, 0x5A)
    torch.cuda.synchronize()
    for _ in range(2):
        gpu_util.xcopy(gpu, (source.data_ptr() + at).astype(np.uint64), (target.data_ptr() + place).astype(np.uint64),
                       np.full(count, size, dtype=np.uint64), native.ROUTE_HBM)
    got = target.view(count, step)[torch.from_numpy(place // step).cuda()]
    assert torch.equal(got[:, :size], source.view(count, step)[torch.from_numpy(at // step).cuda()][:, :size])
    assert bool((got[:, size:] == 0x5A).all())
