"""GPU parity of the local MoE dispatch / combine against the CPU specification in
oracle/mf_oracle.c.  Dispatch is integer/byte work: bit-exact.  Combine is floating point: the
stated tolerance is 1e-2 relative (bf16); because both sides use the same fp32 FMA chain and one
final rounding, the test additionally demands bit-equality, which is the stronger statement."""

import ctypes

import numpy as np
import pytest

from memfabric_hybrid_amd import native, workloads
from tests import gpu_util
from tests.oracle_lib import np_ptr

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def gpu(lib):
    assert lib.hybm_init(0, 0) == 0, native.last_error()
    yield lib
    lib.hybm_uninit()


def _dev(gpu, array):
    a = np.ascontiguousarray(array)
    buf = gpu_util.DeviceBuffer(gpu, max(a.nbytes, 16))
    if a.nbytes:
        buf.upload(a.view(np.uint8).reshape(-1))
    return buf


def _fetch(buf, dtype, shape):
    n = int(np.prod(shape)) * np.dtype(dtype).itemsize
    return buf.download(0, n).view(dtype).reshape(shape)


def _oracle_dispatch(oracle, x, topk, E):
    T, H = x.shape
    K = topk.shape[1]
    out = np.zeros((T * K, H), dtype=np.uint16)
    counts = np.zeros(E, dtype=np.int32)
    offsets = np.zeros(E, dtype=np.int32)
    row_of = np.zeros(T * K, dtype=np.int32)
    src_of = np.zeros(T * K, dtype=np.int32)
    ret = oracle.orc_moe_dispatch(np_ptr(x), np_ptr(topk), T, H, K, E, np_ptr(out), np_ptr(counts), np_ptr(offsets),
                                  np_ptr(row_of), np_ptr(src_of))
    assert ret == 0
    return out, counts, offsets, row_of, src_of


def _gpu_dispatch(gpu, x, topk, E, with_rows=True):
    T, H = x.shape
    K = topk.shape[1]
    ws_bytes = gpu.mf_moe_workspace_bytes(T, K, E)
    bufs = {
        "x": _dev(gpu, x), "topk": _dev(gpu, topk), "out": gpu_util.DeviceBuffer(gpu, max(T * K * H * 2, 16)),
        "counts": gpu_util.DeviceBuffer(gpu, E * 4), "offsets": gpu_util.DeviceBuffer(gpu, E * 4),
        "row_of": gpu_util.DeviceBuffer(gpu, T * K * 4), "src_of": gpu_util.DeviceBuffer(gpu, T * K * 4),
        "ws": gpu_util.DeviceBuffer(gpu, ws_bytes),
    }
    bufs["ws"].fill(0xFF)  # the workspace needs no initialisation
    bufs["src_of"].fill(0xFF)
    ret = gpu.mf_moe_dispatch(bufs["x"].ptr if with_rows else None, bufs["topk"].ptr, T, H, K, E,
                              bufs["out"].ptr if with_rows else None, bufs["counts"].ptr, bufs["offsets"].ptr,
                              bufs["row_of"].ptr, bufs["src_of"].ptr, bufs["ws"].ptr, ws_bytes, None)
    assert ret == 0, native.last_error()
    assert gpu.mfrt_device_sync() == 0
    return bufs


def _free(bufs):
    for b in bufs.values():
        b.free()


def _inputs(oracle, seed, T, H, K, E):
    x, logits = workloads.moe_inputs(seed, T, H, E, K)
    topk = np.zeros((T, K), dtype=np.int32)
    w = np.zeros((T, K), dtype=np.float32)
    oracle.orc_moe_route(np_ptr(logits), T, E, K, np_ptr(topk), np_ptr(w))
    return x, topk, w


@pytest.mark.parametrize("T,H,K,E", [
    (1, 8, 1, 1), (7, 64, 2, 4), (300, 64, 4, 16), (1000, 520, 8, 256), (129, 1024, 8, 300),
    (2050, 72, 16, 512), (4096, 2048, 8, 256), (511, 16384, 3, 37),
    (40000, 64, 8, 300),   # 320 000 entries in 313 rank blocks
    (5000, 8192, 2, 8),    # wide rows in two parts: every wave of the permute takes two or three (token, part) items
])
def test_dispatch_and_combine_match_the_specification(gpu, oracle, T, H, K, E):
    K = min(K, E)
    x, topk, w = _inputs(oracle, 0xC4 + T, T, H, K, E)
    exp_out, exp_counts, exp_offsets, exp_row, exp_src = _oracle_dispatch(oracle, x, topk, E)
    bufs = _gpu_dispatch(gpu, x, topk, E)
    try:
        assert np.array_equal(_fetch(bufs["counts"], np.int32, (E,)), exp_counts)
        assert np.array_equal(_fetch(bufs["offsets"], np.int32, (E,)), exp_offsets)
        assert np.array_equal(_fetch(bufs["row_of"], np.int32, (T * K,)), exp_row)
        assert np.array_equal(_fetch(bufs["src_of"], np.int32, (T * K,)), exp_src)
        assert np.array_equal(_fetch(bufs["out"], np.uint16, (T * K, H)), exp_out)
        assert _fetch(bufs["ws"], np.uint32, (1,))[0] == 0

        wdev = _dev(gpu, w)
        y = gpu_util.DeviceBuffer(gpu, T * H * 2)
        assert gpu.mf_moe_combine(bufs["out"].ptr, bufs["row_of"].ptr, wdev.ptr, T, H, K, y.ptr, None) == 0
        assert gpu.mfrt_device_sync() == 0
        got = _fetch(y, np.uint16, (T, H))
        exp_y = np.zeros((T, H), dtype=np.uint16)
        oracle.orc_moe_combine(np_ptr(exp_out), np_ptr(exp_row), np_ptr(w), T, H, K, np_ptr(exp_y))
        gf = workloads.bf16_words_to_f32(got).astype(np.float64)
        ef = workloads.bf16_words_to_f32(exp_y).astype(np.float64)
        assert np.all(np.abs(gf - ef) <= 1e-2 * np.abs(ef) + 1e-6)   # the stated tolerance
        assert np.array_equal(got, exp_y)                             # and in fact bit-equal
        wdev.free()
        y.free()
    finally:
        _free(bufs)


@pytest.mark.parametrize("T,H,K,E,routing", [
    (2000, 4096, 8, 64, "router"),     # 16 000 entries: fifteen full blocks and a last one of 640 entries
    (2500, 7168, 8, 300, "router"),    # twenty blocks, which the eight streams do not divide
    (2200, 7168, 8, 256, "five"),      # everything lands on five experts, duplicates inside a token included: long runs
    (2200, 5120, 8, 256, "bad ids"),   # some ids out of range: their slots name no row, the lists of their blocks are shorter
    (1200, 4096, 16, 128, "router"),   # sixty-four tokens per block
    (2800, 4096, 6, 64, "router"),     # blocks that begin and end inside a token
    (3000, 8256, 8, 1, "one"),         # one expert: the output is the input, every row eight times; rows that end inside a tile
    (2100, 16384, 8, 256, "router"),   # rows so wide that a step is half a block of entries
    (6000, 4096, 2, 8, "router"),      # top-2: 512 tokens per block, steps of half a block
    (2500, 12288, 8, 512, "bad ids"),  # 512 experts, half-block steps, slots without a row
    (700, 16384, 3, 37, "router"),     # steps of two slices (128 entries) that begin and end inside tokens
    (2100, 1024, 8, 32, "router"),     # rows of one tile
    (4000, 1600, 5, 100, "bad ids"),   # rows of one tile and a part of one
])
def test_output_ordered_permute(gpu, oracle, T, H, K, E, routing):
    """Rows wide enough and blocks enough for the permute that walks the output in runs of consecutive rows per
    expert, in tiles: every output row and every map against the oracle."""
    assert gpu.mf_moe_xcd_streams() == 1        # an MI355X in its default partition: the form under test is the one that runs
    x, topk, _ = _inputs(oracle, 0xD1 + T, T, H, min(K, E), E)
    rng = np.random.default_rng(T)
    if routing == "one":
        topk = np.zeros((T, K), dtype=np.int32)
    elif routing == "five":
        topk = rng.integers(0, 5, (T, K)).astype(np.int32)
        topk[::7, 0] = E - 1
    elif routing == "bad ids":
        topk = topk.copy()
        topk[rng.integers(0, T, 300), rng.integers(0, K, 300)] = E + 3
        topk[5, :] = -1                                     # a token nobody takes
    if routing == "bad ids":
        # the oracle refuses ids out of range; it is asked about the same routing with those entries sent to one
        # more expert behind the others, which leaves every row of the real experts where it is
        bad = (topk < 0) | (topk >= E)
        exp_out, exp_counts, exp_offsets, exp_row, exp_src = _oracle_dispatch(oracle, x, np.where(bad, E, topk).astype(np.int32), E + 1)
        exp_counts, exp_offsets = exp_counts[:E], exp_offsets[:E]
        exp_row = np.where(bad.reshape(-1), -1, exp_row)
    else:
        exp_out, exp_counts, exp_offsets, exp_row, exp_src = _oracle_dispatch(oracle, x, topk, E)
    bufs = _gpu_dispatch(gpu, x, topk, E)
    try:
        valid = int(exp_counts.sum())
        assert np.array_equal(_fetch(bufs["counts"], np.int32, (E,)), exp_counts)
        assert np.array_equal(_fetch(bufs["offsets"], np.int32, (E,)), exp_offsets)
        assert np.array_equal(_fetch(bufs["row_of"], np.int32, (T * K,)), exp_row)
        assert np.array_equal(_fetch(bufs["src_of"], np.int32, (T * K,))[:valid], exp_src[:valid])
        assert np.array_equal(_fetch(bufs["out"], np.uint16, (T * K, H))[:valid], exp_out[:valid])
        assert _fetch(bufs["ws"], np.uint32, (1,))[0] == (1 if routing == "bad ids" else 0)
    finally:
        _free(bufs)


def test_skewed_routing_with_empty_and_hot_experts(gpu, oracle):
    rng = np.random.default_rng(3)
    T, H, K, E = 3000, 128, 8, 256
    x, _ = workloads.moe_inputs(3, T, H, E, K)
    topk = rng.integers(0, 5, (T, K)).astype(np.int32)       # everything lands on 5 experts, duplicates included
    topk[::7, 0] = 255
    exp_out, exp_counts, exp_offsets, exp_row, exp_src = _oracle_dispatch(oracle, x, topk, E)
    bufs = _gpu_dispatch(gpu, x, topk, E)
    try:
        assert np.array_equal(_fetch(bufs["counts"], np.int32, (E,)), exp_counts)
        assert np.array_equal(_fetch(bufs["row_of"], np.int32, (T * K,)), exp_row)
        assert np.array_equal(_fetch(bufs["out"], np.uint16, (T * K, H)), exp_out)
    finally:
        _free(bufs)


@pytest.mark.parametrize("T,K,E", [(300, 8, 256), (600, 8, 64), (1024, 8, 512), (2048, 2, 8), (1100, 5, 17), (1025, 8, 256)])
def test_few_blocks_that_count_one_anothers_entries(gpu, oracle, T, K, E):
    """Two to eight blocks of 1024 entries rank without a histogram launch: each block counts the entries of the
    others.  Everything against the oracle, then with one id out of range in the last block only (block 0 has to
    find it for the status word), then clean again."""
    H = 1024
    x, topk, _ = _inputs(oracle, 0xF0 + T, T, H, K, E)
    exp_out, exp_counts, exp_offsets, exp_row, exp_src = _oracle_dispatch(oracle, x, topk, E)
    bufs = _gpu_dispatch(gpu, x, topk, E)
    try:
        assert _fetch(bufs["ws"], np.uint32, (1,))[0] == 0
        assert np.array_equal(_fetch(bufs["counts"], np.int32, (E,)), exp_counts)
        assert np.array_equal(_fetch(bufs["offsets"], np.int32, (E,)), exp_offsets)
        assert np.array_equal(_fetch(bufs["row_of"], np.int32, (T * K,)), exp_row)
        assert np.array_equal(_fetch(bufs["src_of"], np.int32, (T * K,)), exp_src)
        assert np.array_equal(_fetch(bufs["out"], np.uint16, (T * K, H)), exp_out)
    finally:
        _free(bufs)
    late = topk.copy()
    late[T - 1, K - 1] = E + 7
    sent = np.where(late >= E, E, late).astype(np.int32)
    exp_out, exp_counts, _, exp_row, _ = _oracle_dispatch(oracle, x, sent, E + 1)
    exp_row = np.where((late >= E).reshape(-1), -1, exp_row)
    bufs = _gpu_dispatch(gpu, x, late, E)
    try:
        assert _fetch(bufs["ws"], np.uint32, (1,))[0] == 1
        assert np.array_equal(_fetch(bufs["counts"], np.int32, (E,)), exp_counts[:E])
        assert np.array_equal(_fetch(bufs["row_of"], np.int32, (T * K,)), exp_row)
        assert np.array_equal(_fetch(bufs["out"], np.uint16, (T * K - 1, H)), exp_out[:T * K - 1])
    finally:
        _free(bufs)
    bufs = _gpu_dispatch(gpu, x, topk, E)
    try:
        assert _fetch(bufs["ws"], np.uint32, (1,))[0] == 0
    finally:
        _free(bufs)


def test_out_of_range_expert_ids_are_flagged_not_followed(gpu, oracle):
    T, H, K, E = 500, 64, 4, 32
    x, topk, _ = _inputs(oracle, 9, T, H, K, E)
    bad = topk.copy()
    bad[10, 1] = E
    bad[499, 3] = -3
    bufs = _gpu_dispatch(gpu, x, bad, E)
    try:
        assert _fetch(bufs["ws"], np.uint32, (1,))[0] == 1
        row_of = _fetch(bufs["row_of"], np.int32, (T * K,))
        assert row_of[10 * K + 1] == -1 and row_of[499 * K + 3] == -1
        good = np.delete(np.arange(T * K), [10 * K + 1, 499 * K + 3])
        assert sorted(row_of[good].tolist()) == list(range(T * K - 2))
        assert _fetch(bufs["counts"], np.int32, (E,)).sum() == T * K - 2
        # combine skips the two slots: with a NaN and an infinity in row 0 of the expert-contiguous
        # buffer the result still equals the oracle's, and nothing non-finite appears in y
        rows = _fetch(bufs["out"], np.uint16, (T * K, H)).copy()
        rows[T * K - 2:] = 0        # the two rows nobody was sent to
        row_of = row_of.copy()
        victim = int(np.where(row_of == 0)[0][0])
        rows[0, 0::2] = 0x7FC0
        rows[0, 1::2] = 0x7F80
        row_of[victim] = 1          # nobody reads the poisoned row
        w = np.random.default_rng(10).random((T, K), dtype=np.float32)
        rdev, rodev, wdev = _dev(gpu, rows), _dev(gpu, row_of), _dev(gpu, w)
        y = gpu_util.DeviceBuffer(gpu, T * H * 2)
        assert gpu.mf_moe_combine(rdev.ptr, rodev.ptr, wdev.ptr, T, H, K, y.ptr, None) == 0
        assert gpu.mfrt_device_sync() == 0
        got = _fetch(y, np.uint16, (T, H))
        exp_y = np.zeros((T, H), dtype=np.uint16)
        oracle.orc_moe_combine(np_ptr(rows), np_ptr(row_of), np_ptr(w), T, H, K, np_ptr(exp_y))
        assert np.array_equal(got, exp_y)
        assert not np.any((got & 0x7F80) == 0x7F80)
        for b in (rdev, rodev, wdev, y):
            b.free()
    finally:
        _free(bufs)
    # the same call with valid ids clears the flag again without any reset by the caller
    bufs = _gpu_dispatch(gpu, x, topk, E)
    try:
        assert _fetch(bufs["ws"], np.uint32, (1,))[0] == 0
    finally:
        _free(bufs)


@pytest.mark.parametrize("T,H,K", [
    (3600, 7168, 8),   # 25 200 slices: one period of three read parts for 5120 waves, then one read part and a short second
    (3300, 8000, 8),   # rows of 1000 units in eight slices of 125: ragged slices, a last period of two read parts and a short third
    (3200, 8192, 8),   # 25 600 slices: the last period ends with its second read part
    (3840, 8192, 8),   # 30 720: with its third, two whole periods
    (991, 31744, 8),   # one slice more: a third period of one wave
    (700, 1024, 8),    # narrow rows: one four-wave workgroup per token
    (60, 7168, 8),     # wide rows, few tokens: one workgroup per slice
    (300, 16384, 3),   # any other topK
    (500, 4096, 2),    # the slice kernel compiled for top-2
    (400, 7168, 4),    # ... top-4
    (300, 5120, 6),    # ... top-6
    (5100, 5120, 6),   # top-6, 25 500 slices of rows that a dispatch leaves in the last-level cache
    (5400, 5120, 6),   # top-6, 27 000 slices of more rows than that: waves that stay, as in the first shape
    (3600, 7168, 4),   # top-4 with as many slices: still one workgroup per slice
])
def test_combine_of_rows_that_differ_within_a_token(gpu, oracle, T, H, K):
    """After a dispatch the rows of a token are copies of one another, so a combine that mixed them up would still pass
    the dispatch-then-combine tests; here every row is different.  The first five shapes and the top-6 shape of 5400 tokens have enough tokens of wide rows
    for the combine whose waves stay and alternate between reading and writing: same bits as the oracle at the
    default pace, at a slow and at an absurdly fast one, with slots without a row, and with the form switched off."""
    rng = np.random.default_rng(T)
    rows = (rng.integers(0x3800, 0x4000, (T * K, H), dtype=np.uint16) | (rng.integers(0, 2, (T * K, H), dtype=np.uint16) << 15))
    row_of = rng.permutation(T * K).astype(np.int32)
    row_of[rng.integers(0, T * K, 50)] = -1
    victim = int(np.where(row_of == 0)[0][0]) if np.any(row_of == 0) else None
    if victim is not None:
        row_of[victim] = 1                      # nobody reads row 0, which holds a NaN and an infinity
    rows[0, 0::2] = 0x7FC0
    rows[0, 1::2] = 0x7F80
    w = rng.random((T, K), dtype=np.float32)
    exp_y = np.zeros((T, H), dtype=np.uint16)
    oracle.orc_moe_combine(np_ptr(rows), np_ptr(row_of), np_ptr(w), T, H, K, np_ptr(exp_y))
    rdev, rodev, wdev = _dev(gpu, rows), _dev(gpu, row_of), _dev(gpu, w)
    y = gpu_util.DeviceBuffer(gpu, T * H * 2)
    try:
        for rates in (native.MOE_COMBINE_WINDOWS_DEFAULT, (1000000, 1000000), (16000000, 16000000), (0, 0)):
            assert gpu.mf_moe_combine_windows(*rates) == 0, native.last_error()
            y.fill(0xEE)
            assert gpu.mf_moe_combine(rdev.ptr, rodev.ptr, wdev.ptr, T, H, K, y.ptr, None) == 0, native.last_error()
            assert gpu.mfrt_device_sync() == 0
            got = _fetch(y, np.uint16, (T, H))
            assert np.array_equal(got, exp_y), rates
            assert not np.any((got & 0x7F80) == 0x7F80)
        assert gpu.mf_moe_combine_windows(500, 6500000) == native.BM_INVALID_PARAM
        assert gpu.mf_moe_combine_windows(0, 6500000) == native.BM_INVALID_PARAM
    finally:
        assert gpu.mf_moe_combine_windows(*native.MOE_COMBINE_WINDOWS_DEFAULT) == 0
        for b in (rdev, rodev, wdev, y):
            b.free()


@pytest.mark.parametrize("T,H,K,stays", [
    (3510, 7168, 8, False),   # one token short of 96 slices a CU
    (3511, 7168, 8, True),    # one token more: 24 577 slices, one period and two read parts, the second short
    (2081, 7168, 8, False),   # more than 256 MiB, 57 slices a CU
    (6145, 2048, 8, False),   # the fewest entries beyond the dispatch that counts, 48 slices a CU
    (3845, 7168, 6, False), (3846, 7168, 6, True),      # where those rows end at top-6
    (8192, 3072, 6, False), (8193, 3072, 6, True),      # the fewest entries beyond the dispatch that counts, at 96 slices a CU
    (8200, 3072, 4, False),
])
def test_combine_where_its_waves_begin_to_stay(gpu, oracle, T, H, K, stays):
    assert gpu.mf_moe_combine_stays(T, H, K) == stays
    test_combine_of_rows_that_differ_within_a_token(gpu, oracle, T, H, K)
    assert gpu.mf_moe_combine_windows(0, 0) == 0
    try:
        assert gpu.mf_moe_combine_stays(T, H, K) == 0
    finally:
        assert gpu.mf_moe_combine_windows(*native.MOE_COMBINE_WINDOWS_DEFAULT) == 0


def test_same_workspace_reused_by_calls_of_different_sizes(gpu, oracle):
    """Histograms and status of one call must not leak into the next call on the same workspace."""
    E, K, H = 64, 4, 64
    sizes = [5000, 700, 5000, 33]
    ws_bytes = gpu.mf_moe_workspace_bytes(max(sizes), K, E)
    ws = gpu_util.DeviceBuffer(gpu, ws_bytes)
    ws.fill(0xFF)
    try:
        for i, T in enumerate(sizes):
            x, topk, _ = _inputs(oracle, 0xB0 + i, T, H, K, E)
            _, exp_counts, exp_offsets, exp_row, _ = _oracle_dispatch(oracle, x, topk, E)
            dt = _dev(gpu, topk)
            counts, offsets = gpu_util.DeviceBuffer(gpu, E * 4), gpu_util.DeviceBuffer(gpu, E * 4)
            row_of = gpu_util.DeviceBuffer(gpu, T * K * 4)
            assert gpu.mf_moe_dispatch(None, dt.ptr, T, H, K, E, None, counts.ptr, offsets.ptr, row_of.ptr, None, ws.ptr,
                                       ws_bytes, None) == 0, native.last_error()
            assert gpu.mfrt_device_sync() == 0
            assert np.array_equal(_fetch(counts, np.int32, (E,)), exp_counts)
            assert np.array_equal(_fetch(offsets, np.int32, (E,)), exp_offsets)
            assert np.array_equal(_fetch(row_of, np.int32, (T * K,)), exp_row)
            for b in (dt, counts, offsets, row_of):
                b.free()
    finally:
        ws.free()


def test_argument_errors(gpu):
    p = ctypes.c_void_p(0x1000)
    assert gpu.mf_moe_dispatch(p, None, 4, 8, 2, 4, p, p, p, p, None, p, 1 << 20, None) == native.BM_INVALID_PARAM
    assert gpu.mf_moe_dispatch(p, p, 4, 12, 2, 4, p, p, p, p, None, p, 1 << 20, None) == native.BM_INVALID_PARAM
    assert gpu.mf_moe_dispatch(p, p, 4, 8, 17, 4, p, p, p, p, None, p, 1 << 20, None) == native.BM_INVALID_PARAM
    assert gpu.mf_moe_dispatch(p, p, 4, 8, 2, 513, p, p, p, p, None, p, 1 << 20, None) == native.BM_INVALID_PARAM
    assert gpu.mf_moe_dispatch(p, p, 4, 8, 2, 4, p, p, p, p, None, p, 8, None) == native.BM_INVALID_PARAM
    assert gpu.mf_moe_combine(p, p, None, 4, 8, 2, p, None) == native.BM_INVALID_PARAM
    assert gpu.mf_moe_combine(p, p, p, 4, 9, 2, p, None) == native.BM_INVALID_PARAM


def test_full_size_local_share(gpu, oracle):
    """8192 tokens x 7168 bf16, 256 experts, top-8: whole outputs against the oracle, plus the
    size-independent properties (bijection, counts, one-hot combine returns the token)."""
    T, H, K, E = 8192, 7168, 8, 256
    x, topk, w = _inputs(oracle, 0xC4, T, H, K, E)
    exp_out, exp_counts, exp_offsets, exp_row, exp_src = _oracle_dispatch(oracle, x, topk, E)
    bufs = _gpu_dispatch(gpu, x, topk, E)
    try:
        row_of = _fetch(bufs["row_of"], np.int32, (T * K,))
        counts = _fetch(bufs["counts"], np.int32, (E,))
        assert counts.sum() == T * K
        assert np.array_equal(np.sort(row_of), np.arange(T * K))
        assert np.array_equal(counts, exp_counts)
        assert np.array_equal(_fetch(bufs["offsets"], np.int32, (E,)), exp_offsets)
        assert np.array_equal(row_of, exp_row)
        assert np.array_equal(_fetch(bufs["src_of"], np.int32, (T * K,)), exp_src)
        got_out = _fetch(bufs["out"], np.uint16, (T * K, H))
        assert np.array_equal(got_out, exp_out)
        del got_out

        wdev = _dev(gpu, w)
        y = gpu_util.DeviceBuffer(gpu, T * H * 2)
        assert gpu.mf_moe_combine(bufs["out"].ptr, bufs["row_of"].ptr, wdev.ptr, T, H, K, y.ptr, None) == 0
        assert gpu.mfrt_device_sync() == 0
        got = _fetch(y, np.uint16, (T, H))
        exp_y = np.zeros((T, H), dtype=np.uint16)
        oracle.orc_moe_combine(np_ptr(exp_out), np_ptr(exp_row), np_ptr(w), T, H, K, np_ptr(exp_y))
        gf = workloads.bf16_words_to_f32(got)
        ef = workloads.bf16_words_to_f32(exp_y)
        assert np.all(np.abs(gf - ef) <= 1e-2 * np.abs(ef) + 1e-6)
        assert np.array_equal(got, exp_y)
        # one-hot weights: combine(dispatch(x)) == x
        onehot = np.zeros((T, K), dtype=np.float32)
        onehot[:, 5] = 1.0
        wdev.upload(onehot.view(np.uint8).reshape(-1))
        assert gpu.mf_moe_combine(bufs["out"].ptr, bufs["row_of"].ptr, wdev.ptr, T, H, K, y.ptr, None) == 0
        assert gpu.mfrt_device_sync() == 0
        back = _fetch(y, np.uint16, (T, H))
        # the chain starts from +0, so a -0.0 input comes back as +0.0 (as it does in the oracle)
        assert np.array_equal(np.where(back == 0x8000, 0, back), np.where(x == 0x8000, 0, x))
        wdev.free()
        y.free()
    finally:
        _free(bufs)


@pytest.mark.parametrize("T,H,K,E", [
    (1, 8, 1, 1), (1, 8, 16, 512), (255, 8, 1, 3), (257, 520, 1, 512), (64, 1032, 16, 512), (63, 4104, 4, 8), (171, 7168, 6, 256),
    (4096, 16, 1, 2), (1365, 24, 3, 7), (512, 136, 8, 64), (256, 4096, 16, 16),    # 4095 and 4096 entries: the last in one launch
    (4097, 16, 1, 2), (1366, 24, 3, 7), (513, 1024, 8, 64),                        # the first beyond
])
def test_dispatch_around_the_one_launch_form(gpu, oracle, T, H, K, E):
    """Tails of the ids behind whole vectors and waves, parts of rows that end inside a lane's piece, every width of the
    slot loop, ids out of range, and the permutation alone."""
    x, topk, _ = _inputs(oracle, 0x5A + T, T, H, K, E)
    late = topk.copy()
    late[0, 0], late[T // 2, K - 1] = -1, E
    for ids in (topk, late):
        out_of_range = (ids < 0) | (ids >= E)
        sent = np.where(out_of_range, E, ids).astype(np.int32)
        exp_out, exp_counts, exp_offsets, exp_row, exp_src = _oracle_dispatch(oracle, x, sent, E + 1)
        valid = T * K - int(out_of_range.sum())
        for with_rows in (True, False):
            bufs = _gpu_dispatch(gpu, x, ids, E, with_rows)
            try:
                assert _fetch(bufs["ws"], np.uint32, (1,))[0] == int(valid != T * K)
                assert np.array_equal(_fetch(bufs["counts"], np.int32, (E,)), exp_counts[:E])
                assert np.array_equal(_fetch(bufs["offsets"], np.int32, (E,)), exp_offsets[:E])
                assert np.array_equal(_fetch(bufs["row_of"], np.int32, (T * K,)), np.where(out_of_range.reshape(-1), -1, exp_row))
                assert np.array_equal(_fetch(bufs["src_of"], np.int32, (valid,)), exp_src[:valid])
                if with_rows:
                    assert np.array_equal(_fetch(bufs["out"], np.uint16, (valid, H)), exp_out[:valid])
            finally:
                _free(bufs)


@pytest.mark.parametrize("T,H,K,E", [
    (4100, 10304, 2, 16),     # 84 MB of rows, the first to be read ahead of the permute; nine rank blocks, a last one of a few entries
    (4090, 10304, 2, 16),     # eight blocks, which need no histogram launch
    (14500, 8192, 1, 7),      # 238 MB: more than is read ahead
])
def test_rows_read_ahead_of_the_permute(gpu, oracle, T, H, K, E):
    x = np.arange(T * H, dtype=np.uint32).astype(np.uint16).reshape(T, H) ^ (np.arange(T, dtype=np.uint16)[:, None] * 3)
    topk = np.random.default_rng(T).integers(0, E, (T, K)).astype(np.int32)
    bufs = _gpu_dispatch(gpu, x, topk, E)
    try:
        order = np.argsort(topk.reshape(-1), kind="stable")
        assert np.array_equal(_fetch(bufs["src_of"], np.int32, (T * K,)), order)
        assert np.array_equal(_fetch(bufs["counts"], np.int32, (E,)), np.bincount(topk.reshape(-1), minlength=E))
        assert np.array_equal(_fetch(bufs["out"], np.uint16, (T * K, H)), x[order // K])
    finally:
        _free(bufs)


@pytest.mark.parametrize("T,H,K,E", [
    (185, 7168, 8, 256), (196, 7168, 8, 256), (383, 7168, 2, 8), (395, 7168, 2, 8),   # rows that its stores leave in the caches, or not
    (256, 72, 8, 256), (257, 72, 8, 256), (1025, 8, 16, 512),       # the last call whose tokens look at one another, the first that counts
    (1171, 24, 7, 65), (3073, 16, 3, 1), (2201, 1032, 2, 16),       # ids that end inside a vector; one expert; rows that end inside a wave
    (49152, 8, 1, 17), (49153, 8, 1, 17), (6145, 520, 8, 64),       # the last call that counts, and the first beyond
    (700, 5120, 8, 256), (703, 5128, 8, 256), (1000, 7168, 8, 128), (4100, 7168, 2, 8),   # each form of its stores
    (2674, 7168, 6, 256), (2675, 7168, 6, 256), (6200, 4104, 8, 16),                      # 255.9 and 256.2 MiB of rows; tokens that waves walk
])
def test_dispatch_that_counts_in_one_launch(gpu, T, H, K, E):
    """Against a stable sort; some ids out of range, whose entries get no row."""
    rng = np.random.default_rng(T + K)
    x = np.arange(T * H, dtype=np.uint32).astype(np.uint16).reshape(T, H) ^ (np.arange(T, dtype=np.uint32) * 3).astype(np.uint16)[:, None]
    topk = rng.integers(0, E, (T, K)).astype(np.int32)
    late = topk.copy()
    late.reshape(-1)[[1, T * K // 2, T * K - 1]] = [-1, E, 0x7FFFFFFF]
    for ids, with_rows in ((topk, True), (late, True), (late, False)):
        flat = np.where((ids < 0) | (ids >= E), E, ids).reshape(-1)
        order = np.argsort(flat, kind="stable")[:int((flat < E).sum())]
        row_of = np.full(T * K, -1, dtype=np.int32)
        row_of[order] = np.arange(len(order), dtype=np.int32)
        counts = np.bincount(flat, minlength=E + 1)[:E]
        bufs = _gpu_dispatch(gpu, x, ids, E, with_rows)
        try:
            assert _fetch(bufs["ws"], np.uint32, (1,))[0] == int(len(order) != T * K)
            assert np.array_equal(_fetch(bufs["counts"], np.int32, (E,)), counts)
            assert np.array_equal(_fetch(bufs["offsets"], np.int32, (E,)), np.cumsum(counts) - counts)
            assert np.array_equal(_fetch(bufs["row_of"], np.int32, (T * K,)), row_of)
            assert np.array_equal(_fetch(bufs["src_of"], np.int32, (len(order),)), order)
            if with_rows:
                assert np.array_equal(_fetch(bufs["out"], np.uint16, (len(order), H)), x[order // K])
        finally:
            _free(bufs)


@pytest.mark.parametrize("T,H,K,E", [
    (1, 8, 2, 1), (1, 64, 2, 8), (1, 7168, 3, 256), (2, 1032, 2, 5), (5, 16, 1, 3),       # fewer ids than a lane's four, and a few more
    (128, 4096, 8, 256), (129, 4096, 8, 8), (341, 520, 3, 37), (342, 520, 3, 37),         # a round of 1024 ids, and one that ends inside a vector
    (512, 2056, 4, 64), (1025, 1024, 2, 512), (683, 136, 3, 9), (4096, 64, 1, 256), (2048, 128, 2, 8),    # rounds behind the row's loads
    (320, 4096, 8, 256), (321, 4096, 8, 256), (568, 1024, 6, 64), (569, 1024, 6, 64), (64, 2048, 16, 256), (65, 2048, 16, 256),  # the last that compare
])
def test_dispatch_that_compares_in_one_launch(gpu, T, H, K, E):
    test_dispatch_that_counts_in_one_launch(gpu, T, H, K, E)


@pytest.mark.parametrize("T,H,K,E,counts", [
    (3250, 7168, 8, 256, True), (3251, 7168, 8, 256, False),    # at top-8, the most rows for the dispatch that counts, and a token more
    (3510, 7168, 8, 256, False), (3511, 7168, 8, 256, False), (6144, 4096, 8, 64, False),
    (2080, 7168, 8, 63, True), (2081, 7168, 8, 63, False),      # over few experts
    (3845, 7168, 6, 64, True), (3846, 7168, 6, 64, False), (4681, 7168, 4, 64, True), (4682, 7168, 4, 64, False),
    (4915, 7168, 4, 8, False), (4916, 7168, 4, 8, False), (6241, 7168, 2, 8, True), (6242, 7168, 2, 8, False),
])
def test_dispatch_where_the_tiles_begin(gpu, T, H, K, E, counts):
    assert gpu.mf_moe_dispatch_counts(T, H, K, E) == counts
    test_dispatch_that_counts_in_one_launch(gpu, T, H, K, E)


@pytest.mark.parametrize("T,H,K", [
    (1, 7168, 8), (3, 2048, 2), (33, 2056, 4),           # few entries: one column position per lane, rows of 256 and 257 units
    (512, 2048, 8), (513, 2048, 8),                      # the last call of 4096 entries and one beyond
    (682, 2064, 6),                                      # 4092 entries
    (1700, 4096, 2), (2048, 7168, 2),                    # 56 MB, and 117 MB at 4096 entries
    (9, 2040, 6), (40, 8, 2), (300, 1992, 4), (77, 512, 2), (21, 1536, 8),   # narrow rows: one workgroup per token
])
def test_combine_of_any_values(gpu, oracle, T, H, K):
    """Rows of all bit patterns (infinities, NaN, subnormal numbers) and weights down to 1e-38, tokens with and without
    slots that have no row: the oracle's bits, and NaN where it has NaN (which NaN is the hardware's matter)."""
    rng = np.random.default_rng(T * K + H)
    rows = rng.integers(0, 1 << 16, (T * K, H), dtype=np.uint16)
    plain = rng.random((T * K, H)) < 0.98                # most are ordinary, so that most results are
    rows[plain] = rows[plain] & 0x80FF | 0x3F00
    row_of = rng.permutation(T * K).astype(np.int32).reshape(T, K)
    row_of[rng.random((T, K)) < 0.05] = -1
    w = rng.random((T, K), dtype=np.float32)
    w[::3] *= np.float32(1e-38)
    expected = np.zeros((T, H), dtype=np.uint16)
    row_of = np.ascontiguousarray(row_of)
    oracle.orc_moe_combine(np_ptr(rows), np_ptr(row_of), np_ptr(w), T, H, K, np_ptr(expected))
    bufs = [_dev(gpu, a) for a in (rows, row_of, w)]
    y = gpu_util.DeviceBuffer(gpu, T * H * 2)
    try:
        y.fill(0xEE)
        assert gpu.mf_moe_combine(*[b.ptr for b in bufs], T, H, K, y.ptr, None) == 0, native.last_error()
        assert gpu.mfrt_device_sync() == 0
        got = _fetch(y, np.uint16, (T, H))
        nan = (expected & 0x7FFF) > 0x7F80
        assert np.array_equal((got & 0x7FFF) > 0x7F80, nan)
        assert np.array_equal(got[~nan], expected[~nan])
        assert np.any((expected & 0x7F80) == 0)          # subnormal results are among them
    finally:
        for b in bufs + [y]:
            b.free()


@pytest.mark.parametrize("T,K,E", [
    (3072, 8, 256), (3073, 8, 256),     # 24 blocks that count, 25 with a histogram launch
    (4097, 4, 128), (1229, 7, 130),     # 17 blocks, the last of 4 entries; 9 blocks
    (2048, 8, 64), (2049, 8, 64),       # fewer experts: up to 16 blocks
    (1024, 8, 63), (1025, 8, 63),       # fewer yet: up to 8
    (3000, 8, 512), (9000, 1, 200),     # the widest table; one entry per token
])
def test_more_blocks_that_count_one_anothers_entries(gpu, oracle, T, K, E):
    test_few_blocks_that_count_one_anothers_entries(gpu, oracle, T, K, E)


# Rounds of steps of eight, four and two blocks, of whole ones and of the parts of those that are left: the fewest blocks of each, one to seven left,
# blocks that end inside a token, a last one that is not full.
@pytest.mark.parametrize("T,H,K,E", [
    (8192, 2048, 8, 256), (8065, 2048, 8, 256), (8064, 2048, 8, 256), (6145, 2048, 8, 256), (16385, 2048, 8, 512), (9400, 2112, 7, 300), (6200, 2048, 16, 129),
    (7300, 4096, 8, 512), (7040, 4096, 8, 129), (6300, 4096, 8, 128), (4100, 7168, 8, 256), (5150, 7168, 8, 128), (6400, 7168, 8, 127), (4000, 8192, 8, 512),
    (6000, 7168, 6, 256), (5200, 7168, 4, 8), (5633, 7168, 4, 64), (9999, 4096, 4, 256), (8400, 1024, 8, 256),
])
@pytest.mark.parametrize("refused", [False, True])
def test_tiles_in_steps_of_several_blocks(gpu, T, H, K, E, refused):
    torch = pytest.importorskip("torch")
    g = torch.Generator(device="cuda")
    g.manual_seed(T + K)
    x = torch.randint(-2**63, 2**63 - 1, (T, H // 4), dtype=torch.int64, device="cuda", generator=g)
    ids = torch.randint(0, E, (T, K), dtype=torch.int32, device="cuda", generator=g)
    if refused:                                             # entries without a row, some all of a slice
        ids.view(-1)[torch.randint(0, T * K, (500,), device="cuda", generator=g)] = E
        ids.view(-1)[4096:4160] = -1
    flat = torch.where((ids < 0) | (ids >= E), E, ids).view(-1)
    order = torch.sort(flat, stable=True).indices[:int((flat < E).sum())]
    row_of = torch.full((T * K,), -1, dtype=torch.int32, device="cuda")
    row_of[order] = torch.arange(len(order), dtype=torch.int32, device="cuda")
    counts = torch.bincount(flat, minlength=E + 1)[:E].to(torch.int32)
    room = gpu.mf_moe_workspace_bytes(T, K, E)
    rows = torch.full((T * K + 1, H // 4), 0x5A, dtype=torch.int64, device="cuda")
    got = {name: torch.full((n,), -7, dtype=torch.int32, device="cuda") for name, n in
           (("counts", E), ("offsets", E), ("row_of", T * K), ("source_of", T * K), ("workspace", room // 4 + 1))}
    torch.cuda.synchronize()
    assert gpu.mf_moe_dispatch_counts(T, H, K, E) == 0
    assert gpu.mf_moe_dispatch(x.data_ptr(), ids.data_ptr(), T, H, K, E, rows.data_ptr(), got["counts"].data_ptr(), got["offsets"].data_ptr(),
                               got["row_of"].data_ptr(), got["source_of"].data_ptr(), got["workspace"].data_ptr(), room, None) == 0, native.last_error()
    assert gpu.mfrt_device_sync() == 0
    assert torch.equal(got["counts"], counts) and torch.equal(got["offsets"], (torch.cumsum(counts, 0) - counts).to(torch.int32))
    assert torch.equal(got["row_of"], row_of) and torch.equal(got["source_of"][:len(order)], order.to(torch.int32))
    assert int(got["workspace"][0]) == int(refused) and int(got["workspace"][-1]) == -7
    assert torch.equal(rows[:len(order)], x[order // K]) and bool((rows[len(order):] == 0x5A).all())
