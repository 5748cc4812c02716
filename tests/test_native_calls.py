"""The extension module behind the Python face: integers of every kind of sequence arrive as the same 64-bit words."""

import array
import ctypes
import os
import shutil
import subprocess
import sys
import types

import numpy as np
import pytest

from memfabric_hybrid_amd import bm, native
from memfabric_hybrid_amd.transfer import TransferEngine

VALUES = [0, 1, (1 << 30) - 1, 1 << 30, (1 << 60) - 1, 1 << 60, (1 << 63) - 1]
WIDE = VALUES + [1 << 63, (1 << 64) - 1]

KINDS = {
    "list": list, "tuple": tuple, "array": lambda v: array.array("Q", v),
    "numpy_u64": lambda v: np.array(v, dtype=np.uint64),
    "numpy_strided": lambda v: np.repeat(np.array(v, dtype=np.uint64), 2)[::2],
    "numpy_big_endian": lambda v: np.array(v, dtype=">u8"),
    "numpy_scalars": lambda v: list(np.array(v, dtype=np.uint64)),
    "ctypes": lambda v: (ctypes.c_uint64 * len(v))(*v),
    "numpy_i64": lambda v: np.array(v, dtype=np.uint64).astype(np.int64),
    "numpy_object": lambda v: np.array(v, dtype=object),
}


@pytest.mark.parametrize("kind", KINDS)
@pytest.mark.parametrize("n", [0, 1, 2, len(WIDE)])
def test_words_of_a_sequence(lib, kind, n):
    assert list(native.u64_array(KINDS[kind](WIDE[:n]))) == WIDE[:n]
    assert [p or 0 for p in native.ptr_array(KINDS[kind](WIDE[:n]))] == WIDE[:n]


def test_words_are_taken_modulo_two_to_the_64(lib):
    assert list(native.u64_array([-1, -(1 << 63), (1 << 64) + 5, True, 7.9, np.int32(-2)])) == \
        [(1 << 64) - 1, 1 << 63, 5, 1, 7, (1 << 64) - 2]
    assert list(native.u64_array(np.array([3, -3], dtype=np.int32))) == [3, (1 << 64) - 3]


@pytest.mark.parametrize("bad, error", [(["x"], ValueError), ([None], TypeError), ([[1]], TypeError)])
def test_elements_that_are_no_integers(lib, bad, error):
    with pytest.raises(error):
        native.u64_array(bad)
    with pytest.raises(error):
        bm.BigMemory(0x1000).copy_data_batch([1], bad, [1], 1, bm.BmCopyType.G2G)


def test_a_list_that_changes_while_it_is_read(lib):
    values = [1, 2, 3]

    class Shrinks:
        def __int__(self):
            del values[1:]
            return 1
    values[0] = Shrinks()
    with pytest.raises(RuntimeError):
        native.calls().fill((ctypes.c_uint64 * 3)(), values)


def test_a_module_built_for_another_interpreter_is_not_loaded(lib, tmp_path):
    """The module reads the layout of the interpreter's integers: a file without this interpreter's tag stays unused."""
    package = os.path.dirname(native.__file__)
    there = tmp_path / "memfabric_hybrid_amd"
    (there / "lib").mkdir(parents=True)
    for name in ("__init__.py", "native.py"):
        shutil.copy(os.path.join(package, name), there / name)
    shutil.copy(native.DATAPLANE_PATH, there / "lib")
    for name in ("_calls.so", "_calls.cpython-39-x86_64-linux-gnu.so"):
        shutil.copy(native.CALLS_PATH, there / "lib" / name)
    program = "from memfabric_hybrid_amd import native\ntry:\n    native.calls()\nexcept OSError as e:\n    print('refused', e)\n"
    done = subprocess.run([sys.executable, "-c", program], capture_output=True, text=True, cwd=tmp_path, timeout=120)
    assert done.returncode == 0 and done.stdout.startswith("refused"), (done.stdout, done.stderr[-2000:])


NESTED = """
from memfabric_hybrid_amd import bm
pool = bm.BigMemory(0x1000)
class Nests:
    def __int__(self):
        pool.copy_data_batch([7] * {inner}, [7] * {inner}, [7] * {inner}, {inner}, bm.BmCopyType.G2G)
        return 1
words = [1] * {outer}
words[{outer} // 2] = Nests()
for _ in range(3):
    print(pool.copy_data_batch(words, [2] * {outer}, [3] * {outer}, {outer}, bm.BmCopyType.G2G))
"""


@pytest.mark.parametrize("outer, inner", [(60000, 400000), (400000, 60000), (1000, 2000), (2000, 1000)])
def test_a_batch_call_inside_a_batch_call(lib, outer, inner):
    """The inner call outgrows, or leaves alone, the words the outer one is filling; in a process of its own."""
    done = subprocess.run([sys.executable, "-c", NESTED.format(outer=outer, inner=inner)], capture_output=True, text=True,
                          cwd=os.path.dirname(os.path.dirname(os.path.abspath(__file__))), timeout=120)
    assert done.returncode == 0, done.stderr[-2000:]
    assert done.stdout.split() == [str(native.SM_NOT_INITIALIZED)] * 3


def test_what_stands_for_a_function_is_made_for_one(lib):
    """The type behind lib.mf_moe_combine cannot be instantiated: such an object would have no function to call."""
    kind = type(lib.mf_moe_combine)
    assert kind is not type(lib.mf_xcopy_batch)
    for make in (kind, lambda: kind.__new__(kind), lambda: object.__new__(kind)):
        with pytest.raises(TypeError):
            make()


@pytest.mark.parametrize("content", [b"", b"no library", None])
def test_the_library_loads_beside_a_module_that_does_not(lib, monkeypatch, tmp_path, content):
    """The module's file missing, empty or broken: the library's functions are the ctypes ones, and calls() raises."""
    path = tmp_path / os.path.basename(native.CALLS_PATH)
    if content is not None:
        path.write_bytes(content)
    for name, value in (("CALLS_PATH", str(path)), ("_lib", None), ("_calls", None)):
        monkeypatch.setattr(native, name, value)
    assert issubclass(type(native.lib().mf_moe_combine), ctypes._CFuncPtr)
    assert native.lib().mf_moe_combine(None, None, None, 1, 8, 1, None, None) == lib.mf_moe_combine(None, None, None, 1, 8, 1, None, None) != 0
    with pytest.raises((ImportError, OSError)):
        native.calls()


def test_the_library_loads_beside_an_older_module(lib, monkeypatch):
    older = types.SimpleNamespace(copy_batch=native.calls().copy_batch)
    monkeypatch.setattr(native, "_lib", None)
    monkeypatch.setattr(native, "_calls", older)
    assert issubclass(type(native.lib().mf_moe_combine), ctypes._CFuncPtr)
    assert native.calls() is older


def test_codes_without_a_pool_or_a_session(lib):
    pool = bm.BigMemory(None)
    assert pool.copy_data(1, 2, 3, bm.BmCopyType.G2G) == native.SM_INVALID_PARAM
    assert pool.copy_data_batch([1], [2], [3], 1, bm.BmCopyType.G2G) == native.SM_INVALID_PARAM
    pool = bm.BigMemory(0x1000)
    assert pool.copy_data_batch([1], [2], [3], 1, bm.BmCopyType.G2G) == native.SM_NOT_INITIALIZED
    for count in (2, -1, 1 << 32):    # more than the sequences hold, or no count at all
        assert pool.copy_data_batch([1], [2], [3], count, bm.BmCopyType.G2G) == native.SM_INVALID_PARAM
    engine = TransferEngine()
    assert engine.batch_transfer_sync_write("127.0.0.1:2000", [1], [2], [3]) == -1
    engine._handle = 0x1000
    assert engine.batch_transfer_sync_read("127.0.0.1:2000", [1], [2, 3], [3]) == -1
    assert engine.batch_transfer_sync_read("127.0.0.1:2000", [1], [2], [3]) == native.SM_INVALID_PARAM


@pytest.mark.gpu
@pytest.mark.parametrize("kind", ["list", "tuple", "numpy_u64", "numpy_strided", "numpy_scalars"])
@pytest.mark.parametrize("n", [1, 128, 129, 4000])
def test_batch_copy_from_every_kind_of_sequence(lib, kind, n):
    assert bm.initialize("tcp://127.0.0.1:0", 1, 0) == 0, native.last_error()
    pool = bm.create(1, 0, 32 << 20)
    try:
        dev, rng = pool.peer_rank_ptr(0), np.random.default_rng(n)
        before = rng.integers(0, 256, 32 << 20, dtype=np.uint8)
        assert lib.mfrt_memcpy(dev, before.ctypes.data, before.nbytes) == 0
        sizes = rng.integers(1, 2049, n)
        source, target = rng.permutation(n) * 2048, (16 << 20) + rng.permutation(n) * 2048
        words = [KINDS[kind]((a.astype(np.uint64) + np.uint64(b)).tolist()) for a, b in ((source, dev), (target, dev), (sizes, 0))]
        assert pool.copy_data_batch(*words, n, bm.BmCopyType.G2G) == 0, native.last_error()
        after = np.empty_like(before)
        assert lib.mfrt_memcpy(after.ctypes.data, dev, after.nbytes) == 0
        for s, d, size in zip(source, target, sizes):
            before[d:d + size] = before[s:s + size]
        assert np.array_equal(after, before)
    finally:
        pool.destroy()
        bm.uninitialize()


@pytest.mark.gpu
@pytest.mark.parametrize("n", [1, 128, 129, 4000])
def test_arrays_of_a_batch_are_only_read(lib, tmp_path, n):
    """Addresses in a read-only map of a file and in a bytes object, some with bits above the lower 48."""
    assert bm.initialize("tcp://127.0.0.1:0", 1, 0) == 0, native.last_error()
    pool = bm.create(1, 0, 32 << 20)
    try:
        dev = pool.peer_rank_ptr(0)
        local = np.random.default_rng(n).integers(0, 256, (n, 2048), dtype=np.uint8)
        source = np.uint64(local.ctypes.data) + np.arange(n, dtype=np.uint64) * np.uint64(2048)
        source[::3] |= np.uint64(0x5A5A << 48)
        target = np.uint64(dev) + np.arange(n, dtype=np.uint64) * np.uint64(4096)
        target.tofile(tmp_path / "targets")
        for sources in (memoryview(source.tobytes()).cast("Q"), source):
            kept = bytes(sources)
            assert lib.mfrt_memset(dev, 0, 32 << 20) == 0
            targets = np.memmap(tmp_path / "targets", dtype=np.uint64, mode="r")
            assert pool.copy_data_batch(sources, targets, np.full(n, 2047), n, bm.BmCopyType.H2G) == 0, native.last_error()
            after = np.empty((n, 4096), dtype=np.uint8)
            assert lib.mfrt_memcpy(after.ctypes.data, dev, after.nbytes) == 0
            assert np.array_equal(after[:, :2047], local[:, :2047]) and not after[:, 2047:].any()
            assert bytes(sources) == kept
    finally:
        pool.destroy()
        bm.uninitialize()


@pytest.mark.gpu
@pytest.mark.parametrize("outer, inner", [(300, 200), (300, 3000)])
def test_a_batch_call_inside_a_batch_call_copies_both(lib, outer, inner):
    assert bm.initialize("tcp://127.0.0.1:0", 1, 0) == 0, native.last_error()
    pool = bm.create(1, 0, 32 << 20)
    try:
        dev = pool.peer_rank_ptr(0)
        before = np.random.default_rng(outer + inner).integers(0, 256, 32 << 20, dtype=np.uint8)
        assert lib.mfrt_memcpy(dev, before.ctypes.data, before.nbytes) == 0
        after = before.copy()

        def words(n, source, target):
            for i in range(n):
                after[target + 1024 * i:target + 1024 * i + 1000] = before[source + 1024 * i:source + 1024 * i + 1000]
            return [dev + source + 1024 * i for i in range(n)], [dev + target + 1024 * i for i in range(n)], [1000] * n

        nested = words(inner, 4 << 20, 16 << 20)
        sources, targets, sizes = words(outer, 0, 24 << 20)

        class Nests:
            def __init__(self, value):
                self.value = value

            def __int__(self):
                assert pool.copy_data_batch(*nested, inner, bm.BmCopyType.G2G) == 0, native.last_error()
                return self.value
        sources[outer // 2] = Nests(sources[outer // 2])
        assert pool.copy_data_batch(sources, targets, sizes, outer, bm.BmCopyType.G2G) == 0, native.last_error()
        got = np.empty_like(before)
        assert lib.mfrt_memcpy(got.ctypes.data, dev, got.nbytes) == 0
        assert np.array_equal(got, after)
    finally:
        pool.destroy()
        bm.uninitialize()


class _Int(int):
    pass


@pytest.mark.parametrize("args", [
    (0x1000, 0x2000, 0x3000, 0, 64, 8, 0x4000, None), (None, None, None, 1, 64, 1, None, None),
    (0x1000, 0x2000, 0x3000, 1, 12, 8, 0x4000, 0), (0x1008, 0x2000, 0x3000, 1 << 32, 64, 8, 0x4000, 0),       # numbers modulo 2^32: no tokens
    (0x1000, 0x2000, 0x3000, 1, 64, (1 << 32) + 17, 0x4000, 0), (0x1000, 0x2000, 0x3000, -1, -1, -1, 0x4000, 0),
    ((1 << 64) + 0x1001, 0x2000, 0x3000, 1, 64, 8, 0x4000, 0), (-15, 0x2000, 0x3000, 1, 64, 8, 0x4000, 0),    # addresses modulo 2^64
    (ctypes.c_void_p(0), 0x2000, 0x3000, 1, 64, 8, 0x4000, None), (_Int(0x1001), True, 0x3000, 1, 64, 8, 0x4000, None),
    (0x1001, 0x2000, 0x3000, ctypes.c_uint32(1), 64, 8, 0x4000, None), (0x1001, 0x2000, 0x3000, 1, 64, 8, 0x4000, None, 5),
    (0x1001, 0x2000, 0x3000, 1, 64, 8, 0x4000), (), (1.0, 0, 0, 0, 0, 0, 0, 0), (0, 0, 0, None, 0, 0, 0, 0), (0, "x", 0, 0, 0, 0, 0, 0),
    (np.int64(4096), 0, 0, 0, 0, 0, 0, 0), (0, 0, 0, np.uint32(1), 0, 0, 0, 0),
], ids=str)
def test_calls_past_ctypes_are_what_ctypes_makes_of_them(lib, args):
    """None of them gets to the GPU: what the library refuses, and why, and what ctypes refuses."""
    def outcome(function):
        try:
            return function(*args), native.last_error()
        except Exception as e:
            return type(e), str(e)
    direct, plain = lib.mf_moe_combine, lib["mf_moe_combine"]
    plain.restype, plain.argtypes = native._SIGNATURES["mf_moe_combine"]
    assert type(direct) is not type(plain)
    lib.mf_moe_combine_windows(1, 1)                    # another message in between
    expect = outcome(plain)
    assert expect[0] != 0
    lib.mf_moe_combine_windows(1, 1)
    assert outcome(direct) == expect


def test_a_call_past_ctypes_has_its_attributes(lib):
    direct = lib.mf_moe_dispatch
    assert (direct.restype, direct.argtypes) == native._SIGNATURES["mf_moe_dispatch"] and direct.__name__ == "mf_moe_dispatch" and callable(direct)
    assert ctypes.cast(direct, ctypes.c_void_p).value == ctypes.cast(lib["mf_moe_dispatch"], ctypes.c_void_p).value
    with pytest.raises(AttributeError):
        direct.nothing
    other = native.calls().direct("mf_moe_combine", lib["mf_moe_combine"])
    other.restype, other.argtypes = ctypes.c_bool, native._SIGNATURES["mf_moe_combine"][1]      # what is set holds
    assert other(0, 0, 0, 0, 0, 0, 0, 0) is True
    assert native.calls().direct("hybm_uninit", lib.hybm_uninit) is lib.hybm_uninit
