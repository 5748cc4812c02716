"""What a program that uses this framework spends its time in, as cases that can be timed.

A case is a dict of plain values.  ``prepare`` makes what the program has in hand before the call (a pool and
its contents, the addresses of a batch, expert ids and weights, all from a seed), ``run`` makes the call through
the public entry points and returns everything it wrote.

Kinds of work ("op"), each over the range that ``draw`` spreads its sizes over:

* ``copy``      one contiguous copy inside the HBM pool (4 KiB to 1 GiB): hand-over of one tensor.
* ``kv``        the K and V blocks of every layer of one to sixteen requests, between two places of the HBM pool
                or between it and the pinned host pool (prefix cache hand-over, offload, restore).
* ``host``      tensors in ordinary, unpinned host memory to or from the HBM pool (64 KiB to 256 MiB): weights and
                saved caches that a Python program holds in numpy arrays.
* ``pages``     KV pages of one size gathered from random places of the pool into one buffer, or scattered back;
                the page addresses come as numpy arrays, or as a table that a kernel left in HBM.
* ``transfer``  a batch between two transfer sessions (prefill and decode side), equal blocks or byte lengths at
                arbitrary byte addresses, waited for or submitted to the program's own stream.
* ``moe``       dispatch of bf16 token rows to their experts and the weighted combine back, from the few tokens of
                a decode step to the thousands of a prefill.
* ``reshard``   decoder weights stored as tensor-parallel 8 laid out again as tensor-parallel 4.
"""

import ctypes
import math

import numpy as np
import torch

from memfabric_hybrid_amd import bm, native, workloads
from memfabric_hybrid_amd.transfer import TransferEngine

KIB, MIB, GIB = 1 << 10, 1 << 20, 1 << 30
STORE = "tcp://127.0.0.1:15432"


def listed():
    return [
        # One small tensor, and the caller waits: the latency of a call.
        {"name": "copy_16k", "op": "copy", "bytes": 16 * KIB, "source_offset": 0, "target_offset": 0, "wait": True},
        # The streaming ceiling: one large contiguous copy.
        {"name": "copy_1g", "op": "copy", "bytes": GIB, "source_offset": 0, "target_offset": 0, "wait": False},
        # One request of a 61-layer model, 122 blocks of 128 and 16 KiB: the framework's headline batch.
        {"name": "kv_1_request", "op": "kv", "requests": 1, "layers": 61, "k_bytes": 128 * KIB, "v_bytes": 16 * KIB,
         "path": "hbm", "wait": False},
        # The same blocks of four requests leave the GPU for the pinned host pool.
        {"name": "kv_4_offload", "op": "kv", "requests": 4, "layers": 61, "k_bytes": 128 * KIB, "v_bytes": 16 * KIB,
         "path": "to_host", "wait": True},
        # A numpy array of ordinary host memory goes into the pool.
        {"name": "host_load_64m", "op": "host", "parts": 1, "bytes": 64 * MIB, "path": "load"},
        # 4096 pages of 32 KiB (one K or V page of 16 tokens, 8 heads of 128) out of the pool into one buffer.
        {"name": "pages_gather_4096", "op": "pages", "pages": 4096, "page_bytes": 32 * KIB, "path": "gather",
         "table": "host"},
        # The way back, with the page table where a kernel computed it.
        {"name": "pages_scatter_4096", "op": "pages", "pages": 4096, "page_bytes": 32 * KIB, "path": "scatter",
         "table": "device"},
        # Odd lengths at odd addresses from one session to another, on the program's own stream.
        {"name": "transfer_ragged_2000", "op": "transfer", "segments": 2000, "most_bytes": 70000, "ragged": True,
         "path": "write", "wait": False},
        # A decode step: 64 tokens, 256 experts, top-8.
        {"name": "moe_64", "op": "moe", "tokens": 64, "hidden": 7168, "experts": 256, "topk": 8},
        # A prefill chunk of the same model.
        {"name": "moe_8192", "op": "moe", "tokens": 8192, "hidden": 7168, "experts": 256, "topk": 8},
        # One layer of the decoder, as a pipeline that overlaps the exchange with something else takes it.
        {"name": "reshard_1", "op": "reshard", "layers": 1, "hidden": 3584, "ffn": 18944},
        # The whole 7B decoder.
        {"name": "reshard_28", "op": "reshard", "layers": 28, "hidden": 3584, "ffn": 18944},
    ]


def _log_int(rng, low, high):
    return int(round(math.exp(rng.uniform(math.log(low), math.log(high)))))


def draw(rng):
    op = rng.choice(["copy", "kv", "host", "pages", "transfer", "moe", "reshard"])
    if op == "copy":
        nbytes = _log_int(rng, 4 * KIB, GIB)
        if rng.random() < 0.5:   # a tensor as allocators place it
            return {"op": op, "bytes": (nbytes + 255) // 256 * 256, "source_offset": 0, "target_offset": 0,
                    "wait": rng.random() < 0.5}
        return {"op": op, "bytes": nbytes, "source_offset": rng.randrange(256), "target_offset": rng.randrange(256),
                "wait": rng.random() < 0.5}
    if op == "kv":
        k_bytes, v_bytes = rng.choice([(128 * KIB, 16 * KIB), (32 * KIB, 32 * KIB), (64 * KIB, 64 * KIB)])
        return {"op": op, "requests": _log_int(rng, 1, 16), "layers": rng.choice([28, 32, 61]), "k_bytes": k_bytes,
                "v_bytes": v_bytes, "path": rng.choice(["hbm", "hbm", "to_host", "from_host"]),
                "wait": rng.random() < 0.5}
    if op == "host":
        return {"op": op, "parts": _log_int(rng, 1, 32), "bytes": _log_int(rng, 64 * KIB, 256 * MIB),
                "path": rng.choice(["load", "save"])}
    if op == "pages":
        page_bytes = rng.choice([8 * KIB, 16 * KIB, 32 * KIB, 64 * KIB])
        return {"op": op, "pages": _log_int(rng, 64, 16384), "page_bytes": page_bytes,
                "path": rng.choice(["gather", "scatter"]), "table": rng.choice(["host", "device"])}
    if op == "transfer":
        return {"op": op, "segments": _log_int(rng, 16, 8192), "most_bytes": _log_int(rng, 4 * KIB, 128 * KIB),
                "ragged": rng.random() < 0.5, "path": rng.choice(["write", "read"]), "wait": rng.random() < 0.5}
    if op == "moe":
        return {"op": op, "tokens": _log_int(rng, 1, 8192), "hidden": rng.choice([1024, 2048, 4096, 5120, 7168]),
                "experts": rng.choice([8, 64, 128, 256]), "topk": rng.choice([2, 4, 6, 8])}
    return {"op": op, "layers": _log_int(rng, 1, 28), "hidden": 128 * _log_int(rng, 8, 28),
            "ffn": 64 * _log_int(rng, 44, 296)}


# ---- memory and streams of the program -----------------------------------------------------------------------

class _Memory:
    """A pool and `nbytes` of its HBM for torch.  A tensor made of it holds it, so the pool lives as long as its last view."""

    free_ids = list(range(60, 0, -1))

    def __init__(self, nbytes, dram_bytes):
        self.id = self.free_ids.pop()
        self.handle = None
        self.handle = bm.create(self.id, _whole(dram_bytes), _whole(nbytes))
        self.ptr = self.handle.peer_rank_ptr(0, bm.BmMemType.DEVICE)
        self.__cuda_array_interface__ = {"data": (self.ptr, False), "shape": (nbytes,), "typestr": "|u1", "version": 2,
                                         "strides": None}

    def __del__(self):
        if self.handle is not None:
            torch.cuda.synchronize()
            self.handle.destroy()
        self.free_ids.append(self.id)


class _Pool:
    """A BigMemory pool and its local memory as a tensor (HBM) and an array (pinned host memory)."""

    def __init__(self, hbm_bytes, dram_bytes=0):
        memory = _Memory(hbm_bytes, dram_bytes)
        self.handle, self.hbm = memory.handle, memory.ptr
        self.tensor = torch.as_tensor(memory, device="cuda")
        if dram_bytes:
            self.dram = self.handle.peer_rank_ptr(0, bm.BmMemType.HOST)
            buffer = (ctypes.c_uint8 * dram_bytes).from_address(self.dram)
            buffer.memory = memory
            self.array = np.ctypeslib.as_array(buffer)


class _Session:
    """A transfer session and what it has registered."""

    count = 0

    def __init__(self, role, tensors):
        _start()
        _Session.count += 1
        self.name = f"127.0.0.1:{20000 + _Session.count % 40000}"
        self.engine = TransferEngine()
        self.tensors = tensors
        _ok(self.engine.initialize(STORE, self.name, role, 0))
        for t in tensors:
            _ok(self.engine.register_memory(t.data_ptr(), t.numel()))

    def __del__(self):
        torch.cuda.synchronize()
        for t in self.tensors:
            self.engine.unregister_memory(t.data_ptr())
        self.engine.destroy()


_stream = None


def _start():
    global _stream
    if _stream is None:
        _ok(bm.initialize(STORE, 1, 0))
        _stream = torch.cuda.Stream()


def _ok(code):
    if code != 0:
        raise RuntimeError(f"{code}: {native.last_error()}")


def _whole(nbytes):
    return (nbytes + 2 * MIB - 1) // (2 * MIB) * (2 * MIB)


def _random_bytes(tensor, seed):
    """Uniform bytes in a tensor whose length is a multiple of eight."""
    g = torch.Generator(device="cuda")
    g.manual_seed(seed)
    tensor.view(torch.int64).random_(-(1 << 62), 1 << 62, generator=g)


def _words(tensor):
    return tensor.view(torch.int64)


def _places(rng, sizes, region_bytes, align):
    """Offsets of disjoint ranges in [0, region_bytes), in random order with random gaps."""
    padded = (np.asarray(sizes, dtype=np.int64) + align - 1) // align * align
    slack = (region_bytes - int(padded.sum())) // align
    gaps = rng.multinomial(slack, np.full(len(padded) + 1, 1.0 / (len(padded) + 1)))[:-1] * align
    order = rng.permutation(len(padded))
    offsets = np.empty(len(padded), dtype=np.int64)
    offsets[order] = np.cumsum(gaps + padded[order]) - padded[order]
    return offsets


def _kv_sizes(case):
    one = [case["k_bytes"], case["v_bytes"]] * case["layers"]
    return np.array(one * case["requests"], dtype=np.int64)


def _part_sizes(case):
    """`bytes` split into `parts` tensors, all but the last of one size."""
    parts = case["parts"]
    each = case["bytes"] // parts
    return np.array([each] * (parts - 1) + [case["bytes"] - each * (parts - 1)], dtype=np.int64)


def _transfer_sizes(case, rng):
    n = case["segments"]
    return rng.integers(1, case["most_bytes"] + 1, size=n) if case["ragged"] else np.full(n, case["most_bytes"])


# ---- prepare ---------------------------------------------------------------------------------------------------

def prepare(case, seed):
    rng = np.random.default_rng([seed, 0xC0])
    _start()
    state = {"copy": _prepare_copy, "kv": _prepare_kv, "host": _prepare_host, "pages": _prepare_pages,
             "transfer": _prepare_transfer, "moe": _prepare_moe, "reshard": _prepare_reshard}[case["op"]](case, seed, rng)
    state["op"] = case["op"]
    torch.cuda.synchronize()
    return state


def _prepare_copy(case, seed, rng):
    half = _whole(case["bytes"] + 256)
    pool = _Pool(2 * half)
    _random_bytes(pool.tensor, seed)
    return {"pool": pool, "source": pool.hbm + case["source_offset"], "target": pool.hbm + half + case["target_offset"],
            "bytes": case["bytes"], "flags": 0 if case["wait"] else native.ASYNC_COPY_FLAG,
            "out": _words(pool.tensor[half:])}


def _prepare_kv(case, seed, rng):
    sizes = _kv_sizes(case)
    region = _whole(2 * int(sizes.sum()))
    path = case["path"]
    source = _places(rng, sizes, region, 4 * KIB)
    target = _places(rng, sizes, region, 4 * KIB)
    if path == "hbm":
        pool = _Pool(2 * region)
        source, target, out = source + pool.hbm, target + pool.hbm + region, _words(pool.tensor[region:])
    elif path == "to_host":
        pool = _Pool(region, region)
        source, target, out = source + pool.hbm, target + pool.dram, pool.array
    else:
        pool = _Pool(region, region)
        source, target, out = source + pool.dram, target + pool.hbm, _words(pool.tensor)
    _random_bytes(pool.tensor, seed)
    if path == "to_host":
        pool.array[:] = 0
    if path == "from_host":
        torch.from_numpy(pool.array).copy_(pool.tensor)
        _random_bytes(pool.tensor, seed + 1)
    return {"pool": pool, "sources": source.tolist(), "targets": target.tolist(), "sizes": sizes.tolist(), "out": out,
            "type": bm.BmCopyType.G2G, "flags": 0 if case["wait"] else native.ASYNC_COPY_FLAG}


def _prepare_host(case, seed, rng):
    sizes = _part_sizes(case)
    room = _whole(int(sizes.sum()) + 256 * len(sizes))
    pool = _Pool(room)
    _random_bytes(pool.tensor, seed)
    inside = _places(rng, sizes, room, 256) + pool.hbm
    load = case["path"] == "load"
    flat = np.full(int(sizes.sum()), 0, dtype=np.uint8)
    if load:   # what the program read from somewhere
        fresh = torch.empty(room, dtype=torch.uint8, device="cuda")
        _random_bytes(fresh, seed + 1)
        torch.from_numpy(flat).copy_(fresh[:len(flat)])
    arrays = np.split(flat, np.cumsum(sizes)[:-1])
    outside = [a.ctypes.data for a in arrays]
    return {"pool": pool, "arrays": arrays, "sources": outside if load else inside.tolist(),
            "targets": inside.tolist() if load else outside, "sizes": sizes.tolist(),
            "out": _words(pool.tensor) if load else flat,
            "type": bm.BmCopyType.H2G if load else bm.BmCopyType.G2H, "flags": 0}


def _prepare_pages(case, seed, rng):
    n, page = case["pages"], case["page_bytes"]
    pool = _Pool(_whole(4 * n * page))
    buffer = torch.empty(n * page, dtype=torch.uint8, device="cuda")
    _random_bytes(pool.tensor, seed)
    _random_bytes(buffer, seed + 1)
    paged = np.uint64(pool.hbm) + rng.choice(4 * n, size=n, replace=False).astype(np.uint64) * np.uint64(page)
    flat = np.uint64(buffer.data_ptr()) + np.arange(n, dtype=np.uint64) * np.uint64(page)
    gather = case["path"] == "gather"
    source, target = (paged, flat) if gather else (flat, paged)
    sizes = np.full(n, page, dtype=np.uint64)
    state = {"pool": pool, "buffer": buffer, "out": _words(buffer if gather else pool.tensor), "pages": n,
             "table": None}
    if case["table"] == "device":
        triples = np.stack([source, target, sizes], axis=1).view(np.int64)
        state["table"] = torch.from_numpy(np.ascontiguousarray(triples)).cuda()
    else:
        state.update(sources=source, targets=target, sizes=sizes,
                     type=bm.BmCopyType.G2L if gather else bm.BmCopyType.L2G)
    return state


def _prepare_transfer(case, seed, rng):
    sizes = _transfer_sizes(case, rng)
    align = 1 if case["ragged"] else 256
    region = _whole(2 * int(sizes.sum()) + align * len(sizes))
    own = torch.empty(region, dtype=torch.uint8, device="cuda")
    peer = torch.empty(region, dtype=torch.uint8, device="cuda")
    _random_bytes(own, seed)
    _random_bytes(peer, seed + 1)
    sessions = [_Session("Prefill", [own]), _Session("Decode", [peer])]
    write = case["path"] == "write"
    return {"sessions": sessions, "write": write, "wait": case["wait"], "out": _words(peer if write else own),
            "own": (_places(rng, sizes, region, align) + own.data_ptr()).tolist(),
            "peer": (_places(rng, sizes, region, align) + peer.data_ptr()).tolist(), "sizes": sizes.tolist()}


def _prepare_moe(case, seed, rng):
    tokens, hidden, experts, topk = case["tokens"], case["hidden"], case["experts"], case["topk"]
    g = torch.Generator(device="cuda")
    g.manual_seed(seed)
    x = torch.randn(tokens, hidden, generator=g, device="cuda").to(torch.bfloat16)
    picked, ids = torch.randn(tokens, experts, generator=g, device="cuda").topk(topk, dim=1)

    def whole(n):
        return torch.zeros(n, dtype=torch.int32, device="cuda")

    room = native.lib().mf_moe_workspace_bytes(tokens, topk, experts)
    return {"x": x, "ids": ids.to(torch.int32).contiguous(), "weights": picked.softmax(dim=1).contiguous(),
            "rows": torch.zeros(tokens * topk, hidden, dtype=torch.bfloat16, device="cuda"),
            "counts": whole(experts), "offsets": whole(experts), "row_of": whole(tokens * topk),
            "source_of": whole(tokens * topk), "y": torch.zeros_like(x), "room": room,
            "workspace": torch.empty(room, dtype=torch.uint8, device="cuda"),
            "tokens": tokens, "hidden": hidden, "experts": experts, "topk": topk}


def _prepare_reshard(case, seed, rng):
    tensors = workloads.reshard_tensors(case["hidden"], case["ffn"])
    _, _, source_bytes, target_bytes = workloads.reshard_layout(tensors, case["layers"])
    first = _whole(source_bytes)
    pool = _Pool(first + _whole(target_bytes))
    _random_bytes(pool.tensor, seed)
    segments, rectangles = workloads.reshard_plan(tensors, case["layers"], pool.hbm, pool.hbm + first)
    return {"pool": pool, "sources": [s for s, _, _ in segments], "targets": [d for _, d, _ in segments],
            "sizes": [n for _, _, n in segments], "out": _words(pool.tensor[first:]),
            "rectangles": (native.Copy2dDesc * len(rectangles))(*[native.Copy2dDesc(*r) for r in rectangles])}


# ---- run -------------------------------------------------------------------------------------------------------

def run(state):
    return {"copy": _run_copy, "kv": _run_batch, "host": _run_batch, "pages": _run_pages, "transfer": _run_transfer,
            "moe": _run_moe, "reshard": _run_reshard}[state["op"]](state)


def _run_copy(s):
    _ok(s["pool"].handle.copy_data(s["source"], s["target"], s["bytes"], bm.BmCopyType.G2G, s["flags"]))
    return s["out"]


def _run_batch(s):
    _ok(s["pool"].handle.copy_data_batch(s["sources"], s["targets"], s["sizes"], len(s["sizes"]), s["type"], s["flags"]))
    return s["out"]


def _run_pages(s):
    if s["table"] is None:
        _ok(s["pool"].handle.copy_data_batch(s["sources"], s["targets"], s["sizes"], s["pages"], s["type"],
                                             native.ASYNC_COPY_FLAG))
    else:
        _ok(native.lib().mf_xcopy_device_table(s["table"].data_ptr(), s["pages"], native.ROUTE_HBM, _stream.cuda_stream))
    return s["out"]


def _run_transfer(s):
    engine, peer = s["sessions"][0].engine, s["sessions"][1].name
    if s["wait"]:
        call = engine.batch_transfer_sync_write if s["write"] else engine.batch_transfer_sync_read
        _ok(call(peer, s["own"], s["peer"], s["sizes"]))
    else:
        call = engine.batch_transfer_async_write_submit if s["write"] else engine.batch_transfer_async_read_submit
        _ok(call(peer, s["own"], s["peer"], s["sizes"], _stream.cuda_stream))
    return s["out"]


def _run_moe(s):
    lib, stream = native.lib(), _stream.cuda_stream
    _ok(lib.mf_moe_dispatch(s["x"].data_ptr(), s["ids"].data_ptr(), s["tokens"], s["hidden"], s["topk"], s["experts"],
                            s["rows"].data_ptr(), s["counts"].data_ptr(), s["offsets"].data_ptr(), s["row_of"].data_ptr(),
                            s["source_of"].data_ptr(), s["workspace"].data_ptr(), s["room"], stream))
    # (a program runs its experts on the rows here)
    _ok(lib.mf_moe_combine(s["rows"].data_ptr(), s["row_of"].data_ptr(), s["weights"].data_ptr(), s["tokens"], s["hidden"],
                           s["topk"], s["y"].data_ptr(), stream))
    return {"rows": s["rows"].view(torch.int16), "counts": s["counts"], "offsets": s["offsets"], "row_of": s["row_of"],
            "source_of": s["source_of"], "y": s["y"]}


def _run_reshard(s):
    _ok(s["pool"].handle.copy_data_batch(s["sources"], s["targets"], s["sizes"], len(s["sizes"]), bm.BmCopyType.G2G,
                                         native.ASYNC_COPY_FLAG))
    _ok(native.lib().mf_xcopy_2d_batch(s["rectangles"], len(s["rectangles"]), native.ROUTE_HBM, None))
    return s["out"]


# ---- what a pass cannot do without -----------------------------------------------------------------------------

def work(case):
    op = case["op"]
    if op == "moe":
        tokens, hidden, entries = case["tokens"], case["hidden"], case["tokens"] * case["topk"]
        dispatch = 2 * tokens * hidden + 2 * entries * hidden + 12 * entries + 8 * case["experts"]
        combine = 2 * entries * hidden + 8 * entries + 2 * tokens * hidden
        return {"bytes": dispatch + combine, "flops": 2 * entries * hidden}
    if op in ("copy", "host"):
        payload = case["bytes"]
    elif op == "kv":
        payload = int(_kv_sizes(case).sum())
    elif op == "pages":
        payload = case["pages"] * case["page_bytes"]
    elif op == "transfer":   # lengths of a ragged batch are uniform from 1 byte on
        payload = case["segments"] * (case["most_bytes"] + 1) // 2 if case["ragged"] else \
            case["segments"] * case["most_bytes"]
    else:
        payload = workloads.reshard_layout(workloads.reshard_tensors(case["hidden"], case["ffn"]), case["layers"])[3]
    return {"bytes": 2 * payload, "flops": 0}


def tolerance(case):
    # Copies, permutations and their indexes are bytes and whole numbers; only the combined rows are rounded, to bf16.
    return {"rel": 5e-3, "max": 5e-2} if case["op"] == "moe" else "exact"
