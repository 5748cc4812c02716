// Batched discrete copy ("xcopy") for gfx950: one fused launch moves every
// segment of a batch, whatever mix of lengths it holds.
//
// Replaces the device side of the reference's copy plugin
// (src/hybm/csrc/copy_extend/hybm_copy_kernel.cpp:44-119: 32 blocks, whole
// segments per block, one 64 KiB staging tile, load and store serialised).
// Here a workgroup owns a chunk of bytes, not a segment; data goes
// register-to-register with four 128-bit loads in flight per lane, and
// the descriptor lookup costs one memory round trip (the table comes out of
// the kernel-argument block into registers, two rows per lane) for batches
// of up to 128 segments.
//
// Bound: HBM bandwidth (2 bytes of traffic per payload byte) for device to
// device, the host link (1 byte per payload byte) when one side is pinned
// host memory.  No LDS, no MFMA: nothing here is reused or contracted.
#include <hip/hip_runtime.h>
#include <hip/hip_ext.h>
#include <stdint.h>

#include <atomic>
#include <mutex>
#include <type_traits>
#include <vector>

#include <cstdlib>

#include "xcopy_plan.h"
#include "launch.h"
#include "through.h"
#include "window_clock.h"
#include "../rt/mf_rt.h"

namespace mf {
namespace {

typedef uint32_t u32x4 __attribute__((ext_vector_type(4)));
typedef u32x4 u32x4_any __attribute__((aligned(1)));  // source side may sit at any byte address

#define MF_GLOBAL __attribute__((address_space(1)))
typedef const MF_GLOBAL u32x4_any *GSrcUnit;
typedef MF_GLOBAL u32x4 *GDstUnit;
typedef const MF_GLOBAL uint8_t *GSrcByte;
typedef MF_GLOBAL uint8_t *GDstByte;

// Cache policy of one launch.  Addressing is the same for all of them.
//   HBM to HBM          streaming loads and streaming stores (nothing is reused)
//   to pinned host      plain loads, stores written through at system scope as they are issued
//   from pinned host    streaming loads, plain stores into HBM
enum StoreMode : int { kStorePlain = 0, kStoreStream = 1, kStoreThrough = 2 };

struct Policy {
    bool ntLoad;
    int store;
};

template <bool kNtLoad>
__device__ __forceinline__ u32x4 LoadUnit(uint64_t addr)
{
    GSrcUnit p = reinterpret_cast<GSrcUnit>(addr);
    if (kNtLoad) {
        return __builtin_nontemporal_load(p);
    }
    return *p;
}

__device__ __forceinline__ u32x4 LoadAligned(uint64_t addr)
{
    return __builtin_nontemporal_load(reinterpret_cast<const MF_GLOBAL u32x4 *>(addr));
}

// kStoreStream: nontemporal hint, the line may still linger dirty in L2 until the end of the kernel.
// kStoreThrough: nontemporal and written through at system scope, so that the write-back of the
// destination overlaps the copy instead of trailing it.
template <int kStore>
__device__ __forceinline__ void StoreUnit(uint64_t addr, u32x4 v)
{
    GDstUnit p = reinterpret_cast<GDstUnit>(addr);
    if (kStore == kStoreThrough) {
        StoreThrough16(addr, v);
    } else if (kStore == kStoreStream) {
        __builtin_nontemporal_store(v, p);
    } else {
        *p = v;
    }
}

template <int kStore>
__device__ __forceinline__ void CopyByte(uint64_t src, uint64_t dst)
{
    GDstByte p = reinterpret_cast<GDstByte>(dst);
    const uint8_t v = *reinterpret_cast<GSrcByte>(src);
    if (kStore == kStoreThrough) {
        StoreThrough1(dst, v);
    } else {
        *p = v;
    }
}

// The unit of the source that the next lane holds; lane 63 gets `wrap`.
__device__ __forceinline__ uint32_t NextLane(uint32_t v, uint32_t wrap)
{
    const uint32_t next = __builtin_amdgcn_update_dpp(0u, v, 0x130, 0xf, 0xf, true);   // wave_shl:1
    return (threadIdx.x & 63u) == 63u ? wrap : next;
}

// Sixteen bytes from byte 4 * kWords + bytes of the pair (a, b) on.
template <uint32_t kWords>
__device__ __forceinline__ u32x4 Straddle(u32x4 a, u32x4 b, uint32_t bytes)
{
    const uint32_t w[8] = {a[0], a[1], a[2], a[3], b[0], b[1], b[2], b[3]};
    u32x4 r;
#pragma unroll
    for (uint32_t i = 0; i < 4; ++i) {
        r[i] = __builtin_amdgcn_alignbyte(w[i + kWords + 1], w[i + kWords], bytes);
    }
    return r;
}

// A source that differs from its destination modulo 16, read in whole aligned units: loads that straddle units cost twice the cache
// accesses (4.9 MB of ragged segments 4.7 / 3.9 us, 69 MB 30.4 / 29.2).  A wave takes kUnits * 64 consecutive ones from u0 on, of
// those 0 ... end that hold any of the bytes, so that what a lane lacks is in the next lane's unit; `last` is what lane 63 of
// its last unit lacks.  Up to 15 bytes beside the source are read, of units that hold some of its bytes, and none in front of unit `lead`.
template <uint32_t kUnits>
__device__ __forceinline__ void LoadApart(u32x4 (&v)[kUnits], u32x4 &last, uint64_t aligned, uint32_t u0, uint32_t end, uint32_t lead = 0)
{
    const uint32_t u = u0 + (threadIdx.x & 63u);
#pragma unroll
    for (uint32_t j = 0; j < kUnits; ++j) {
        if (u + j * 64 - lead <= end - lead) {
            v[j] = LoadAligned(aligned + (u + j * 64) * kUnitBytes);
        }
    }
    const uint32_t behind = u0 + kUnits * 64 < end ? u0 + kUnits * 64 : end;
    last = LoadAligned(aligned + behind * kUnitBytes);
}

template <int kStore, uint32_t kUnits>
__device__ __forceinline__ void StoreApart(const u32x4 (&v)[kUnits], u32x4 last, uint64_t dst, uint32_t u0, uint32_t end, uint32_t apart,
                                           uint32_t lane = threadIdx.x & 63u, uint32_t lead = 0)
{
    const uint32_t u = u0 + lane;
    auto store = [&](auto words) {
#pragma unroll
        for (uint32_t j = 0; j < kUnits; ++j) {
            u32x4 next;
#pragma unroll
            for (uint32_t i = 0; i < 4; ++i) {
                const uint32_t wrap = j + 1 < kUnits ? v[j + 1 < kUnits ? j + 1 : 0][i] : last[i];
                next[i] = NextLane(v[j][i], __builtin_amdgcn_readfirstlane(wrap));
            }
            const u32x4 r = Straddle<decltype(words)::value>(v[j], next, apart & 3u);
            if (u + j * 64 - lead < end - lead) {
                StoreUnit<kStore>(dst + (u + j * 64) * kUnitBytes, r);
            }
        }
    };
    switch (apart >> 2) {
        case 0: store(std::integral_constant<uint32_t, 0>()); break;
        case 1: store(std::integral_constant<uint32_t, 1>()); break;
        case 2: store(std::integral_constant<uint32_t, 2>()); break;
        default: store(std::integral_constant<uint32_t, 3>()); break;
    }
}

constexpr uint32_t kDepth = 4;                          // 128-bit loads in flight per lane

// Wait until `ticks` of the constant-rate clock have passed since t0, after the loads have landed (so
// that the wait runs concurrently with the load latency instead of on top of it).
__device__ __forceinline__ void HoldStores(uint64_t t0, uint32_t ticks)
{
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
    while (wall_clock64() - t0 < ticks) {
        __builtin_amdgcn_s_sleep(1);
    }
}

// Copy chunk k of one segment.  All arguments are wave-uniform.  lanes: 64, 128 or 256, the launcher's choice.  kHold: the stores of the first step wait
// for HoldStores(t0, ticks).
template <bool kNtLoad, int kStore, bool kHold = false>
__device__ __forceinline__ void CopyChunk(uint64_t src, uint64_t dst, uint64_t len, uint64_t k, uint32_t units, uint64_t t0 = 0,
                                          uint32_t ticks = 0, uint32_t lanes = blockDim.x, uint32_t tid = threadIdx.x)
{
    const SegGeom g = SegmentGeometry(dst, len);
    const uint64_t u0 = k * units;
    const uint64_t left = g.body > u0 ? g.body - u0 : 0;
    const uint32_t n = left < units ? static_cast<uint32_t>(left) : units;
    const uint64_t s = src + g.head + u0 * kUnitBytes;
    const uint64_t d = dst + g.head + u0 * kUnitBytes;
    const uint32_t kTile = kDepth * lanes;              // units one workgroup moves per step

    uint32_t i = 0;
    const uint32_t apart = static_cast<uint32_t>(s) & (kUnitBytes - 1);
    if (kStore == kStoreStream && apart != 0) {
        for (; i < n; i += kTile) {
            u32x4 v[kDepth];
            u32x4 last;
            const uint32_t u = i + (tid >> 6) * kDepth * 64;
            LoadApart(v, last, s - apart, u, n);
            if (kHold && i == 0) {
                HoldStores(t0, ticks);
            }
            StoreApart<kStore>(v, last, d, u, n, apart);
        }
    }
    for (; i + kTile <= n; i += kTile) {
        u32x4 v[kDepth];
#pragma unroll
        for (uint32_t j = 0; j < kDepth; ++j) {
            v[j] = LoadUnit<kNtLoad>(s + static_cast<uint64_t>(i + j * lanes + tid) * kUnitBytes);
        }
        if (kHold && i == 0) {
            HoldStores(t0, ticks);
        }
#pragma unroll
        for (uint32_t j = 0; j < kDepth; ++j) {
            StoreUnit<kStore>(d + static_cast<uint64_t>(i + j * lanes + tid) * kUnitBytes, v[j]);
        }
    }
    if (i < n) {
        u32x4 v[kDepth];
#pragma unroll
        for (uint32_t j = 0; j < kDepth; ++j) {
            const uint32_t u = i + j * lanes + tid;
            if (u < n) {
                v[j] = LoadUnit<kNtLoad>(s + static_cast<uint64_t>(u) * kUnitBytes);
            }
        }
        if (kHold && i == 0) {
            HoldStores(t0, ticks);
        }
#pragma unroll
        for (uint32_t j = 0; j < kDepth; ++j) {
            const uint32_t u = i + j * lanes + tid;
            if (u < n) {
                StoreUnit<kStore>(d + static_cast<uint64_t>(u) * kUnitBytes, v[j]);
            }
        }
    }
    if (k == 0 && tid < g.head) {
        CopyByte<kStore>(src + tid, dst + tid);
    }
    if (u0 + units >= g.body && tid < g.tail) {
        const uint64_t off = g.head + g.body * kUnitBytes + tid;
        CopyByte<kStore>(src + off, dst + off);
    }
}

__device__ __forceinline__ uint64_t ReadLane64(uint64_t v, uint32_t lane)
{
    const uint32_t lo = __builtin_amdgcn_readlane(static_cast<uint32_t>(v), lane);
    const uint32_t hi = __builtin_amdgcn_readlane(static_cast<uint32_t>(v >> 32), lane);
    return (static_cast<uint64_t>(hi) << 32) | lo;
}

// The plan sits in the kernel-argument block.  Every lane fetches "its" two
// table rows (rows lane and lane + 64) with loads that depend on nothing but
// the lane id, so the whole table is in registers after ONE memory round
// trip; the owner of a chunk is then found with two ballots and read out of
// the owning lane.  (A scalar search would chain three dependent loads, each
// a full L2 round trip, before the first byte of payload is requested.)
struct InlineChunk {
    uint64_t src;
    uint64_t dst;
    uint32_t len;
    uint32_t k;
};

struct InlineRows {
    uint32_t f0, f1, l0, l1;
    uint64_t s0, s1, d0, d1;

    __device__ __forceinline__ explicit InlineRows(const InlinePlan &p)
    {
        const uint32_t lane = threadIdx.x & 63u;
        f0 = p.first[lane];
        f1 = p.first[lane + 64];
        s0 = p.src[lane];
        s1 = p.src[lane + 64];
        d0 = p.dst[lane];
        d1 = p.dst[lane + 64];
        l0 = p.len[lane];
        l1 = p.len[lane + 64];
    }
    // rows are ordered by prefix: the owner is the last row whose prefix is <= c
    __device__ __forceinline__ InlineChunk Owner(uint32_t c) const
    {
        const uint32_t below = __popcll(__ballot(f0 <= c)) + __popcll(__ballot(f1 <= c));
        const uint32_t s = below - 1;
        const uint32_t row = s & 63u;
        InlineChunk r;
        if (s < 64) {
            r.src = ReadLane64(s0, row);
            r.dst = ReadLane64(d0, row);
            r.len = __builtin_amdgcn_readlane(l0, row);
            r.k = c - __builtin_amdgcn_readlane(f0, row);
        } else {
            r.src = ReadLane64(s1, row);
            r.dst = ReadLane64(d1, row);
            r.len = __builtin_amdgcn_readlane(l1, row);
            r.k = c - __builtin_amdgcn_readlane(f1, row);
        }
        return r;
    }
};

// kHold: every wave keeps its loaded data until `holdTicks` of the constant-rate clock after its own
// start, which separates the read burst of the launch from its write burst (HoldNanosFor has the
// rule); such a launch has one chunk per workgroup: of 4 KiB (kHoldShallow, four loads per lane) or, for
// batches whose 4 KiB chunks would outnumber the waves the chip holds at once, of 16 KiB (kHoldDeep).
enum HoldMode : int { kHoldNone = 0, kHoldShallow = 1, kHoldDeep = 2 };

template <bool kNtLoad, int kStore, int kHold>
__device__ __forceinline__ void CopyChunkHeld(uint64_t src, uint64_t dst, uint64_t len, uint64_t k, uint32_t units, uint64_t t0,
                                              uint32_t ticks, uint32_t lanes = blockDim.x);

template <bool kNtLoad, int kStore, int kHold = kHoldNone>
__global__ __launch_bounds__(kXcopyThreads) void XcopyInlineKernel(const InlinePlan p, uint32_t holdTicks)
{
    const uint64_t t0 = kHold != kHoldNone ? wall_clock64() : 0;
    const InlineRows rows(p);
    const uint32_t nchunk = p.nchunk;
    const uint32_t units = p.units;
    // The host launches at most nchunk workgroups (and never this kernel for an empty plan), so
    // the first chunk needs no bound check and the table loads above are not held behind one.
    uint32_t c = blockIdx.x;
    do {
        const InlineChunk r = rows.Owner(c);
        CopyChunkHeld<kNtLoad, kStore, kHold>(r.src, r.dst, r.len, r.k, units, t0, holdTicks);
        c += gridDim.x;
    } while (c < nchunk);
}

// Read and write windows.  A copy that runs for hundreds of microseconds streams faster when the whole chip
// alternates between reading and writing than when every wave stores as soon as its loads have landed:
// HBM then sees long bursts of one direction instead of a mix (6.7 against 6.2 TB/s on 1 to 2 GiB).  The
// waves need no communication for that beyond the start, only the constant-rate clock every wave can read:
// a period is cut into a read half and a write half, wave i of a launch of G waves issues the 16 loads per
// lane of its next 16 KiB chunk at offset i * (period / 2) / G into the read half, waits for them, and
// issues the stores at the same offset into the write half.  The period is the time the launch's
// 2 * G * 16 KiB per round need at a target rate; up to a rate the part sustains, the copy runs at the pace
// the clock sets, beyond it the windows dissolve and the copy runs as it does without them.  A wave that
// is late proceeds at once (skipping to a later period made a dissolved launch slower).
constexpr uint32_t kWindowDepth = 16;                       // 128-bit loads per lane and round
constexpr uint32_t kWindowUnits = 64 * kWindowDepth;        // 16 KiB chunks, one wave each
constexpr uint32_t kWindowWaves = 4096;                     // 16 per CU
// XcopyWindowKernel's, XcopyPieceWindowKernel's and XcopySampledKernel's, 24 per CU.  A period of half as many waves again is as much
// longer, so a wave whose loads land late has more of it to catch up in, and HBM turns round less often.  The mean of sixteen launches in
// pairs, us:
//                                        waves   4096   5120   6144
//   128 segments of 9 MB at 7.1 TB/s              359    355    346
//   the same at 7.4                               377    357    351
//   128 of 2.4 MB at 7.4                          102     93     90
//   170 MiB at 7.6                               56.4   55.8   52.2
//   512 MiB shifted at 7.1                        164    168    161
// 7168 waves are as many as there are registers for the data of, and spill what else they need (170 MiB at 7.6 52.5).  The read and the
// write part as long as each other: 47 and 53 % of the period for reads are no better; nor are parts that issue in 95 or 90 % of their
// time and leave the rest for stragglers (128 segments of 9 MB at 7.2 346 and 379, at 100 % 348).
constexpr uint32_t kLongWavesPerSimd = 6;
constexpr uint32_t kLongWaves = 6144;
static_assert(kLongWaves <= kHeldMaxPieces && kLongWaves % kPieceGroup == 0,
              "a round of pieces is whole groups, and a table of more than kPlannedSegments has a workgroup for each wave");

// Chunk c of a segment; with onLines one of LineChunks(), as a segment of its own.
struct SegChunk {
    uint64_t src;
    uint64_t dst;
    uint64_t len;
    uint32_t k;
};
__device__ __forceinline__ SegChunk ChunkOn(bool onLines, uint64_t src, uint64_t dst, uint64_t len, uint32_t c, uint32_t units)
{
    if (!onLines) {
        return SegChunk{src, dst, len, c};
    }
    const LineSpan span = LineChunk(dst, len, c, units);
    return SegChunk{src + span.begin, dst + span.begin, span.end - span.begin, 0};
}

// One chunk under a hold mode.  kHoldDeep: a chunk of up to kWindowUnits units is read by a single wave with up to
// 16 loads per lane in flight and stored when the wave's hold is over; units past the end of the segment's
// body are skipped lane by lane, head and tail bytes travel as in CopyChunk.
template <bool kNtLoad, int kStore, int kHold>
__device__ __forceinline__ void CopyChunkHeld(uint64_t src, uint64_t dst, uint64_t len, uint64_t k, uint32_t units, uint64_t t0,
                                              uint32_t ticks, uint32_t lanes)
{
    if (kHold != kHoldDeep) {
        CopyChunk<kNtLoad, kStore, kHold == kHoldShallow>(src, dst, len, k, units, t0, ticks, lanes);
        return;
    }
    const SegGeom g = SegmentGeometry(dst, len);
    const uint64_t u0 = k * kWindowUnits;
    const uint64_t left = g.body > u0 ? g.body - u0 : 0;
    const uint32_t n = left < kWindowUnits ? static_cast<uint32_t>(left) : kWindowUnits;
    const uint32_t tid = threadIdx.x;                       // 64 lanes
    const uint64_t s = src + g.head + u0 * kUnitBytes + tid * kUnitBytes;
    const uint64_t d = dst + g.head + u0 * kUnitBytes + tid * kUnitBytes;
    u32x4 v[kWindowDepth];
    if (n == kWindowUnits) {    // the common case without a test per load: the sixteen loads leave back to back
#pragma unroll
        for (uint32_t j = 0; j < kWindowDepth; ++j) {
            v[j] = LoadUnit<kNtLoad>(s + j * 64 * kUnitBytes);
        }
        HoldStores(t0, ticks);
#pragma unroll
        for (uint32_t j = 0; j < kWindowDepth; ++j) {
            StoreUnit<kStore>(d + j * 64 * kUnitBytes, v[j]);
        }
    } else {
#pragma unroll
        for (uint32_t j = 0; j < kWindowDepth; ++j) {
            if (j * 64 + tid < n) {
                v[j] = LoadUnit<kNtLoad>(s + j * 64 * kUnitBytes);
            }
        }
        HoldStores(t0, ticks);
#pragma unroll
        for (uint32_t j = 0; j < kWindowDepth; ++j) {
            if (j * 64 + tid < n) {
                StoreUnit<kStore>(d + j * 64 * kUnitBytes, v[j]);
            }
        }
    }
    if (k == 0 && tid < g.head) {
        CopyByte<kStore>(src + tid, dst + tid);
    }
    if (u0 + kWindowUnits >= g.body && tid < g.tail) {
        const uint64_t off = g.head + g.body * kUnitBytes + tid;
        CopyByte<kStore>(src + off, dst + off);
    }
}

// A single segment needs no table: its three words travel as plain kernel arguments (28 bytes instead of
// the 3080-byte plan), which is cheaper for the host to hand over and spares every wave the table fetch (one copy behind the
// other, us, against the same bytes as two halves in a table: 8 MiB 3.8 / 5.1, 24 MiB 8.0 / 9.0, 64 MiB 21.2 / 21.5; short ones that
// are waited for take XcopySingleDoneKernel).  From about 200 MiB on the table form is 1 % faster, hence the limit.
// A destination off a line has its chunks cut on the lines (onLines): chunks that begin with the segment end inside lines that two workgroups
// write, each a part.  Back to back, us, chunks of the segment / of the lines: 12 / 16 / 20 / 24 MB 5.7 / 5.0, 6.9 / 6.1, 8.2 / 7.2, 9.5 / 8.3, as long
// as with a destination on a line; where the source differs modulo 16 too 130 / 200 / 400 MB 46.3 / 43.8, 70.1 / 65.9, 138 / 131, so beyond the limit too.
constexpr uint32_t kSingleMaxChunks = 49152;
template <bool kNtLoad, int kStore, int kHold = kHoldNone>
__global__ __launch_bounds__(kXcopyThreads) void XcopySingleKernel(uint64_t src, uint64_t dst, uint32_t len, uint32_t nchunk,
                                                                   uint32_t units, uint32_t holdTicks, uint32_t lanes, uint32_t groups,
                                                                   uint32_t onLines)
{
    const uint64_t t0 = kHold != kHoldNone ? wall_clock64() : 0;
    uint32_t c = blockIdx.x;
    do {
        const SegChunk m = ChunkOn(onLines != 0, src, dst, len, c, units);
        CopyChunkHeld<kNtLoad, kStore, kHold>(m.src, m.dst, m.len, m.k, units, t0, holdTicks, lanes);
        c += groups;
    } while (c < nchunk);
}

// Completion word (of the plugin ABI for tables and words in device memory, and of blocking calls,
// whose host thread polls it).  It is written by a launch of its own right behind the copy
// launch on the same stream: the copy kernel's end-of-kernel release makes every store visible once
// for the whole grid.  (Signalling from inside the copy kernel needs a system-scope release in
// every workgroup before it may count itself done, an L2 write-back each: 77 us instead of 5.5 us
// for an 9 MB batch.)  An empty batch gets the word alone.
__global__ void XcopySignalKernel(uint64_t mask, uint32_t maskValue)
{
    if (threadIdx.x == 0 && blockIdx.x == 0) {
        __hip_atomic_store(Buffer<uint64_t>(mask), static_cast<uint64_t>(maskValue), __ATOMIC_RELEASE, __HIP_MEMORY_SCOPE_SYSTEM);
    }
}

// A short blocking copy that says itself when it is done.  It is bound by the chain of launch, kernel and the word's way to the host;
// a signal launch behind the copy adds a launch to the host's side and a launch boundary to the GPU's.  Blocking calls with the
// signal launch / with this kernel: 16 KiB in HBM 10.5 / 8.4 us, 2 MiB 11.4 / 9.5, 122 blocks of 8 KiB 11.9 / 10.6, 32 x 4 KiB to the
// host 12.2 / 11.0.  Workgroups of 16 KiB (four 128-bit accesses per lane of four waves): every workgroup beyond the first
// costs an atomic, and those on one word wait for each other, so many workgroups count in two steps (4 MiB: 11.5 with all on one
// word, as much as the signal launch, so 9.6); 64 KiB in one workgroup of sixteen waves gain nothing in HBM (8.9 / 8.9) and lose
// over the link (from the host 12.5 / 10.6).
struct DoneMark {
    uint64_t *word;         // pinned host memory, polled by the caller
    uint32_t *counter;      // device memory of kDoneCounterBytes, 0 between launches
    uint32_t value;
    uint32_t groups;        // of the launch
};

// Workgroup `group` of `groups` counts itself in, on its own of kDoneCounters lines where they are many.  Every counter is 0 again when
// the last has come.
__device__ __forceinline__ bool InTwoSteps(uint32_t groups)
{
    return groups > kDoneFewGroups;
}

__device__ __forceinline__ uint32_t ArrivalLimit(uint32_t groups, uint32_t group)
{
    return (InTwoSteps(groups) ? (groups + kDoneCounters - 1 - group % kDoneCounters) / kDoneCounters : groups) - 1;
}

__device__ __forceinline__ uint32_t Arrive(uint32_t *counter, uint32_t groups, uint32_t group)
{
    uint32_t *own = InTwoSteps(groups) ? counter + (1 + group % kDoneCounters) * kDoneCounterWords : counter;
    return atomicInc(own, ArrivalLimit(groups, group));
}

// Whether it was the last of all; `seen` is what Arrive() returned.
__device__ __forceinline__ bool LastArrival(uint32_t *counter, uint32_t groups, uint32_t group, uint32_t seen)
{
    if (seen != ArrivalLimit(groups, group)) {
        return false;
    }
    return !InTwoSteps(groups) || atomicInc(counter, kDoneCounters - 1) == kDoneCounters - 1;
}

// Every store of the launch is written through (kStoreThrough), so it has reached memory once vmcnt says so, and the last
// workgroup to count itself done may tell the host without waiting for the end of the kernel.
__device__ __forceinline__ void MarkDone(const DoneMark &mark, uint32_t group = blockIdx.x)
{
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
    __syncthreads();
    if (threadIdx.x != 0) {
        return;
    }
    if (mark.groups > 1 && !LastArrival(mark.counter, mark.groups, group, Arrive(mark.counter, mark.groups, group))) {
        return;
    }
    __hip_atomic_store(mark.word, static_cast<uint64_t>(mark.value), __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_SYSTEM);
}

// (Arguments one by one: the 56 bytes are in scalar registers when a wave starts, those of a struct are memory it has to read.)
template <bool kNtLoad>
__global__ __launch_bounds__(kXcopyThreads) void XcopySingleDoneKernel(uint64_t src, uint64_t dst, uint32_t len, uint32_t nchunk,
                                                                       uint32_t units, uint32_t lanes, uint64_t word, uint64_t counter,
                                                                       uint32_t value, uint32_t groups)
{
    for (uint32_t c = blockIdx.x; c < nchunk; c += groups) {
        CopyChunk<kNtLoad, kStoreThrough>(src, dst, len, c, units, 0, 0, lanes);
    }
    MarkDone(DoneMark{Buffer<uint64_t>(word), Buffer<uint32_t>(counter), value, groups});
}

template <bool kNtLoad>
__global__ __launch_bounds__(kXcopyThreads) void XcopyInlineDoneKernel(const InlinePlan p, DoneMark mark)
{
    const InlineRows rows(p);
    const uint32_t nchunk = p.nchunk;
    const uint32_t units = p.units;
    uint32_t c = blockIdx.x;
    do {
        const InlineChunk r = rows.Owner(c);
        CopyChunk<kNtLoad, kStoreThrough>(r.src, r.dst, r.len, r.k, units);
        c += mark.groups;
    } while (c < nchunk);
    MarkDone(mark);
}

// The table form: any number of segments, {src, dst, len} triples in memory.  A wave finds the owner of its
// chunk either by a division (chunk counts that repeat: pages of one size, K and V blocks in turn) or
// through the group map: two map entries bound the owner to a short range of segments, whose prefix
// entries AND triples the lanes then fetch side by side, one segment per lane, so that the descriptor is
// in registers two dependent loads after the wave started, whatever the size of the table.  (The form
// this replaces searched the whole prefix 64 ways per round: three rounds for 262 144 segments, then the
// prefix entry, then the triple.)  A wave that walks several chunks fetches what the next lookup starts
// from before it copies the current chunk.
struct ChunkRef {
    uint64_t src;
    uint64_t dst;
    uint64_t len;
    uint32_t k;
};

// Owner of chunk c, known to lie in segments [lo, hiEx): first[lo] <= c < first[hiEx].
__device__ __forceinline__ ChunkRef OwnerOf(const uint64_t *__restrict__ triples, const uint32_t *__restrict__ first, uint32_t lo,
                                            uint32_t hiEx, uint32_t c, uint32_t lane)
{
    // more than 64 candidates (a run of empty segments, or a map with coarse groups): narrow 64 ways per round
    while (hiEx - lo > 64) {
        const uint32_t span = hiEx - lo;
        const uint32_t step = (span + 63u) >> 6;
        const uint32_t probe = lo + (lane + 1) * step;
        const bool inside = probe < hiEx;
        const uint32_t v = inside ? first[probe] : 0xFFFFFFFFu;
        const uint32_t hits = __popcll(__ballot(inside && v <= c));
        lo += hits * step;
        const uint32_t cap = lo + step;
        hiEx = cap < hiEx ? cap : hiEx;
    }
    const uint32_t probe = lo + lane;
    const bool inside = probe < hiEx;
    uint32_t f = 0xFFFFFFFFu;
    uint64_t ts = 0;
    uint64_t td = 0;
    uint64_t tl = 0;
    if (inside) {
        f = first[probe];
        const uint64_t *t = triples + 3ull * probe;
        ts = t[0];
        td = t[1];
        tl = t[2];
    }
    const uint32_t row = __popcll(__ballot(inside && f <= c)) - 1;   // first[lo] <= c: at least one hit
    ChunkRef r;
    r.src = ReadLane64(ts, row);
    r.dst = ReadLane64(td, row);
    r.len = ReadLane64(tl, row);
    r.k = c - __builtin_amdgcn_readlane(f, row);
    return r;
}

// A value every lane holds alike, moved to a scalar register: what a wave loads from a uniform address after its
// first store lands in vector registers, and addresses and lengths computed from it would be computed per lane.
__device__ __forceinline__ uint32_t Uniform(uint32_t v)
{
    return __builtin_amdgcn_readfirstlane(v);
}

__device__ __forceinline__ uint64_t Uniform(uint64_t v)
{
    return (static_cast<uint64_t>(Uniform(static_cast<uint32_t>(v >> 32))) << 32) | Uniform(static_cast<uint32_t>(v));
}

template <bool kNtLoad, int kStore>
__global__ __launch_bounds__(kXcopyThreads) void XcopyTableKernel(const TablePlan plan)
{
    const uint32_t nchunk = plan.nchunk;
    const uint32_t shift = plan.groupShift;
    const ChunkPattern pattern = plan.pattern;
    uint32_t c = blockIdx.x;
    if (c >= nchunk) {
        return;
    }
    const uint32_t units = plan.units;
    if (pattern.period != 0) {
        uint32_t seg;
        uint32_t k;
        PatternOwner(pattern, c, seg, k);
        const uint64_t *t = plan.triples + 3ull * seg;
        uint64_t src = t[0];
        uint64_t dst = t[1];
        uint64_t len = t[2];
        for (;;) {
            const uint32_t next = c + gridDim.x;
            const bool more = next < nchunk;
            uint64_t nsrc = 0;
            uint64_t ndst = 0;
            uint64_t nlen = 0;
            uint32_t nk = 0;
            if (more) {   // requested now, needed after the copy
                PatternOwner(pattern, next, seg, nk);
                t = plan.triples + 3ull * seg;
                nsrc = t[0];
                ndst = t[1];
                nlen = t[2];
            }
            CopyChunk<kNtLoad, kStore>(src, dst, len, k, units);
            if (!more) {
                return;
            }
            src = Uniform(nsrc);
            dst = Uniform(ndst);
            len = Uniform(nlen);
            k = nk;
            c = next;
        }
    }
    const uint32_t lane = threadIdx.x & 63u;
    // even lanes fetch the map entry of the chunk's group, odd lanes the one behind it
    uint32_t bounds = plan.group[(c >> shift) + (lane & 1u)];
    for (;;) {
        const uint32_t lo = __builtin_amdgcn_readlane(bounds, 0);
        const uint32_t hiEx = __builtin_amdgcn_readlane(bounds, 1) + 1;
        const ChunkRef r = OwnerOf(plan.triples, plan.first, lo, hiEx, c, lane);
        const uint32_t next = c + gridDim.x;
        const bool more = next < nchunk;
        if (more) {
            bounds = plan.group[(next >> shift) + (lane & 1u)];
        }
        CopyChunk<kNtLoad, kStore>(r.src, r.dst, r.len, r.k, units);
        if (!more) {
            return;
        }
        c = next;
    }
}

// Units of the destination's cache line in front of a piece's first one.  A piece that counts its units from the line on stores whole
// lines with every instruction; counted from the first unit on, each instruction of a piece that begins inside a line, as a quarter to a
// half of those of ragged segments do, ends in a line that the next one has to complete.  us back to back, counted from the first unit / from
// the line: ragged segments of up to 70 000 bytes 35 / 70 / 95 / 140 MB 14.2 / 13.7, 27.2 / 25.7, 37.8 / 36.1, 55.9 / 53.2, of up to 128 KiB 26 / 66 /
// 262 MB 10.7 / 10.5, 24.7 / 23.7, 101.5 / 98.2; in four waves that hold nothing 287 / 537 MB 119.7 / 117.5, 217.8 / 215.1.
__device__ __forceinline__ uint32_t LeadUnits(uint64_t first, uint32_t body, uint32_t most)
{
    const uint32_t lead = static_cast<uint32_t>(first & (kLineBytes - 1)) / kUnitBytes;
    return lead + body <= most ? lead : 0;
}

// Pieces of up to kLanes * kUnits units (xcopy_plan.h), one per workgroup.  HBM is the bound; what the form saves is everything in
// front of the first load: descriptors are fetched in one step from the host's memory, where a table with a chunk prefix and
// an owner map had to be moved to HBM by a launch of its own first, and no wave looks anything up.
// Shapes, measured on the kernel alone: single waves of 4 KiB as long as those are resident together, for their held stores;
// single waves of 16 KiB, held (XcopyPieceHeldKernel), beyond; and without hold four waves of 16 KiB, or as many as the usual segment fills: 4096 pages of 32 KiB
// gathered 45.8 / 49.4 / 46.4 us with 4 KiB waves / 16 KiB waves / four waves, scattered 49.9 / 51.4 / 49.2, and a quarter of the
// descriptors for the host to write.
// `meanwhile`: what is done while the loads are on their way.
template <uint32_t kLanes, uint32_t kUnits, bool kHold, int kStore, class F>
__device__ __forceinline__ void CopyPiece(const Piece &p, uint64_t t0, uint32_t holdTicks, F meanwhile)
{
    const uint64_t srcWord = Uniform(p.src);
    const uint64_t dstWord = Uniform(p.dst);
    const uint64_t src = srcWord & kPieceAddress;
    const uint64_t dst = dstWord & kPieceAddress;
    const SegGeom g = SegmentGeometry(dst, PieceLength(srcWord, dstWord));
    const uint32_t body = static_cast<uint32_t>(g.body);
    const uint32_t lead = LeadUnits(dst + g.head, body, kLanes * kUnits);
    const uint32_t units = lead + body;
    const uint64_t s = src + g.head - lead * kUnitBytes;
    const uint64_t d = dst + g.head - lead * kUnitBytes;
    const uint32_t tid = threadIdx.x;
    const uint32_t apart = static_cast<uint32_t>(s) & (kUnitBytes - 1);
    u32x4 v[kUnits];
    if (apart == 0 && body == kLanes * kUnits) {
#pragma unroll
        for (uint32_t j = 0; j < kUnits; ++j) {
            v[j] = LoadAligned(s + (j * kLanes + tid) * kUnitBytes);
        }
        meanwhile();
        if (kHold) {
            HoldStores(t0, holdTicks);
        }
#pragma unroll
        for (uint32_t j = 0; j < kUnits; ++j) {
            StoreUnit<kStore>(d + (j * kLanes + tid) * kUnitBytes, v[j]);
        }
    } else if (apart == 0) {
#pragma unroll
        for (uint32_t j = 0; j < kUnits; ++j) {
            if (j * kLanes + tid - lead < body) {
                v[j] = LoadAligned(s + (j * kLanes + tid) * kUnitBytes);
            }
        }
        meanwhile();
        if (kHold) {
            HoldStores(t0, holdTicks);
        }
#pragma unroll
        for (uint32_t j = 0; j < kUnits; ++j) {
            if (j * kLanes + tid - lead < body) {
                StoreUnit<kStore>(d + (j * kLanes + tid) * kUnitBytes, v[j]);
            }
        }
    } else if (body != 0) {
        u32x4 last;
        const uint32_t u0 = (tid >> 6) * kUnits * 64;
        LoadApart(v, last, s - apart, u0, units, lead);
        meanwhile();
        if (kHold) {
            HoldStores(t0, holdTicks);
        }
        StoreApart<kStore>(v, last, d, u0, units, apart, tid & 63u, lead);
    } else {
        meanwhile();
    }
    if (tid < g.head) {
        CopyByte<kStore>(src + tid, dst + tid);
    }
    if (tid < g.tail) {
        const uint64_t off = g.head + g.body * kUnitBytes + tid;
        CopyByte<kStore>(src + off, dst + off);
    }
}

// A launch of a stream starts when those before it have ended, and has then no more use for what they have read: one that is
// told a word in host memory says so there.
__device__ __forceinline__ void MarkStarted(uint64_t started, uint32_t value)
{
    if (started != 0 && blockIdx.x == 0 && threadIdx.x == 0) {
        __hip_atomic_store(Buffer<uint64_t>(started), static_cast<uint64_t>(value), __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_SYSTEM);
    }
}

// By a scalar load, which the compiler makes of a plain read only where it sees that nothing has been written before: a list is not
// written while a launch reads it.  As a vector load, which the loads of the piece wait for, 18 / 36 MB of K and V blocks took
// 8.7 / 14.65 us and not 8.6 / 14.5, 65 MB of blocks on a caller's stream 23.5 and not 23.1.  It has arrived at the return and is not
// read a second time.
__device__ __forceinline__ Piece PieceAt(uint64_t list, uint32_t at)
{
    const auto *p = reinterpret_cast<const __attribute__((address_space(4))) uint64_t *>(list + at * sizeof(Piece));
    uint64_t src = p[0];
    uint64_t dst = p[1];
    asm volatile("" : "+s"(src), "+s"(dst));
    return Piece{src, dst};
}

// `word` gets `value` when the launch starts or, with a counter, when every wave has its piece: the list is the host's again then.
// The counting is done beside the loads.
template <uint32_t kLanes, uint32_t kUnits, bool kHold>
__global__ __launch_bounds__(kLanes) void XcopyPieceKernel(uint64_t list, uint32_t count, uint32_t holdTicks, uint32_t value, uint64_t word,
                                                           uint64_t counter)
{
    const uint64_t t0 = kHold ? wall_clock64() : 0;
    const uint32_t at = PieceOf(blockIdx.x);
    if (at >= count) {
        return;
    }
    if (counter == 0) {
        MarkStarted(word, value);
    }
    const Piece p = PieceAt(list, at);
    // every wave fetches the piece for itself
    constexpr uint32_t kWaves = kLanes / 64;
    const uint32_t waves = count * kWaves;
    const uint32_t wave = at * kWaves + threadIdx.x / 64;
    const bool counts = counter != 0 && threadIdx.x % 64 == 0;
    uint32_t seen = 0;
    if (counts) {
        seen = Arrive(Buffer<uint32_t>(counter), waves, wave);
    }
    CopyPiece<kLanes, kUnits, kHold, kStoreStream>(p, t0, holdTicks, [&] {
        if (counts && LastArrival(Buffer<uint32_t>(counter), waves, wave, seen)) {
            __hip_atomic_store(Buffer<uint64_t>(word), static_cast<uint64_t>(value), __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_SYSTEM);
        }
    });
}

// A piece of up to kUnits * 64 units by one wave that holds all of it, in as few registers as there can be: every access is a
// scalar base and the lane's offset, lanes past the end load the last unit, what lane 63 lacks of the unit behind its last
// one comes by a scalar load, and the lane is hidden from the compiler, which would work all offsets out at the start.
// Units are counted from the cache line that the piece begins in (LeadUnits).
template <uint32_t kUnits, class F>
__device__ __forceinline__ void CopyPieceHeld(uint64_t src, uint64_t dst, uint32_t length, uint64_t t0, uint32_t holdTicks, F meanwhile)
{
    const SegGeom g = SegmentGeometry(dst, length);
    const uint32_t body = static_cast<uint32_t>(g.body);
    const uint32_t lane = threadIdx.x;
    const uint32_t lead = LeadUnits(dst + g.head, body, kUnits * 64);
    const uint32_t units = lead + body;
    const uint64_t d = dst + g.head - lead * kUnitBytes;
    const uint32_t apart = static_cast<uint32_t>(src + g.head) & (kUnitBytes - 1);
    const uint64_t s = src + g.head - apart - lead * kUnitBytes;
    auto hidden = [&] {
        uint32_t l = lane;
        asm volatile("" : "+v"(l));
        return l;
    };
    auto load = [&](uint64_t base, uint32_t unit) {
        return __builtin_nontemporal_load(
            reinterpret_cast<const MF_GLOBAL u32x4 *>(reinterpret_cast<const MF_GLOBAL uint8_t *>(base) + unit * kUnitBytes));
    };
    auto store = [&](uint32_t j, uint32_t unit, u32x4 v) {
        __builtin_nontemporal_store(
            v, reinterpret_cast<MF_GLOBAL u32x4 *>(reinterpret_cast<MF_GLOBAL uint8_t *>(d + j * 64 * kUnitBytes) + unit * kUnitBytes));
    };
    auto hold = [&] {       // `meanwhile` once the loads have landed: what it needs meets no address or load of theirs
        asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
        meanwhile();
        HoldStores(t0, holdTicks);
    };
    u32x4 v[kUnits];
    if (body == 0) {
        meanwhile();
    } else if (apart == 0 && body == kUnits * 64) {
#pragma unroll
        for (uint32_t j = 0; j < kUnits; ++j) {
            v[j] = load(s + j * 64 * kUnitBytes, lane);
        }
        hold();
#pragma unroll
        for (uint32_t j = 0; j < kUnits; ++j) {
            store(j, lane, v[j]);
        }
    } else {
        const uint32_t end = apart != 0 ? units : units - 1;      // the last unit that holds any of the bytes
        const uint32_t behind = kUnits * 64 < end ? kUnits * 64 : end;
        const auto *lacks = reinterpret_cast<const __attribute__((address_space(4))) uint32_t *>(s + behind * kUnitBytes);
        uint32_t last[4] = {lacks[0], lacks[1], lacks[2], lacks[3]};
#pragma unroll
        for (uint32_t j = 0; j < kUnits; ++j) {
            if (j * 64 <= end) {
                const uint32_t u = j * 64 + hidden();
                const uint32_t upTo = u < end ? u : end;
                v[j] = load(s, j == 0 && upTo < lead ? lead : upTo);
            }
        }
        asm volatile("" : "+s"(last[0]), "+s"(last[1]), "+s"(last[2]), "+s"(last[3]));
        hold();
        if (apart == 0) {
#pragma unroll
            for (uint32_t j = 0; j < kUnits; ++j) {
                const uint32_t l = hidden();
                if (j * 64 + l - lead < body) {
                    store(j, l, v[j]);
                }
            }
        } else {
            auto shifted = [&](auto words) {
#pragma unroll
                for (uint32_t j = 0; j < kUnits; ++j) {
                    u32x4 next;
#pragma unroll
                    for (uint32_t i = 0; i < 4; ++i) {
                        const uint32_t wrap = j + 1 < kUnits ? __builtin_amdgcn_readfirstlane(v[j + 1 < kUnits ? j + 1 : 0][i]) : last[i];
                        next[i] = NextLane(v[j][i], wrap);
                    }
                    const u32x4 r = Straddle<decltype(words)::value>(v[j], next, apart & 3u);
                    const uint32_t l = hidden();
                    if (j * 64 + l - lead < body) {
                        store(j, l, r);
                    }
                }
            };
            switch (apart >> 2) {
                case 0: shifted(std::integral_constant<uint32_t, 0>()); break;
                case 1: shifted(std::integral_constant<uint32_t, 1>()); break;
                case 2: shifted(std::integral_constant<uint32_t, 2>()); break;
                default: shifted(std::integral_constant<uint32_t, 3>()); break;
            }
        }
    }
    if (lane < g.head) {
        CopyByte<kStoreStream>(src + lane, dst + lane);
    }
    if (lane < g.tail) {
        const uint64_t off = g.head + g.body * kUnitBytes + lane;
        CopyByte<kStoreStream>(src + off, dst + off);
    }
}

// Waves of 16 KiB that hold their stores: 72 registers, 28 waves per CU, so kHeldMaxPieces (112 MiB, most of the chip's registers) are
// resident and the launch reads all of the batch before it writes any of it.  HBM is the bound.  XcopyPieceKernel's form of sixteen
// units has 100 registers, 4096 waves.  us back to back, without hold (4 KiB a wave or four waves of them, the better) / in windows cut for 6.0
// or 6.4 TB/s, the better / XcopyPieceKernel<64, 16, true> / so.  Pages of 32 KiB scattered 28 MB 12.9 / - / 10.8 / 10.8, 72 MB 29.5 / 26.7 / - / 25.7,
// 88 MB 35.5 / 32.0 / - / 31.2, 104 MB 41.8 / 37.4 / - / 37.0, gathered 56 MB 21.7 / - / 19.7 / 18.9, 104 MB 38.0 / 35.1 / - / 33.9.  Ragged segments of
// up to 70 000 bytes, 8 MB 6.8 / - / 6.3 / 5.9, 22 MB 12.0 / - / 10.5 / 9.9, 55 MB 25.2 / - / - / 22.1, 74 MB 32.1 / - / - / 28.4, 89 MB 38.0 / - / - / 34.1;
// of up to 8000, 28 MB 15.3 / - / - / 14.0; of up to 16 000, 57 MB 26.6 / - / - / 25.2.  What is short of full is skipped unit by unit by the whole
// wave: lanes that loaded the last unit over and over cost 50 MB in segments of 50 688 bytes 20.3, so 18.2.
// Not taken: 12 KiB in eight waves per SIMD or 20 and 24 KiB in five and four, within 2 %; units beyond the registers kept in LDS (28 and 4 KiB
// in four waves per SIMD, 4096 pages of 32 KiB 44.5, two launches of 4096 waves 45.2).
constexpr uint32_t kHeldWavesPerSimd = 7;
__global__ __launch_bounds__(64) __attribute__((amdgpu_waves_per_eu(kHeldWavesPerSimd, kHeldWavesPerSimd))) void XcopyPieceHeldKernel(
    uint64_t list, uint32_t count, uint32_t holdTicks, uint32_t value, uint64_t word, uint64_t counter)
{
    const uint64_t t0 = wall_clock64();
    const uint32_t at = PieceOf(blockIdx.x);
    if (at >= count) {
        return;
    }
    if (counter == 0) {
        MarkStarted(word, value);
    }
    const Piece p = PieceAt(list, at);
    CopyPieceHeld<kDeepUnits / 64>(p.src & kPieceAddress, p.dst & kPieceAddress, PieceLength(p.src, p.dst), t0, holdTicks, [&] {
        if (counter != 0 && threadIdx.x == 0 &&
            LastArrival(Buffer<uint32_t>(counter), count, at, Arrive(Buffer<uint32_t>(counter), count, at))) {
            __hip_atomic_store(Buffer<uint64_t>(word), static_cast<uint64_t>(value), __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_SYSTEM);
        }
    });
}

// A single segment in chunks of LineChunks(), one a wave of the kernel above without a list.  HBM bounds it.  us back to back, from 16 KiB in
// 100 registers up to 64 MiB and 4 KiB without hold beyond, the chunks the segment's / so: 32 MB 10.9 / 10.3, 48 16.3 / 15.4, 66 20.9 / 20.6, 90
// 29.9 / 28.4, 110 36.2 / 34.0; destination off a line by 48 bytes 12.1 / 10.4, 18.1 / 15.7, 23.8 / 20.6, 31.7 / 28.8, 38.4 / 34.3; source and destination
// different modulo 16, before from a list of pieces up to 64 MiB, 11.9 / 10.9, 17.0 / 15.7, 22.9 / 21.0, 32.9 / 29.4, 40.0 / 35.2.  Beside a kernel of another
// stream that holds half the CUs 63 MB 27.8 / 24.1, 72 28.7 / 26.6, 110 42.0 / 45.0; 32 of 72 MB beside eight elementwise kernels over 1 GiB, both together
// 2151 / 2237.
__global__ __launch_bounds__(64) __attribute__((amdgpu_waves_per_eu(kHeldWavesPerSimd, kHeldWavesPerSimd))) void XcopySingleHeldKernel(
    uint64_t src, uint64_t dst, uint32_t len, uint32_t holdTicks)
{
    const uint64_t t0 = wall_clock64();
    const LineSpan span = LineChunk(dst, len, blockIdx.x, kDeepUnits);
    if (span.begin < len) {
        CopyPieceHeld<kDeepUnits / 64>(src + span.begin, dst + span.begin, static_cast<uint32_t>(span.end - span.begin), t0, holdTicks, [] {});
    }
}

// The rows of an InlinePlan in LDS, for waves that look them up again and again: held in registers, as InlineRows does, they would take the
// place of a wave.
struct SharedRows {
    uint64_t src[kInlineSegs];
    uint64_t dst[kInlineSegs];
    uint32_t len[kInlineSegs];
    uint32_t first[kInlineSegs];

    // by a workgroup of one wave
    __device__ __forceinline__ void Keep(const InlineRows &r)
    {
        const uint32_t lane = threadIdx.x;
        src[lane] = r.s0;
        src[lane + 64] = r.s1;
        dst[lane] = r.d0;
        dst[lane + 64] = r.d1;
        len[lane] = r.l0;
        len[lane + 64] = r.l1;
        first[lane] = r.f0;
        first[lane + 64] = r.f1;
        __syncthreads();
    }
    __device__ __forceinline__ InlineChunk Owner(uint32_t c) const
    {
        uint32_t lane = threadIdx.x;
        asm volatile("" : "+v"(lane));      // read anew in every round
        const uint32_t s = __popcll(__ballot(first[lane] <= c)) + __popcll(__ballot(first[lane + 64] <= c)) - 1;
        return InlineChunk{Uniform(src[s]), Uniform(dst[s]), Uniform(len[s]), c - Uniform(first[s])};
    }
};

// The inline plan in chunks of LineChunks(), whatever source and destination are modulo 16, in windows: single-wave workgroups walk the
// chunks with stride gridDim.x, one per period each, as XcopyPieceHeldKernel copies a piece, so that a chunk that is not whole, or whose
// bytes are shifted, keeps to the windows too.  HBM is the bound.  us back to back, the mean of two processes, 4096 waves that keep the
// table in registers and are cut for 7.1 TB/s (one segment on lines 7.4, shifted 6.8) / this, cut for 7.3 (7.375, 7.0):
//   one segment on lines   136 MB 42.6 / 40.7, 370 MB 107.6 / 104.9, 512 MiB 154 / 151, 900 MB 281 / 254, 1 GiB 310 / 302
//   off a line             300 MB 93.1 / 86.0, 700 MB 213 / 198, 1 GiB 323 / 303
//   shifted                200 MB 65.7 / 61.2
//   128 segments           of 2.4 MB 96.9 / 88.8, of 9 MB 338 / 327
//   reshards with their rectangles   13 layers of 1280 548 / 533, 28 of 3584 3873 / 3831
// Beside elementwise kernels of another stream over 1 GiB, both together, 18 of 512 MiB 6333 / 6341, 31 of 128 x 2.4 MB 6485 / 6337; over
// 256 MB 13 of 512 MiB 4358 / 4288, 46 of 128 x 1 MB 3842 / 4048, 20 shifted of 300 MB 3700 / 3863; beside products of matrices the
// same three 3643 / 3658, 3704 / 3466, 3513 / 3450.
__global__ __launch_bounds__(64) __attribute__((amdgpu_waves_per_eu(kLongWavesPerSimd, kLongWavesPerSimd))) void XcopyWindowKernel(
    const InlinePlan p, uint32_t period, uint32_t seq)
{
    __shared__ SharedRows rows;
    const InlineRows fetched(p);            // on their way while the start is agreed
    const uint32_t nchunk = p.nchunk;
    const uint32_t groups = gridDim.x;
    const uint32_t half = period / 2;
    uint64_t slot = AgreedStart(seq) + static_cast<uint64_t>(blockIdx.x) * half / groups;
    rows.Keep(fetched);
    for (uint32_t c = blockIdx.x; c < nchunk; c += groups, slot += period) {
        const InlineChunk r = rows.Owner(c);
        const LineSpan span = LineChunk(r.dst, r.len, r.k, kDeepUnits);
        WaitForClock(slot);
        CopyPieceHeld<kDeepUnits / 64>(r.src + span.begin, r.dst + span.begin, static_cast<uint32_t>(span.end - span.begin), slot, half, [] {});
    }
}

// A short blocking batch that says itself when it is done, as XcopySingleDoneKernel.  A blocking call with the signal launch / so, us:
// 129 / 200 / 500 segments of 5000 bytes 14.0 / 15.2 / 19.7 and 12.5 / 13.4 / 17.0, 244 K and V blocks of 16 KiB 18.1 and 16.1, 200 of 16 000
// bytes 17.0 and 13.8, 1000 ragged ones of up to 5000 bytes 23.6 and 22.8; 4000 of 2000 bytes 52.6 and 53.3, so not that many.
__global__ __launch_bounds__(64) void XcopyPieceDoneKernel(uint64_t list, uint32_t count, uint64_t word, uint64_t counter, uint32_t value)
{
    const uint32_t at = PieceOf(blockIdx.x);
    if (at >= count) {
        return;
    }
    CopyPiece<64, kDepth, false, kStoreThrough>(PieceAt(list, at), 0, 0, [] {});
    MarkDone(DoneMark{Buffer<uint64_t>(word), Buffer<uint32_t>(counter), value, count}, at);
}

// Pieces of kWindowUnits units in read and write windows, as XcopyWindowKernel walks chunks, each copied as XcopyPieceHeldKernel copies it,
// whatever its addresses.  A wave fetches a descriptor across the link when it has issued its stores and has half a period for it.  Bound: HBM, whose rows a random place opens for 256 bytes a channel, so the rate that
// holds is lower than that of long segments.  us back to back, held launches or 4096 waves at the rates those held / 6144 waves at
// theirs (PieceWindowRate), two processes each:
//   gathered    pages of 32 KiB, 4096 49.3 / 44.7, 16 384 185 / 171; 16 384 of 16 KiB 95.0 / 87.0; 12 000 of 20 KiB 85.7 / 80.5
//   scattered   pages of 32 KiB, 4096 48.7 / 47.1, 16 384 186 / 180; 16 384 of 16 KiB 95.8 / 93.0; 12 000 of 64 KiB 255 / 245
//   at random places on both sides   8000 of 50 048 bytes 158 / 142, 3500 of 81 920 100.0 / 95.5, 6000 of 110 720 230 / 218,
//               16 384 of 32 KiB 213 / 190, K and V blocks of 128 and 16 KiB, 72 MB, 53.0 / 50.6; 3800 of 28 032 39.9 / 40.6
// Beside elementwise kernels of another stream over 1 GiB, both together, 37 x 8000 pages of 32 KiB 6159 / 6231; over 256 MB 44 x 4096
// scattered 3942 / 4006, gathered 3980 / 3941, 22 x 8000 gathered 3728 / 3867; beside products of matrices 3738 / 3680, 3600 / 3583,
// 3555 / 3465.
// (A schedule that stretches when sampled waves fall behind it was tried: it overshoots, 20 to 50 % slower than none.)
__global__ __launch_bounds__(64) __attribute__((amdgpu_waves_per_eu(kLongWavesPerSimd, kLongWavesPerSimd))) void XcopyPieceWindowKernel(
    uint64_t list, uint32_t count, uint32_t period, uint32_t reading, uint32_t seq, uint32_t groups, uint32_t value, uint64_t started)
{
    MarkStarted(started, value);
    uint64_t slot = AgreedStart(seq) + static_cast<uint64_t>(blockIdx.x) * reading / groups;
    const uint32_t hold = reading + static_cast<uint32_t>(static_cast<uint64_t>(blockIdx.x) * (period - reading) / groups) -
                          static_cast<uint32_t>(static_cast<uint64_t>(blockIdx.x) * reading / groups);
    for (uint32_t at = PieceOf(blockIdx.x); at < count; at += groups, slot += period) {
        const Piece p = PieceAt(list, at);
        WaitForClock(slot);
        CopyPieceHeld<kDeepUnits / 64>(p.src & kPieceAddress, p.dst & kPieceAddress, PieceLength(p.src, p.dst), slot, hold, [] {});
    }
}

// How a launch of a device table paces itself; 0: not.
struct TablePace {
    uint32_t holdTicks;         // of the clock, what a wave waits before it stores, where all waves of the launch are resident together,
    uint32_t holdMoreTicks;     // and what more per 64 MiB of the table;
    uint32_t equalTicks;        // the same where its segments are of one length, whose descriptors are there sooner
    uint32_t equalMoreTicks;
    uint32_t windowTicks;       // period in which 64 MiB pass at the rate of random blocks,
    uint32_t shortTicks;        // of such of one length below kWindowLongBlockBytes, whose write part is the longer one,
    uint32_t longTicks;         // of such of one length from there on,
    uint32_t orderedTicks;      // and of blocks of one length that are written one behind the other
    uint32_t seq;               // of AgreedStart
};

// The windows that a table of segments of length len0 holds, by 64 segments of it, one a lane: whether they are written, or read, one behind the other, and
// whether they all lie on multiples of kWindowLongBlockBytes.  `loose`: its chunks of 16 KiB are so short that it holds a higher rate anywhere.  (With all lanes: what
// one that is switched off holds is not defined.)
struct TableWindows {
    uint32_t ticks;             // period in which 64 MiB pass
    uint32_t reading;           // 64ths of it that are the read part
};
__device__ __forceinline__ TableWindows WindowsOf(const TablePace &pace, uint32_t from, uint32_t to, uint64_t len0, uint32_t sample, bool loose)
{
    const uint32_t lane = threadIdx.x & 63u;
    const uint32_t length = static_cast<uint32_t>(len0);
    const bool pair = lane + 1 < sample;
    const uint32_t behind = __shfl_down(to, 1, 64);
    const uint32_t ahead = __shfl_down(from, 1, 64);
    const bool inOrder = __popcll(__ballot(pair && behind - to == length)) * 4 >= static_cast<int>(sample - 1) * 3;
    const bool readInOrder = __popcll(__ballot(pair && ahead - from == length)) * 4 >= static_cast<int>(sample - 1) * 3;
    const bool onGrid = __ballot(((from | to | length) & (kWindowLongBlockBytes - 1)) != 0) == 0;
    const bool faster = !inOrder && (readInOrder || onGrid || (len0 >= kWindowLongBlockBytes && loose));
    const bool shortPages = faster && len0 < kWindowLongBlockBytes;
    return TableWindows{inOrder ? pace.orderedTicks : !faster ? pace.windowTicks : shortPages ? pace.shortTicks : pace.longTicks, shortPages ? 29u : 32u};
}

__device__ __forceinline__ void ListRest(RestList *rest, uint32_t capacity, uint64_t src, uint64_t dst, uint64_t left)
{
    if (threadIdx.x == 0) {
        const uint64_t taken = __hip_atomic_fetch_add(&rest->taken, kRestEntry + RestPieces(left), __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        if (taken / kRestEntry < capacity) {   // which nseg is not more than: calls that share a list against the rules stay inside it
            rest->entry[taken / kRestEntry] = RestSegment{taken % kRestEntry, src, dst, left};
        }
    }
}

// What the first kDirectSample segments of a table say of it, and, kAcross, as many that lie across it.
struct DirectSample {
    uint32_t parts;             // chunks of the longest of the first, up to kDirectMaxParts
    bool equal;                 // all have one length, `length`,
    uint64_t length;
    bool aligned;               // and lie on units, sources and destinations
};
// Of 2^32, the golden section: its multiples lie evenly, and not with the period of a table of layers or of powers of two.
constexpr uint32_t kAcrossStep = 0x9E3779B9u;
template <bool kAcross>
__device__ __forceinline__ DirectSample SampleOf(const uint64_t *__restrict__ triples, uint32_t nseg, uint32_t units)
{
    const uint32_t lane = threadIdx.x & 63u;
    const uint32_t across = kAcross ? __umulhi(nseg, (lane % kDirectSample + 1) * kAcrossStep) : 0;
    const uint32_t row = lane < kDirectSample && lane < nseg ? lane : across;
    const uint64_t src = triples[3ull * row];
    const uint64_t dst = triples[3ull * row + 1];
    const uint64_t len = triples[3ull * row + 2];
    const uint64_t sampled = SegmentChunks(dst, len, units);
    uint32_t parts = 1;
    uint32_t least = kDirectMaxParts;
#pragma unroll
    for (uint32_t i = 0; i < kDirectSample; ++i) {
        const uint32_t chunks = __builtin_amdgcn_readlane(sampled < kDirectMaxParts ? static_cast<uint32_t>(sampled) : kDirectMaxParts, i);
        parts = chunks > parts ? chunks : parts;
        least = chunks < least ? chunks : least;
    }
    parts |= least == parts ? 0u : 1u;      // odd in a ragged table: every XCD gets each of them in turn
    const uint64_t length = Uniform(len);
    return DirectSample{parts, __ballot(len != length) == 0, length, __ballot(((src | dst | len) & (kUnitBytes - 1)) != 0) == 0};
}

// A table that only the GPU can read, copied as xcopy_plan.h says: item (segment, part), parts in a row.  The launch is sized from
// the segment count alone, so a workgroup walks the items with the grid as its stride; it fetches the next item's triple before
// it copies the current item.  What bounds it is HBM; a launch in front of it that planned the table (chunk prefix, owner map,
// repeating pattern) took 8 us, after which the copy was no faster: 4096 pages of 32 KiB scattered 60.0 / 52.8 us with the
// planner / so, 16 080 pages of 8 KiB 76.7 / 57.9, 100 pages 10.0 / 7.1.
// A ragged table has an odd number of parts: workgroups go to the eight XCDs in turn, and with an even number the first parts,
// which every segment has, went to some and the last, which few have, to others.  In the slower / faster of the two modes that
// the place of a pool decides, us with the planner, with an even number and so: 16 384 segments of 2 to 14 KB 87.1 / 77.5, 79.4 / 74.1,
// 66 / 57.5; 4000 K and V blocks 139.4 / 138.1, 160 / 160, 135.5 / 135.5; 2000 of up to 70 KB 43.4 / 38.7, 40.2 / 35.4, 39.3 / 34.6 and spread over
// 48 GiB 45.4 / 40.4, 50.5 / 46.3, 41.4 / 36.5.  16 384 of up to 262 KB are none the faster for it: 949 / 778, 967 / 774, 967 / 773.
// Not taken: eight workgroups per segment, 1 to 7 % faster where segments have dozens of chunks, 16 080 pages of 8 KiB 24 % slower;
// part numbers that turn from segment to segment, pages 1 % slower; the triples of 64 items at a time, one per lane, so that
// empty items cost no wait, more registers than eight waves per SIMD have, 10 to 60 % slower on short tables; two triples ahead
// instead of one, 16 384 segments of 2 to 14 KB 4 % slower.
template <bool kNtLoad, int kStore>
__device__ __forceinline__ void CopyDirect(const uint64_t *__restrict__ triples, uint32_t nseg, uint32_t units, RestList *__restrict__ rest,
                                           uint32_t capacity, uint32_t parts)
{
    uint32_t seg = blockIdx.x / parts;
    uint32_t part = blockIdx.x - seg * parts;
    if (seg >= nseg) {
        return;
    }
    const uint32_t segStep = gridDim.x / parts;
    const uint32_t partStep = gridDim.x - segStep * parts;
    const uint64_t own = static_cast<uint64_t>(parts) * kDirectRounds;     // chunks of a segment that are copied here
    uint64_t src = triples[3ull * seg];
    uint64_t dst = triples[3ull * seg + 1];
    uint64_t len = triples[3ull * seg + 2];
    for (;;) {
        const uint32_t carry = part + partStep >= parts ? 1 : 0;
        const uint64_t next = static_cast<uint64_t>(seg) + segStep + carry;
        const bool more = next < nseg;
        const uint64_t *t = triples + 3 * (more ? next : seg);             // requested now, needed after the copy
        const uint64_t nsrc = t[0];
        const uint64_t ndst = t[1];
        const uint64_t nlen = t[2];
        const uint64_t chunks = SegmentChunks(dst, len, units);
        for (uint64_t c = part; c < chunks && c < own; c += parts) {
            CopyChunk<kNtLoad, kStore>(src, dst, len, c, units);
        }
        if (part == 0 && chunks > own) {
            const uint64_t at = SegmentGeometry(dst, len).head + own * units * kUnitBytes;
            ListRest(rest, capacity, src + at, dst + at, len - at);
        }
        if (!more) {
            return;
        }
        seg = static_cast<uint32_t>(next);
        part = part + partStep - (carry != 0 ? parts : 0);
        src = Uniform(nsrc);
        dst = Uniform(ndst);
        len = Uniform(nlen);
    }
}

template <bool kNtLoad, int kStore>
__global__ __launch_bounds__(kXcopyThreads) void XcopyDirectKernel(const uint64_t *__restrict__ triples, uint32_t nseg, uint32_t units,
                                                                   RestList *__restrict__ rest, uint32_t capacity)
{
    CopyDirect<kNtLoad, kStore>(triples, nseg, units, rest, capacity, SampleOf<false>(triples, nseg, units).parts);
}

// kWindowUnits units on units, of kParts places, loads and stores by the clock.
template <uint32_t kParts>
__device__ __forceinline__ void CopyWholeWindowed(const uint64_t (&src)[kParts], const uint64_t (&dst)[kParts], uint64_t loadAt, uint64_t storeAt)
{
    constexpr uint32_t kEach = kWindowDepth / kParts;
    const uint32_t lane = threadIdx.x * kUnitBytes;     // beside a scalar base in every access
    u32x4 v[kWindowDepth];
    WaitForClock(loadAt);
#pragma unroll
    for (uint32_t j = 0; j < kWindowDepth; ++j) {
        const uint64_t at = src[j / kEach] + j % kEach * 64 * kUnitBytes;
        v[j] = __builtin_nontemporal_load(reinterpret_cast<const MF_GLOBAL u32x4 *>(reinterpret_cast<const MF_GLOBAL uint8_t *>(at) + lane));
    }
    asm volatile("s_waitcnt vmcnt(0)" : : : "memory");
    WaitForClock(storeAt);
#pragma unroll
    for (uint32_t j = 0; j < kWindowDepth; ++j) {
        const uint64_t at = dst[j / kEach] + j % kEach * 64 * kUnitBytes;
        __builtin_nontemporal_store(v[j], reinterpret_cast<MF_GLOBAL u32x4 *>(reinterpret_cast<MF_GLOBAL uint8_t *>(at) + lane));
    }
}

// The same of four places on units, `bytes` of each, up to a quarter of kWindowUnits units.
__device__ __forceinline__ void CopyPartWindowed(const uint64_t (&src)[4], const uint64_t (&dst)[4], const uint32_t (&bytes)[4], uint64_t loadAt,
                                                 uint64_t storeAt)
{
    constexpr uint32_t kEach = kWindowDepth / 4;
    const uint32_t lane = threadIdx.x * kUnitBytes;
    u32x4 v[kWindowDepth];
    WaitForClock(loadAt);
#pragma unroll
    for (uint32_t j = 0; j < kWindowDepth; ++j) {
        const uint64_t at = src[j / kEach] + j % kEach * 64 * kUnitBytes;
        if (lane + j % kEach * 64 * kUnitBytes < bytes[j / kEach] / kUnitBytes * kUnitBytes) {
            v[j] = __builtin_nontemporal_load(reinterpret_cast<const MF_GLOBAL u32x4 *>(reinterpret_cast<const MF_GLOBAL uint8_t *>(at) + lane));
        }
    }
    asm volatile("s_waitcnt vmcnt(0)" : : : "memory");
    WaitForClock(storeAt);
#pragma unroll
    for (uint32_t j = 0; j < kWindowDepth; ++j) {
        const uint64_t at = dst[j / kEach] + j % kEach * 64 * kUnitBytes;
        if (lane + j % kEach * 64 * kUnitBytes < bytes[j / kEach] / kUnitBytes * kUnitBytes) {
            __builtin_nontemporal_store(v[j], reinterpret_cast<MF_GLOBAL u32x4 *>(reinterpret_cast<MF_GLOBAL uint8_t *>(at) + lane));
        }
    }
#pragma unroll
    for (uint32_t q = 0; q < 4; ++q) {
        if (threadIdx.x < bytes[q] % kUnitBytes) {
            const uint64_t at = bytes[q] / kUnitBytes * kUnitBytes + threadIdx.x;
            CopyByte<kStoreStream>(src[q] + at, dst[q] + at);
        }
    }
}

// XcopyDirectKernel for tables of more than kPlannedSegments between HBM addresses, one wave a workgroup.  Where the sampled segments are
// pages of one length, whole chunks of 16 KiB or a half or a quarter of one, and lie on units, the first waves copy all of the table in
// windows as those of XcopyPlannedKernel do, by the rates that it has measured, and the others leave.  HBM is the bound; without windows
// it sees reads and writes mixed.  us without / so:
//               gathered                                           scattered
//      4 KiB    16 384 35.3 / 25.8; 6140 14.8 / 12.9; 5000 12.6     16 384 38.2 / 30.8; 6140 15.3 / 14.2; 5000 12.7
//               / 12.6; 4400 11.6 / 12.5                            / 12.6; 4400 11.6 / 12.1
//      8 KiB    16 384 54.4 / 45.8; 5000 19.6 / 17.9               16 384 63.3 / 57.7, 60 000 226 / 201; 5000 20.8 / 19.9
//     16 KiB    16 384 95.0 / 86.1; 9000 54.6 / 49.7               16 384 110 / 106; 9000 61.8 / 57.8
//     32 KiB    16 384 188 / 167; 9000 105.6 / 94.0                16 384 217 / 216; 9000 121 / 115
//     64 KiB    9000 212 / 182                                     9000 241 / 238
//
// A page that is unlike those sampled takes its slot if it is shorter and lies on units, else it is listed for the second launch.
// Listing costs 11 ns of one word that all XCDs count on, so tables with many such pages are not for this: that is what the segments
// across the table are looked at for.  All listed / by CopyDirect(): 8192 pages of 16 KiB with all sources off units 204 / 52.8, 4096 of
// 8 KiB and then 4096 of 32 KiB 118 / 66.2, of 16 and 128 KiB 278 / 243; 16 384 of 8 KiB with 5 % shorter 72.2 listed, 52.6 in their slots.
// Pages as sampled are copied in loops of their own, which are left for one that is not: in one loop with its code 16 384 scattered pages
// of 8 KiB take 58.3 and not 57.7, 9000 of 32 KiB 117 and not 116.
//
// Every other table pays for the look and for six waves per SIMD where XcopyDirectKernel has eight, and gains by a smaller grid
// (SubmitDeviceTable): 16 384 segments of 2 to 14 KB 57.3 / 58.6, at odd addresses 63.7 / 63.7, of 2 KiB 25.4 / 23.0, 100 000 142 / 88,
// 8000 of 64 KiB and 8000 of 100 bytes 214.5 / 217.5.
//
// Not taken: 64 segments looked at by every wave (16 384 of 2 to 14 KB 85.8); CopyDirect()'s code for an unlike page where it is met (1 % of
// 16 384 of 16 KiB, 95.9, 131: it is in no instruction cache by then); a second, longer look by the waves that stay (ones of 6144 copy
// what is left 4 to 18 % slower than all would); the look by scalar loads (sixteen rows take more scalar registers than there are); the
// stores of up to 5120 waves held instead (8000 of 8 KiB 28.2 / 29.5); pages that are no whole chunks, whose code would cost the registers.
constexpr uint32_t kSampledWavesPerSimd = 6;
__global__ __launch_bounds__(64) __attribute__((amdgpu_waves_per_eu(kSampledWavesPerSimd, kSampledWavesPerSimd))) void XcopySampledKernel(
    uint64_t table, uint32_t nseg, uint64_t list, uint32_t capacity, TablePace pace)
{
    if (nseg == 0) {
        return;
    }
    const uint64_t *const triples = Buffer<const uint64_t>(table);
    RestList *const rest = Buffer<RestList>(list);
    constexpr uint32_t kDeepBytes = kWindowUnits * kUnitBytes;
    const DirectSample seen = SampleOf<true>(triples, nseg, kXcopyThreads);
    const uint64_t len0 = seen.length;
    const uint32_t together = len0 == kDeepBytes / 2 ? 2 : len0 == kDeepBytes / 4 ? 4 : 1;    // segments a wave
    const uint32_t each = together != 1 ? 1 : len0 % kDeepBytes == 0 && len0 <= kSampledMostBytes ? static_cast<uint32_t>(len0) / kDeepBytes : 0;
    if (!seen.equal || !seen.aligned || each == 0) {
        CopyDirect<true, kStoreStream>(triples, nseg, kXcopyThreads, rest, capacity, seen.parts);
        return;
    }
    auto asSeen = [&](const uint64_t (&row)[3]) { return row[2] == len0 && ((row[0] | row[1]) & (kUnitBytes - 1)) == 0; };
    // by scalar loads: a table is not written while a launch reads it
    const auto *const rows = reinterpret_cast<const __attribute__((address_space(4))) uint64_t *>(table);
    const uint32_t items = (nseg + together - 1) / together * each;
    const uint32_t rounds = (items + kLongWaves - 1) / kLongWaves;
    const uint32_t waves = (items + rounds - 1) / rounds;
    uint32_t item = blockIdx.x;
    if (item >= waves) {
        return;
    }
    const uint64_t *t = triples + 3ull * threadIdx.x;           // more than kPlannedSegments: a row for every lane
    const TableWindows w = WindowsOf(pace, static_cast<uint32_t>(t[0]), static_cast<uint32_t>(t[1]), len0, 64, false);
    const uint32_t period = static_cast<uint32_t>(static_cast<uint64_t>(w.ticks) * (waves * kDeepBytes) >> 26);
    const uint32_t reading = w.reading == 32 ? period / 2 : period / 64 * w.reading;
    const uint64_t start = Uniform(AgreedStart(pace.seq));
    uint64_t loadAt = start + static_cast<uint64_t>(item) * reading / waves;
    uint64_t storeAt = start + reading + static_cast<uint64_t>(item) * (period - reading) / waves;
    // To this wave's next item; false where it has none.
    auto onward = [&] {
        const bool more = items - item > waves;
        item += more ? waves : 0;
        loadAt += period;
        storeAt += period;
        return more;
    };
    // Copies items as seen, up to the first that is not; false: no item is left.
    auto several = [&](auto count) {
        constexpr uint32_t kParts = decltype(count)::value;
        do {
            uint64_t src[kParts];
            uint64_t dst[kParts];
            bool all = true;
#pragma unroll
            for (uint32_t j = 0; j < kParts; ++j) {
                const uint32_t at = item * kParts + j < nseg ? item * kParts + j : nseg - 1;       // the last again rather than none
                const uint64_t row[3] = {rows[3ull * at], rows[3ull * at + 1], rows[3ull * at + 2]};
                src[j] = row[0];
                dst[j] = row[1];
                all = all && asSeen(row);
            }
            if (!all) {
                return true;
            }
            CopyWholeWindowed<kParts>(src, dst, loadAt, storeAt);
        } while (onward());
        return false;
    };
    auto one = [&] {
        uint32_t seg = item / each;
        uint64_t row[3] = {rows[3ull * seg], rows[3ull * seg + 1], rows[3ull * seg + 2]};
        for (;;) {
            const uint32_t k = item - seg * each;
            seg = items - item > waves ? (item + waves) / each : seg;
            const uint64_t next[3] = {rows[3ull * seg], rows[3ull * seg + 1], rows[3ull * seg + 2]};      // requested now, needed after the copy
            if (!asSeen(row)) {
                return true;
            }
            CopyWholeWindowed<1>({row[0] + k * kDeepBytes}, {row[1] + k * kDeepBytes}, loadAt, storeAt);
            if (!onward()) {
                return false;
            }
            row[0] = next[0];
            row[1] = next[1];
            row[2] = next[2];
        }
    };
    do {
        const bool unlike = together == 1 ? one() : together == 2 ? several(std::integral_constant<uint32_t, 2>()) : several(std::integral_constant<uint32_t, 4>());
        if (!unlike) {
            return;
        }
        // a quarter of 16 KiB at a time
        const uint32_t first = together == 1 ? item / each : item * together;
        const uint32_t k = together == 1 ? item - first * each : 0;
        uint64_t src[4];
        uint64_t dst[4];
        uint32_t bytes[4];
#pragma unroll
        for (uint32_t q = 0; q < 4; ++q) {
            const uint32_t at = first + q * together / 4;
            const uint32_t begin = together == 1 ? k * kDeepBytes + q * (kDeepBytes / 4) : q * (kDeepBytes / 4) % (kDeepBytes / together);
            const bool there = at < nseg;
            const uint32_t r = there ? at : first;
            const uint64_t len = there ? rows[3ull * r + 2] : 0;
            src[q] = rows[3ull * r] + begin;
            dst[q] = rows[3ull * r + 1] + begin;
            const bool fits = len <= len0 && ((src[q] | dst[q]) & (kUnitBytes - 1)) == 0;
            if (!fits && len != 0 && begin == 0) {
                ListRest(rest, capacity, src[q], dst[q], len);
            }
            const uint32_t left = fits && len > begin ? static_cast<uint32_t>(len) - begin : 0;
            bytes[q] = left < kDeepBytes / 4 ? left : kDeepBytes / 4;
        }
        if ((bytes[0] | bytes[1] | bytes[2] | bytes[3]) != 0) {
            CopyPartWindowed(src, dst, bytes, loadAt, storeAt);
        }
    } while (onward());
}

// The sum of the lanes up to and with this one.
__device__ __forceinline__ uint32_t LanesUpTo(uint32_t v)
{
    v += __builtin_amdgcn_update_dpp(0u, v, 0x111, 0xf, 0xf, false);       // row_shr:1, 2, 4, 8
    v += __builtin_amdgcn_update_dpp(0u, v, 0x112, 0xf, 0xf, false);
    v += __builtin_amdgcn_update_dpp(0u, v, 0x114, 0xf, 0xf, false);
    v += __builtin_amdgcn_update_dpp(0u, v, 0x118, 0xf, 0xf, false);
    v += __builtin_amdgcn_update_dpp(0u, v, 0x142, 0xa, 0xf, false);       // row_bcast:15 into the rows 1 and 3
    v += __builtin_amdgcn_update_dpp(0u, v, 0x143, 0xc, 0xf, false);       // row_bcast:31 into the rows 2 and 3
    return v;
}

// The last of n ascending words that is not above c; the first is 0.
__device__ __forceinline__ uint32_t LastUpTo(const uint32_t *first, uint32_t n, uint32_t c)
{
    const uint32_t lane = threadIdx.x & 63u;
    uint32_t lo = 0;
    while (n > 1) {
        const uint32_t step = (n + 63u) >> 6;
        const uint32_t probe = lane * step;
        const uint32_t at = (__popcll(__ballot(probe < n && first[lo + (probe < n ? probe : 0)] <= c)) - 1) * step;
        lo += at;
        n = n - at < step ? n - at : step;
    }
    return lo;
}

// Chunk k of kWindowUnits units of a segment, whatever its addresses, by one wave with sixteen loads per lane in flight: loads from
// `loadAt` on the clock, stores from `storeAt` on, and `meanwhile` while the loads are on their way.  What a lane past the end of the
// chunk loads is the last unit (XcopyPieceWindowKernel says why).
template <class F>
__device__ __forceinline__ void CopyDeepChunk(uint64_t src, uint64_t dst, uint64_t len, uint32_t k, uint64_t loadAt, uint64_t storeAt,
                                              F meanwhile)
{
    uint32_t tid = threadIdx.x & 63u;
    asm volatile("" : "+v"(tid));
    const SegGeom g = SegmentGeometry(dst, len);
    const uint64_t u0 = static_cast<uint64_t>(k) * kWindowUnits;
    const uint64_t left = g.body > u0 ? g.body - u0 : 0;
    const uint32_t n = left < kWindowUnits ? static_cast<uint32_t>(left) : kWindowUnits;
    const uint64_t s = src + g.head + u0 * kUnitBytes;
    const uint64_t d = dst + g.head + u0 * kUnitBytes;
    const uint32_t apart = static_cast<uint32_t>(s) & (kUnitBytes - 1);
    if (n != 0) {
        const uint64_t from = s - apart;
        const uint32_t most = apart != 0 ? n : n - 1;
        u32x4 v[kWindowDepth];
        WaitForClock(loadAt);
#pragma unroll
        for (uint32_t j = 0; j < kWindowDepth; ++j) {
            if (j * 64 <= most) {
                const uint32_t u = j * 64 + tid < most ? j * 64 + tid : most;
                v[j] = LoadAligned(from + u * kUnitBytes);
            }
        }
        const u32x4 last = LoadAligned(from + most * kUnitBytes);
        meanwhile();
        asm volatile("s_waitcnt vmcnt(0)" : "+v"(tid) : : "memory");     // offsets are computed again, not held
        WaitForClock(storeAt);
        if (apart == 0) {
#pragma unroll
            for (uint32_t j = 0; j < kWindowDepth; ++j) {
                if (j * 64 + tid < n) {
                    StoreUnit<kStoreStream>(d + (j * 64 + tid) * kUnitBytes, v[j]);
                }
            }
        } else {
            StoreApart<kStoreStream>(v, last, d, 0, n, apart, tid);
        }
    } else {
        meanwhile();
    }
    // (the last chunk of a segment may have been counted without its head, and hold nothing)
    if (k == 0 && tid < g.head) {
        CopyByte<kStoreStream>(src + tid, dst + tid);
    }
    if ((u0 < g.body || k == 0) && u0 + kWindowUnits >= g.body && tid < g.tail) {
        const uint64_t off = g.head + g.body * kUnitBytes + tid;
        CopyByte<kStoreStream>(src + off, dst + off);
    }
}

// Four chunks of 4 KiB, of up to four segments, as one of 16 KiB; all begin on units and hold one at least.
struct QuadChunk {
    uint64_t src;
    uint64_t dst;
    uint32_t n;         // units
};
__device__ __forceinline__ void CopyQuad(const QuadChunk (&q)[4], uint64_t loadAt, uint64_t storeAt)
{
    uint32_t tid = threadIdx.x & 63u;
    asm volatile("" : "+v"(tid));
    u32x4 v[kWindowDepth];
    WaitForClock(loadAt);
#pragma unroll
    for (uint32_t j = 0; j < kWindowDepth; ++j) {
        const QuadChunk &c = q[j / kDepth];
        const uint32_t u = j % kDepth * 64 + tid;
        v[j] = LoadAligned(c.src + (u < c.n ? u : c.n - 1) * kUnitBytes);
    }
    asm volatile("s_waitcnt vmcnt(0)" : "+v"(tid) : : "memory");
    WaitForClock(storeAt);
#pragma unroll
    for (uint32_t j = 0; j < kWindowDepth; ++j) {
        const QuadChunk &c = q[j / kDepth];
        const uint32_t u = j % kDepth * 64 + tid;
        if (u < c.n) {
            StoreUnit<kStoreStream>(c.dst + u * kUnitBytes, v[j]);
        }
    }
}

// Chunk k of 4 KiB of a segment, by one wave of a workgroup.
__device__ __forceinline__ void CopyCountedChunk(uint64_t src, uint64_t dst, uint64_t len, uint32_t k, uint32_t lane)
{
    if (k < SegmentChunks(dst, len, kXcopyThreads)) {      // it may have been counted without the segment's head, and hold nothing
        CopyChunk<true, kStoreStream, false>(src, dst, len, k, kXcopyThreads, 0, 0, 64, lane);
    }
}

// Chunk c of a table whose chunk prefix is `first`, and of one whose segments have `each` chunks.
__device__ __forceinline__ ChunkRef ChunkOf(const uint64_t *__restrict__ triples, uint32_t seg, uint32_t k)
{
    const uint64_t *t = triples + 3ull * seg;
    return ChunkRef{Uniform(t[0]), Uniform(t[1]), Uniform(t[2]), k};
}
__device__ __forceinline__ ChunkRef PlannedOwner(const uint64_t *__restrict__ triples, const uint32_t *first, uint32_t nseg, uint32_t c)
{
    const uint32_t seg = Uniform(LastUpTo(first, nseg, c));
    return ChunkOf(triples, seg, c - Uniform(first[seg]));
}
__device__ __forceinline__ ChunkRef EqualOwner(const uint64_t *__restrict__ triples, uint32_t each, uint32_t c)
{
    const uint32_t seg = Uniform(c / each);
    return ChunkOf(triples, seg, c - seg * each);
}

// The chunks c to c + 3, of 4 KiB; false unless all four are there, begin on units and end with one.
__device__ __forceinline__ bool PlannedQuad(const uint64_t *__restrict__ triples, const uint32_t *first, uint32_t nseg, uint32_t c,
                                            uint32_t nchunk, QuadChunk (&q)[4])
{
    if (nchunk - c < 4) {
        return false;
    }
    const uint32_t lane = threadIdx.x & 63u;
    const uint32_t seg0 = Uniform(LastUpTo(first, nseg, c));
    const uint32_t near = seg0 + lane < nseg ? first[seg0 + lane] : 0xFFFFFFFFu;      // of this segment and those behind it
    bool whole = true;
#pragma unroll
    for (uint32_t j = 0; j < 4; ++j) {
        const uint32_t row = __popcll(__ballot(near <= c + j)) - 1;
        whole = whole && row < 63;          // more than 60 empty ones between two
        const uint64_t *t = triples + 3ull * (seg0 + row);
        const uint64_t src = Uniform(t[0]);
        const uint64_t dst = Uniform(t[1]);
        const uint64_t len = Uniform(t[2]);
        const uint64_t at = static_cast<uint64_t>(c + j - __builtin_amdgcn_readlane(near, row)) * kXcopyThreads * kUnitBytes;
        q[j].src = src + at;
        q[j].dst = dst + at;
        q[j].n = len - at < kXcopyThreads * kUnitBytes ? static_cast<uint32_t>(len - at) / kUnitBytes : kXcopyThreads;
        whole = whole && ((src | dst | len) & (kUnitBytes - 1)) == 0;
    }
    return whole;
}

// A table that only the GPU can read, of up to kPlannedSegments segments between HBM addresses, in one launch of kWindowWaves waves:
// every workgroup reads the lengths of all of it and has their chunk prefix in LDS after two sums over its lanes.  So it knows what a
// host that could read the table would: the total, which chooses the form, and the owner of every chunk.  No list of long segments,
// no second launch, no event.  Bound: the chain of launch, lengths, prefix, descriptor and first load (4 us) for short tables, HBM for
// long ones.  With the two launches of XcopyDirectKernel / so, us: 64 pages of 8 KiB 9.2 / 3.8, 1000 9.7 / 6.6, 4096 17.7 / 15.5; 500 of
// 32 KiB 11.7 / 8.0, 2000 29.7 / 25.2, 4096 scattered 55.6 / 50.3; 1952 K and V blocks 65.4 / 53.9; 1000 / 4000 ragged segments of up to
// 70 000 bytes 24.0 / 16.6, 71.2 / 65.6; 300 of 2 MB 240 / 206.  Longer tables cost each workgroup more lanes' worth of lengths: with
// kPlannedRun 16, 8000 pages of 8 KiB 28.3 / 30.9, 16 384 ragged of 14 000 bytes 60.3 / 68.9, and that much more code made all others
// 1 to 3 us slower.  Looking four chunks ahead of a quad up while it loads: registers spill, 8000 pages of 8 KiB 33.3.
// Segments of one length, as pages are, take a shorter way: one barrier says that they are, and the owner of a chunk is a division instead of
// a prefix and a search.  us before / so, gathered and scattered: 300 of 32 KiB 5.8 / 5.2, 700 / 1000 / 2000 / 4096 pages of 8 KiB 5.8 / 4.3,
// 6.6 / 4.8, 8.8 / 7.5, 15.4 and 16.1 / 12.9 and 14.1; 1000 of 32 KiB 13.1 and 13.8 / 12.3 and 12.9, 1000 of 64 KiB 24.1 and 26.3 / 22.7 and
// 24.3; 3000 of 8200 bytes at odd addresses 13.5 / 11.4.  All of that way stands behind the other one's code: between its parts, instructions
// that a wave only steps over cost short tables 0.3 us (K and V blocks of 3 MB: no shorter way 4.84, behind 4.91, between 5.28).  Finding out
// that segments differ costs up to 0.25 us from 513 on (1281 blocks of 26 MB 12.70 / 12.95; 1240 of 32 912 bytes, equal but not full enough, 18.4 / 19.1), of which the shorter
// chunks' skipped units give back more to short ones: 4000 ragged segments of up to 9000 bytes 13.4 / 12.6.  Not
// taken: descriptors fetched ahead of that barrier, and all lengths requested by one stretch of code, whatever their number (each
// request of 64 lengths is 24 lines of the L1): 600 / 1000 ragged ones 11.6 / 17.8.
// In windows cut for 6.0 / 6.2 / 6.4 / 6.6 / 6.8 TB/s, the same to 0.5 in four processes: 4096 pages of 32 KiB gathered 49.8 / 48.4 / 47.1 / 46.0 / 45.3,
// scattered 50.2 / 51.2 / 54 / 54 / 54; of 64 KiB gathered 94.5 / 91.7 / 89.4 / 87.3 / 85.7 (7.0: 91), scattered 95.0 / 92.8 / 90.5 / 87.8 / 97 to 102;
// 1000 of 256 KiB scattered 92.0 / 89.6 / 87.1 / 85.2 / 86.7 to 91.6: 6.6 for what is written in order, 6.4 for scattered pages of 64 KiB and more.
// Blocks that are neither read nor written in order hold 6.4 only on multiples of 64 KiB (300 MB at 6.0 / 6.4: 128 KiB there 106.3 / 101.5, on lines 107.4 /
// 114.4; 80 KiB 108.2 / 119.6; 500 and 700 MB of 256 KiB on lines 173.7 / 177.5, 247 / 253) or where their last pieces are so short, which the
// period does not count on, that all have less than kPlannedLoosePercent (72 KiB, 90 %, 117.1 / 110.2; 200 000 bytes, 94 %, 112.0 / 107.3; 110 776, 97 %, 110.1
// / 107.5 to 114.2), and shorter ones of them no uneven parts (32 KiB, 130 MB 50.1 / 53.4).
// Shorter ones that are read in order are stored at random places no faster than 5.6, but read faster: with a read part of 0.40 / 0.44 / 0.47 / 0.50 / 0.53 of the period, 4096
// of 32 KiB at 6.0 50.6 / 50.1 / 50.2 / 50.1 / 51.5, at 6.2 50.5 / 48.9 / 48.9 / 49.8 / 53.8, at 6.4 51.6 / 48.7 / 48.8 / 53.2 / 54.7; so 29/64 at 6.3, 47.9.  The others
// gain nothing from uneven parts.
template <uint32_t kWaves, uint32_t kRun>
__global__ __launch_bounds__(64 * kWaves) __attribute__((amdgpu_waves_per_eu(4, 4)))
void XcopyPlannedKernel(uint64_t table, uint32_t nseg, TablePace pace)
{
    constexpr uint32_t kGroups = kWindowWaves / kWaves;     // the launch's workgroups
    const uint64_t *const triples = Buffer<const uint64_t>(table);
    extern __shared__ uint32_t words[];                     // PlannedLds()
    if (nseg == 0) {
        return;
    }
    const uint64_t t0 = wall_clock64();
    const uint32_t lane = threadIdx.x & 63u;
    const uint32_t wave = threadIdx.x >> 6;
    uint32_t *sums = words;                                 // [4][kWaves]
    uint32_t *first = words + 4 * kWaves;                   // [nseg + 1]: chunks of 4 KiB of each segment, then the prefix of its chunks
    const uint32_t run = (nseg + 64 * kWaves - 1) / (64 * kWaves);
    const uint64_t len0 = reinterpret_cast<const __attribute__((address_space(4))) uint64_t *>(table)[2];     // by a scalar load
    const uint64_t *t = triples + 3ull * (lane < nseg ? lane : 0);
    const uint32_t from = static_cast<uint32_t>(t[0]);      // of the first 64 segments, the same for every wave
    const uint32_t to = static_cast<uint32_t>(t[1]);
    const uint32_t bits = from | to;
    uint64_t len[kRun];
#pragma unroll
    for (uint32_t r = 0; r < kRun; ++r) {
        const uint32_t seg = r * 64 * kWaves + threadIdx.x;
        // (a branch waits for what is on its way: one wave asks for all, sixteen for no more than they need)
        len[r] = kWaves == 1 || r < run ? triples[3ull * (seg < nseg ? seg : 0) + 2] : 0;
    }
    uint32_t spare = 0;
    bool other = false;
#pragma unroll
    for (uint32_t r = 0; r < kRun; ++r) {
        const uint32_t seg = r * 64 * kWaves + threadIdx.x;
        if (r < run && seg < nseg) {
            first[seg] = static_cast<uint32_t>((len[r] + 4095) >> 12);
            spare += PlannedSpare(len[r]);
            other = other || len[r] != len0;
        }
    }
    // The form: short tables a chunk of 4 KiB per wave; others 16 KiB, of one segment where those are nearly full or where a source and
    // its destination may differ modulo 16, else of up to four.
    constexpr uint32_t grid = kWindowWaves;
    constexpr uint64_t kDeepBytes = static_cast<uint64_t>(kWindowUnits) * kUnitBytes;
    uint32_t item = wave * kGroups + blockIdx.x;            // neighbouring ones on neighbouring XCDs
    const bool aligned = __ballot(bits % kUnitBytes != 0) == 0;
    // (Each owner with a loop of its own: code that a wave only steps over is fetched all the same, at 0.3 us.)
    auto deepChunks = [&](auto owner, uint32_t items, uint32_t waves, uint64_t loadAt, uint64_t storeAt, uint32_t step) {
        // the next chunk's owner is looked up while the loads of this one are on their way
        ChunkRef r = owner(item);
        for (;;) {
            const bool more = items - item > waves;
            ChunkRef next = r;
            CopyDeepChunk(r.src, r.dst, r.len, r.k, loadAt, storeAt, [&] {
                if (more) {
                    next = owner(item + waves);
                }
            });
            if (!more) {
                return;
            }
            r = next;
            item += waves;
            loadAt += step;
            storeAt += step;
        }
    };
    auto shallowChunks = [&](auto owner, uint32_t items, uint32_t waves) {
        for (; item < items; item += waves) {
            const ChunkRef r = owner(item);
            CopyCountedChunk(r.src, r.dst, r.len, r.k, lane);
        }
    };
    bool equal = __ballot(other) == 0;
    if (kWaves > 1 && lane == 0) {
        sums[3 * kWaves + wave] = equal ? 1 : 0;
    }
    __syncthreads();
    if (kWaves > 1) {
        equal = __ballot(lane < kWaves && sums[3 * kWaves + (lane < kWaves ? lane : 0)] == 0) == 0;
    }
    // Segments that all have the length of the first need neither sums nor a prefix.  Pages of up to 16 KiB never go as quads.
    if (__builtin_expect(equal, 0)) {
        const uint32_t shallow0 = static_cast<uint32_t>((len0 + 4095) >> 12);
        const uint32_t deep0 = (shallow0 + 3) / 4;
        const uint32_t total = PlannedTotal(nseg * deep0, nseg * PlannedSpare(len0));
        const bool large = total > kPlannedShallowChunks;
        if (shallow0 != 0 && !(large && aligned && shallow0 > 4 && !PlannedFull(total, nseg * deep0))) {
            const uint32_t each = large ? deep0 : shallow0;
            const uint32_t items = nseg * each;
            const bool held = large && items <= grid && total <= kPlannedHeldChunks;
            const bool paced = large && total > kPlannedHeldChunks && aligned && pace.windowTicks != 0 && PlannedFull(total, items);
            const uint32_t rounds = (items + grid - 1) / grid;
            const uint32_t waves = paced ? (items + rounds - 1) / rounds : grid;
            if (item >= items || item >= waves) {
                return;
            }
            auto divided = [&](uint32_t c) { return EqualOwner(triples, each, c); };
            if (!large) {
                shallowChunks(divided, items, waves);
                return;
            }
            uint64_t loadAt = 0;
            uint64_t storeAt = 0;
            uint32_t period = 0;
            if (paced) {
                const TableWindows w = WindowsOf(pace, from, to, len0, nseg < 64 ? nseg : 64,
                                                 total * 25ull < items * static_cast<uint64_t>(kPlannedLoosePercent));
                period = static_cast<uint32_t>(w.ticks * (waves * kDeepBytes) >> 26);
                const uint32_t reading = w.reading == 32 ? period / 2 : period / 64 * w.reading;
                const uint64_t start = AgreedStart(pace.seq);
                loadAt = start + static_cast<uint64_t>(item) * reading / waves;
                storeAt = start + reading + static_cast<uint64_t>(item) * (period - reading) / waves;
            } else if (held && pace.holdTicks != 0) {
                storeAt = t0 + pace.equalTicks + static_cast<uint32_t>(static_cast<uint64_t>(pace.equalMoreTicks) * total >> 14);
            }
            deepChunks(divided, items, waves, loadAt, storeAt, period);
            return;
        }
    }
    uint32_t count[kRun];
    uint32_t shallow = 0;       // chunks of 4 KiB,
    uint32_t deep = 0;          // of 16 KiB
#pragma unroll
    for (uint32_t r = 0; r < kRun; ++r) {
        const uint32_t seg = threadIdx.x * run + r;
        count[r] = r < run && seg < nseg ? first[seg] : 0;
        shallow += count[r];
        deep += (count[r] + 3) / 4;
    }
    const uint32_t shallowUpTo = LanesUpTo(shallow);
    const uint32_t deepUpTo = LanesUpTo(deep);
    uint32_t spareAll = __builtin_amdgcn_readlane(LanesUpTo(spare), 63);
    uint32_t shallowAll = __builtin_amdgcn_readlane(shallowUpTo, 63);
    uint32_t deepAll = __builtin_amdgcn_readlane(deepUpTo, 63);
    uint32_t shallowBase = 0;
    uint32_t deepBase = 0;
    if (kWaves > 1) {
        if (lane == 0) {
            sums[wave] = shallowAll;
            sums[kWaves + wave] = deepAll;
            sums[2 * kWaves + wave] = spareAll;
        }
        __syncthreads();
        const uint32_t at = lane < kWaves ? lane : 0;
        const uint32_t a = LanesUpTo(lane < kWaves ? sums[at] : 0);
        const uint32_t b = LanesUpTo(lane < kWaves ? sums[kWaves + at] : 0);
        spareAll = __builtin_amdgcn_readlane(LanesUpTo(lane < kWaves ? sums[2 * kWaves + at] : 0), 63);
        shallowBase = wave == 0 ? 0 : __builtin_amdgcn_readlane(a, wave == 0 ? 0 : wave - 1);
        deepBase = wave == 0 ? 0 : __builtin_amdgcn_readlane(b, wave == 0 ? 0 : wave - 1);
        shallowAll = __builtin_amdgcn_readlane(a, 63);
        deepAll = __builtin_amdgcn_readlane(b, 63);
    }
    const uint32_t total = PlannedTotal(deepAll, spareAll);
    const bool large = total > kPlannedShallowChunks;
    const bool quads = large && aligned && !PlannedFull(total, deepAll);
    const bool byDeep = large && !quads;
    uint32_t before = byDeep ? deepBase + deepUpTo - deep : shallowBase + shallowUpTo - shallow;
#pragma unroll
    for (uint32_t r = 0; r < kRun; ++r) {
        const uint32_t seg = threadIdx.x * run + r;
        if (r < run && seg < nseg) {
            first[seg] = before;
            before += byDeep ? (count[r] + 3) / 4 : count[r];
        }
    }
    const uint32_t nchunk = byDeep ? deepAll : shallowAll;
    if (threadIdx.x == 0) {
        first[nseg] = nchunk;
    }
    __syncthreads();

    const uint32_t items = quads ? (nchunk + 3) / 4 : nchunk;
    const bool held = large && items <= grid && total <= kPlannedHeldChunks;
    const bool paced = large && total > kPlannedHeldChunks && aligned && pace.windowTicks != 0 && PlannedFull(total, items);
    const uint32_t rounds = (items + grid - 1) / grid;
    const uint32_t waves = paced ? (items + rounds - 1) / rounds : grid;
    if (item >= items || item >= waves) {
        return;
    }
    const uint32_t period = static_cast<uint32_t>(pace.windowTicks * (waves * kDeepBytes) >> 26);
    const uint32_t hold = pace.holdTicks + static_cast<uint32_t>(static_cast<uint64_t>(pace.holdMoreTicks) * total >> 14);
    uint64_t loadAt = paced ? AgreedStart(pace.seq) + static_cast<uint64_t>(item) * (period / 2) / waves : 0;
    uint64_t storeAt = paced ? loadAt + period / 2 : held && pace.holdTicks != 0 ? t0 + hold : 0;
    const uint32_t step = paced ? period : 0;
    auto planned = [&](uint32_t c) { return PlannedOwner(triples, first, nseg, c); };
    if (byDeep) {
        deepChunks(planned, items, waves, loadAt, storeAt, step);
        return;
    }
    if (quads) {
        for (; item < items; item += waves) {
            QuadChunk q[4];
            if (PlannedQuad(triples, first, nseg, item * 4, nchunk, q)) {
                CopyQuad(q, loadAt, storeAt);
            } else {
                WaitForClock(storeAt);
                const uint32_t end = item * 4 + 4 < nchunk ? item * 4 + 4 : nchunk;
#pragma unroll 1
                for (uint32_t c = item * 4; c < end; ++c) {
                    const ChunkRef r = planned(c);
                    CopyCountedChunk(r.src, r.dst, r.len, r.k, lane);
                }
            }
            loadAt += step;
            storeAt += step;
        }
        return;
    }
    shallowChunks(planned, items, waves);
}

// The segments of a list that a wave is at, one per lane, so that the owner of a piece is found without a load.
struct RestRows {
    uint64_t first = ~0ull;     // of the lane's segment
    uint64_t src = 0;
    uint64_t dst = 0;
    uint64_t len = 0;
    uint64_t end;               // pieces of the segments up to these, ~0 when they are the last

    __device__ __forceinline__ RestRows(const RestList *rest, uint32_t lo, uint32_t count)
    {
        const uint32_t i = lo + (threadIdx.x & 63u);
        if (i < count) {
            const RestSegment r = rest->entry[i];
            first = r.first;
            src = r.src;
            dst = r.dst;
            len = r.len;
        }
        end = lo + 64 < count ? Uniform(rest->entry[lo + 64].first) : ~0ull;
    }
};

// The last segment of [lo, count) whose `first` is <= p; that of lo is.
__device__ __forceinline__ uint32_t RestOwner(const RestList *rest, uint32_t lo, uint32_t count, uint64_t p)
{
    const uint32_t lane = threadIdx.x & 63u;
    while (count - lo > 1) {
        const uint32_t step = (count - lo + 63u) >> 6;
        const uint32_t probe = lo + lane * step;
        const uint32_t hits = __popcll(__ballot(probe < count && rest->entry[probe < count ? probe : lo].first <= p));
        lo += hits > 1 ? (hits - 1) * step : 0;
        count = count - lo < step ? count : lo + step;
    }
    return lo;
}

// Whether this is the last of `all` calls on a counter, which it leaves at 0.
__device__ __forceinline__ bool CountsLast(uint64_t *counter, uint64_t all)
{
    if (__hip_atomic_fetch_add(counter, 1ull, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) != all - 1) {
        return false;
    }
    __hip_atomic_store(counter, 0ull, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    return true;
}

// The segments XcopyDirectKernel has listed; usually none.  The last workgroup leaves the list empty.  HBM is the bound; two workgroups
// of eight waves per CU, sixteen of them on neighbouring chunks of one MiB, is the shape that loses on no kind of table.  By where the
// allocator has put a pool a copy runs in one of two modes; us in the slower / faster one, with the planner that listed chunks, with a
// list of pieces (room for sixteen segments of 256 MiB, what came after was copied by one wave each) and so:
//   1 GiB among 4096 short segments   434 / 408    421 / 390         411 / 389
//   one of 1 GiB                      410 / 396    409 / 383         398 / 376
//   16 x 256 MiB                     1742 / 1414  1578 / 1487       1660 / 1419
//   32 x 512 MiB                     7100 / 5774  145768 / 145898   6815 / 5711
//   300 x 32 MiB at odd addresses    4244 / 3556  58363 / 58413     4244 / 3496
// Half the lanes: aligned segments 0 to 5 % faster in the slower mode, odd ones 3 to 11 % slower; twice the workgroups: 1 to 5 % slower.
// Neighbouring waves on neighbouring pieces of 64 KiB instead: 1 GiB 421 / 401.  Every workgroup that counts itself done on one word costs
// 35 to 70 ns at the end (1024 of them: 256 MiB 146 us, on sixteen words 112), hence the groups.
template <bool kNtLoad, int kStore>
__global__ __launch_bounds__(kRestLanes) void XcopyRestKernel(RestList *rest, uint32_t capacity, uint32_t units)
{
    const uint64_t taken = Uniform(__hip_atomic_load(&rest->taken, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT));
    if (taken == 0) {
        return;
    }
    const uint32_t count = taken / kRestEntry < capacity ? static_cast<uint32_t>(taken / kRestEntry) : capacity;
    const uint64_t pieces = taken % kRestEntry;
    uint32_t lo = 0;
    RestRows rows(rest, lo, count);
    for (uint64_t p = blockIdx.x; p < pieces; p += gridDim.x) {
        if (p >= rows.end) {
            lo = RestOwner(rest, lo + 64, count, p);
            rows = RestRows(rest, lo, count);
        }
        const uint32_t row = __popcll(__ballot(rows.first <= p)) - 1;
        const uint64_t src = ReadLane64(rows.src, row);
        const uint64_t dst = ReadLane64(rows.dst, row);
        const uint64_t len = ReadLane64(rows.len, row);
        const uint64_t mine = p - ReadLane64(rows.first, row);
        const uint64_t all = RestPieces(len);
        if (mine >= all) {
            continue;       // not with a list of one call's
        }
        // pieces side by side share a stretch of the segment chunk by chunk
        const uint64_t stretch = mine / kRestShare * kRestShare;
        const uint32_t share = all - stretch < kRestShare ? static_cast<uint32_t>(all - stretch) : kRestShare;
        const uint64_t from = stretch * kRestPieceBytes;
        const uint64_t bytes = len - from < share * kRestPieceBytes ? len - from : share * kRestPieceBytes;
        const uint64_t chunks = SegmentChunks(dst + from, bytes, units);
        for (uint64_t c = mine - stretch; c < chunks; c += share) {
            CopyChunk<kNtLoad, kStore>(src + from, dst + from, bytes, c, units);
        }
    }
    __syncthreads();
    if (threadIdx.x != 0) {
        return;
    }
    const uint32_t group = blockIdx.x % kRestGroups;
    const uint32_t groups = gridDim.x < kRestGroups ? gridDim.x : kRestGroups;
    if (CountsLast(&rest->done[group].count, (gridDim.x - group + kRestGroups - 1) / kRestGroups) &&
        CountsLast(&rest->done[kRestGroups].count, groups)) {
        __hip_atomic_store(&rest->taken, 0ull, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    }
}

// The heads of lists that are new, one a workgroup.
__global__ void XcopyClearListsKernel(uint8_t *lists, uint64_t stride)
{
    uint64_t *head = reinterpret_cast<uint64_t *>(lists + blockIdx.x * stride);
    for (uint32_t i = threadIdx.x; i < kRestHeadBytes / 8; i += blockDim.x) {
        head[i] = 0;
    }
}

Policy PolicyOf(int route)
{
    switch (route) {
        case MFRT_ROUTE_TO_HOST:
            // measured over the host link with 122-segment batches: write-through 56.0 GB/s,
            // plain 54.4 GB/s, nontemporal-only 49 GB/s
            return Policy{false, kStoreThrough};
        case MFRT_ROUTE_FROM_HOST:
            return Policy{true, kStorePlain};
        default:
            // HBM to HBM, measured on the 9 MB batch: streaming loads and stores 5.2 us, plain 6.3 us,
            // stores written through 6.5 us (they are 4 % faster on a 1 GiB copy only)
            return Policy{true, kStoreStream};
    }
}

// Runs `launch` with the template instance matching a run-time policy.
template <class Launch>
int WithPolicy(const Policy &policy, Launch launch)
{
    if (policy.ntLoad) {
        switch (policy.store) {
            case kStoreThrough:
                return launch(std::true_type{}, std::integral_constant<int, kStoreThrough>{});
            case kStoreStream:
                return launch(std::true_type{}, std::integral_constant<int, kStoreStream>{});
            default:
                return launch(std::true_type{}, std::integral_constant<int, kStorePlain>{});
        }
    }
    switch (policy.store) {
        case kStoreThrough:
            return launch(std::false_type{}, std::integral_constant<int, kStoreThrough>{});
        case kStoreStream:
            return launch(std::false_type{}, std::integral_constant<int, kStoreStream>{});
        default:
            return launch(std::false_type{}, std::integral_constant<int, kStorePlain>{});
    }
}

// Lanes per workgroup: a workgroup moves its chunk in one step of kDepth accesses per lane, so the
// chunk size picks the workgroup size (4 KiB: one wave, 8 KiB: two, 16 KiB and more: four).
// Measured on a 9 MB batch and on 1 MiB ... 1 GiB copies: single-wave workgroups on 4 KiB chunks are
// the fastest shape at every size (KV batch 4.8 us against 5.5 us with four waves on 16 KiB).
uint32_t LanesFor(uint32_t units, int route)
{
    if (route == MFRT_ROUTE_TO_HOST || route == MFRT_ROUTE_FROM_HOST) {
        return kXcopyThreads;   // link routes were tuned with four-wave workgroups, few of them (GridFor)
    }
    const uint32_t lanes = units / kDepth;
    return lanes <= 64 ? 64u : (lanes <= 128 ? 128u : kXcopyThreads);
}

// Rate of the current device's constant-rate clock, the one wall_clock64() reads; 0 where it is not known, and nothing waits.
uint32_t ClockKhz()
{
    static std::atomic<int> khzOf[64];
    int dev = 0;
    if (hipGetDevice(&dev) != hipSuccess || dev < 0 || dev >= 64) {
        return 0;
    }
    int khz = khzOf[dev].load(std::memory_order_relaxed);
    if (khz == 0) {
        if (hipDeviceGetAttribute(&khz, hipDeviceAttributeWallClockRate, dev) != hipSuccess || khz <= 0) {
            khz = -1;
        }
        khzOf[dev].store(khz, std::memory_order_relaxed);
    }
    return khz < 0 ? 0 : static_cast<uint32_t>(khz);
}

uint32_t TicksOf(uint32_t nanos, uint32_t khz)
{
    const uint64_t capped = nanos < kHoldMaxNanos ? nanos : kHoldMaxNanos;   // no wave ever waits longer
    return static_cast<uint32_t>(capped * khz / 1000000u);
}

uint32_t HoldTicks(uint32_t nanos)
{
    return nanos == 0 ? 0 : TicksOf(nanos, ClockKhz());
}

// anyOrder: the launch carries no barrier, so the command processor may start it while launches queued
// before it on the same stream still run (hipExtAnyOrderLaunch; a 9 MB batch on one stream: 5.3 against 5.9 us).
// holdNanos: the caller's HoldNanosFor(); the launch qualifies only if it has one chunk per workgroup, of
// 4 KiB (stores of four loads per lane held) or of kWindowUnits units (of sixteen).
template <bool kNtLoad, int kStore>
int LaunchInline(const InlinePlan &plan, uint32_t grid, uint32_t lanes, hipStream_t stream, bool anyOrder, uint32_t holdNanos)
{
    const uint32_t flags = anyOrder ? hipExtAnyOrderLaunch : 0u;
    const bool deep = plan.units == kWindowUnits && grid == plan.nchunk && holdNanos != 0 && !anyOrder;
    if (deep) {
        lanes = 64;
    }
    const uint32_t ticks = grid == plan.nchunk && lanes == 64 ? HoldTicks(holdNanos) : 0;
    const bool single = plan.first[1] == kNoChunk;
    const uint32_t lineChunks = single ? static_cast<uint32_t>(LineChunks(plan.dst[0], plan.len[0], plan.units)) : 0;
    if (single && deep && ticks != 0 && lineChunks <= kHeldMaxPieces) {
        return Launch(XcopySingleHeldKernel, lineChunks, 64, 0, stream, plan.src[0], plan.dst[0], plan.len[0], ticks);
    }
    const bool offLine = kStore == kStoreStream && single && (plan.dst[0] & (kLineBytes - 1)) != 0;
    if (single && (offLine || plan.nchunk <= kSingleMaxChunks)) {
        // (A chunk more than the waves that hold their stores together would be read when all others have been stored.)
        const uint32_t onLines = offLine && (ticks == 0 || lineChunks <= kHoldMaxChunks) ? 1 : 0;
        const uint32_t nchunk = onLines != 0 ? lineChunks : plan.nchunk;
        grid = grid == plan.nchunk ? nchunk : grid;
        if (anyOrder) {
            hipExtLaunchKernelGGL((XcopySingleKernel<kNtLoad, kStore>), dim3(grid), dim3(lanes), 0, stream, nullptr, nullptr, flags,
                                  plan.src[0], plan.dst[0], plan.len[0], nchunk, plan.units, 0u, lanes, grid, onLines);
            return static_cast<int>(hipGetLastError());
        }
        const auto kernel = ticks == 0 ? XcopySingleKernel<kNtLoad, kStore, kHoldNone> : XcopySingleKernel<kNtLoad, kStore, kHoldShallow>;
        return Launch(kernel, grid, lanes, 0, stream, plan.src[0], plan.dst[0], plan.len[0], nchunk, plan.units, ticks, lanes, grid, onLines);
    }
    // The ordered launches go through hipLaunchKernel with an argument array: the triple-chevron form pushes and pops a
    // launch configuration around the same call, 0.15 us of host time per launch with this 3 KiB argument block.
    uint32_t holdTicks = ticks;
    void *args[] = {const_cast<InlinePlan *>(&plan), &holdTicks};
    const void *kernel = reinterpret_cast<const void *>(&XcopyInlineKernel<kNtLoad, kStore, kHoldNone>);
    if (ticks != 0 && !anyOrder) {
        kernel = deep ? reinterpret_cast<const void *>(&XcopyInlineKernel<kNtLoad, kStore, kHoldDeep>)
                      : reinterpret_cast<const void *>(&XcopyInlineKernel<kNtLoad, kStore, kHoldShallow>);
    }
    if (anyOrder) {
        hipExtLaunchKernelGGL((XcopyInlineKernel<kNtLoad, kStore>), dim3(grid), dim3(lanes), 0, stream, nullptr, nullptr, flags, plan,
                              0u);
        return static_cast<int>(hipGetLastError());
    }
    return static_cast<int>(hipLaunchKernel(kernel, dim3(grid), dim3(lanes), args, 0, stream));
}

// The plan with the chunks of LineChunks(), which are others also where a segment on a line ends with a few bytes behind its last whole chunk.
InlinePlan CutOnLines(const InlinePlan &plan)
{
    InlinePlan lines = plan;
    uint64_t chunks = 0;
    for (uint32_t i = 0; i < kInlineSegs && plan.first[i] != kNoChunk; ++i) {
        lines.first[i] = static_cast<uint32_t>(chunks);
        chunks += LineChunks(plan.dst[i], plan.len[i], plan.units);
    }
    lines.nchunk = static_cast<uint32_t>(chunks);
    return lines;
}

// windowMBps: the rate (MB/s of HBM traffic, read + written) the period of a windowed launch is cut for.
int LaunchWindowed(const InlinePlan &plan, uint32_t windowMBps, hipStream_t stream)
{
    const InlinePlan lines = CutOnLines(plan);
    const uint32_t grid = WindowGrid(lines.nchunk, kLongWaves);
    const uint32_t ticks = WindowPeriodTicks(2ull * grid * kWindowUnits * kUnitBytes, windowMBps);
    if (ticks == 0) {
        return static_cast<int>(hipErrorInvalidValue);
    }
    hipLaunchKernelGGL(XcopyWindowKernel, dim3(grid), dim3(64), 0, stream, lines, ticks, NextWindowSeq());
    return static_cast<int>(hipGetLastError());
}

// A launch whose own end is what `event` (may be null) stands for: an event recorded behind a launch is a packet of its own, 2.8 us
// of the stream's time (launches of 10 us with an event each 13.8 us, so 11.0, without 11.0).
template <typename... Params, typename... Args>
int LaunchWithEvent(void (*kernel)(Params...), uint32_t grid, uint32_t lanes, hipStream_t stream, hipEvent_t event, Args... args)
{
    if (event == nullptr) {
        return Launch(kernel, grid, lanes, 0, stream, args...);
    }
    hipExtLaunchKernelGGL(kernel, dim3(grid), dim3(lanes), 0, stream, nullptr, event, 0, args...);
    return static_cast<int>(hipGetLastError());
}

int LaunchPieces(void (*kernel)(uint64_t, uint32_t, uint32_t, uint32_t, uint64_t, uint64_t), uint32_t lanes, const void *pieces, uint32_t count,
                 uint32_t ticks, hipStream_t stream, hipEvent_t event, void *word, uint32_t value, void *counter)
{
    const uint32_t grid = (count + kPieceGroup - 1) / kPieceGroup * kPieceGroup;
    return LaunchWithEvent(kernel, grid, lanes, stream, event, At(pieces), count, ticks, value, At(word), At(counter));
}

// `pace`: of tables that may go as XcopySampledKernel's, else null.
template <bool kNtLoad, int kStore>
int LaunchDirect(const uint64_t *triples, uint32_t nseg, uint32_t units, uint32_t grid, uint32_t restGrid, uint32_t lanes, RestList *rest,
                 uint32_t capacity, hipStream_t stream, hipEvent_t event, const TablePace *pace = nullptr)
{
    hipError_t err = hipSuccess;
    if (kStore == kStoreStream && pace != nullptr && lanes == 64) {
        err = static_cast<hipError_t>(Launch(XcopySampledKernel, grid, 64, 0, stream, At(triples), nseg, At(rest), capacity, *pace));
    } else {
        hipLaunchKernelGGL((XcopyDirectKernel<kNtLoad, kStore>), dim3(grid), dim3(lanes), 0, stream, triples, nseg, units, rest, capacity);
        err = hipGetLastError();
    }
    if (err != hipSuccess) {
        return static_cast<int>(err);
    }
    const bool link = kStore != kStoreStream;
    err = static_cast<hipError_t>(LaunchWithEvent(XcopyRestKernel<kNtLoad, kStore>, restGrid, link ? lanes : kRestLanes, stream, event, rest,
                                                  capacity, link ? units : kDepth * kRestLanes));
    if (err != hipSuccess) {   // what the first launch has listed must not be taken for the next call's
        (void)Launch(XcopySignalKernel, 1, 64, 0, stream, At(&rest->taken), 0u);
    }
    return static_cast<int>(err);
}

// longWaves: for kLongWaves of them instead of kWindowWaves (XcopySampledKernel has the figures).
TablePace PaceOf(uint32_t holdNanos, uint32_t holdMoreNanos, uint32_t windowMBps, bool longWaves)
{
    const uint32_t sooner = holdMoreNanos != 0 ? kTableHoldNanos - kTableEqualNanos : 0;     // a wait set by hand is what it is
    const uint32_t equalNanos = holdNanos > sooner ? holdNanos - sooner : holdNanos;
    const uint32_t khz = ClockKhz();
    return TablePace{TicksOf(holdNanos, khz),
                     TicksOf(holdMoreNanos, khz),
                     TicksOf(equalNanos, khz),
                     TicksOf(holdMoreNanos != 0 ? holdMoreNanos + kTableEqualMoreNanos - kTableHoldMoreNanos : 0, khz),
                     WindowPeriodTicksAt(2ull << 26, windowMBps, khz),
                     WindowPeriodTicksAt(2ull << 26, windowMBps / 20 * 21, khz),
                     WindowPeriodTicksAt(2ull << 26, longWaves ? windowMBps / 60 * 67 : windowMBps / 15 * 16, khz),
                     WindowPeriodTicksAt(2ull << 26, longWaves ? windowMBps / 60 * 67 : windowMBps / 20 * 22, khz),
                     NextWindowSeq()};
}

int Signal(void *mask, uint32_t maskValue, hipStream_t stream)
{
    if (mask == nullptr) {
        return 0;
    }
    return Launch(XcopySignalKernel, 1, 64, 0, stream, At(mask), maskValue);
}

}  // namespace
}  // namespace mf

extern "C" int mfk_xcopy_inline(const void *inlinePlan, int route, uint32_t grid, void *mask, uint32_t maskValue,
                                void *stream, int anyOrder, uint32_t holdNanos)
{
    const mf::InlinePlan &plan = *static_cast<const mf::InlinePlan *>(inlinePlan);
    hipStream_t s = static_cast<hipStream_t>(stream);
    if (plan.nchunk == 0) {
        return mf::Signal(mask, maskValue, s);
    }
    if (grid == 0 || grid > plan.nchunk) {
        grid = plan.nchunk;
    }
    if (grid > (1u << 24) - 1) {
        grid = (1u << 24) - 1;   // the grid size in lanes must stay below 2^32; workgroups loop over the rest
    }
    const int err = mf::WithPolicy(mf::PolicyOf(route), [&](auto ntLoad, auto store) {
        return mf::LaunchInline<decltype(ntLoad)::value, decltype(store)::value>(plan, grid, mf::LanesFor(plan.units, route), s,
                                                                                 anyOrder != 0, holdNanos);
    });
    return err != 0 ? err : mf::Signal(mask, maskValue, s);
}

extern "C" int mfk_xcopy_done(const void *inlinePlan, int route, uint32_t grid, void *word, uint32_t value, void *counter, void *stream)
{
    using namespace mf;
    const InlinePlan &plan = *static_cast<const InlinePlan *>(inlinePlan);
    if (plan.nchunk == 0 || grid == 0) {
        return static_cast<int>(hipErrorInvalidValue);
    }
    grid = grid < plan.nchunk ? grid : plan.nchunk;
    hipStream_t s = static_cast<hipStream_t>(stream);
    DoneMark mark{static_cast<uint64_t *>(word), static_cast<uint32_t *>(counter), value, grid};
    uint64_t src = plan.src[0];
    uint64_t dst = plan.dst[0];
    uint32_t len = plan.len[0];
    uint32_t nchunk = plan.nchunk;
    uint32_t units = plan.units;
    uint32_t lanes = LanesFor(plan.units, route);
    void *singleArgs[] = {&src, &dst, &len, &nchunk, &units, &lanes, &mark.word, &mark.counter, &mark.value, &mark.groups};
    void *args[] = {const_cast<InlinePlan *>(&plan), &mark};
    const bool single = plan.first[1] == kNoChunk;
    const bool nt = PolicyOf(route).ntLoad;
    const void *kernel = nt ? reinterpret_cast<const void *>(&XcopyInlineDoneKernel<true>)
                            : reinterpret_cast<const void *>(&XcopyInlineDoneKernel<false>);
    if (single) {
        kernel = nt ? reinterpret_cast<const void *>(&XcopySingleDoneKernel<true>)
                    : reinterpret_cast<const void *>(&XcopySingleDoneKernel<false>);
    }
    return static_cast<int>(hipLaunchKernel(kernel, dim3(grid), dim3(lanes), single ? singleArgs : args, 0, s));
}

extern "C" uint32_t mfk_xcopy_window_units(void)
{
    return mf::kWindowUnits;
}

// 1 when the period of a windowed launch can be computed on the current device (its constant-rate clock is known).
extern "C" int mfk_xcopy_windows_available(void)
{
    return mf::WindowPeriodTicks(2ull * mf::kWindowWaves * mf::kWindowUnits * mf::kUnitBytes, 6800000u) != 0 ? 1 : 0;
}

extern "C" int mfk_xcopy_windowed(const void *inlinePlan, uint32_t windowMBps, void *mask, uint32_t maskValue, void *stream)
{
    using namespace mf;
    const InlinePlan &plan = *static_cast<const InlinePlan *>(inlinePlan);
    hipStream_t s = static_cast<hipStream_t>(stream);
    if (plan.units != kWindowUnits || plan.nchunk == 0 || windowMBps == 0) {
        return -1;
    }
    const int err = LaunchWindowed(plan, windowMBps, s);
    return err != 0 ? err : Signal(mask, maskValue, s);
}

extern "C" int mfk_xcopy_signal(void *word, uint32_t value, void *stream)
{
    return mf::Signal(word, value, static_cast<hipStream_t>(stream));
}

namespace mf {
namespace {

bool IsList(const void *pieces, uint32_t count)
{
    return pieces != nullptr && count != 0 && count <= kPieceMaxCount;
}

// In the form that `units` and the hold ask for, or in windows of windowMBps where that is not 0, whose read part is `reading` 64ths of a period (0: half of it).
int SubmitPieceList(const void *pieces, uint32_t count, uint64_t bytes, uint32_t units, uint32_t holdNanos, uint32_t windowMBps, uint32_t reading, hipStream_t s,
                    hipEvent_t end, void *word, uint32_t value, void *counter)
{
    if (!IsList(pieces, count) || (units != 256 && units != 512 && units != 1024)) {
        return -1;
    }
    if (windowMBps != 0) {
        // whole groups of pieces, evenly over the rounds; the last group of the list may be short
        const uint32_t grid = (WindowGrid(count, kLongWaves) + kPieceGroup - 1) / kPieceGroup * kPieceGroup;
        const uint32_t period = WindowPeriodTicks(2 * bytes * grid / (count > grid ? count : grid), windowMBps);
        return period == 0 ? static_cast<int>(hipErrorInvalidValue)
                           : LaunchWithEvent(XcopyPieceWindowKernel, grid, 64, s, end, At(pieces), count, period,
                                             reading == 0 ? period / 2 : period / 64 * reading, NextWindowSeq(), grid, value, At(word));
    }
    const uint32_t ticks = HoldTicks(PieceHoldNanos(holdNanos, count, bytes, units));
    if (units == 256) {
        return ticks != 0 ? LaunchPieces(XcopyPieceKernel<64, 4, true>, 64, pieces, count, ticks, s, end, word, value, counter)
                          : LaunchPieces(XcopyPieceKernel<64, 4, false>, 64, pieces, count, 0, s, end, word, value, counter);
    }
    if (units == 512) {
        return ticks != 0 ? LaunchPieces(XcopyPieceKernel<128, 4, true>, 128, pieces, count, ticks, s, end, word, value, counter)
                          : LaunchPieces(XcopyPieceKernel<128, 4, false>, 128, pieces, count, 0, s, end, word, value, counter);
    }
    return ticks != 0 ? LaunchPieces(XcopyPieceHeldKernel, 64, pieces, count, ticks, s, end, word, value, counter)
                      : LaunchPieces(XcopyPieceKernel<256, 4, false>, 256, pieces, count, 0, s, end, word, value, counter);
}

}  // namespace
}  // namespace mf

// pieces: `count` mf::Piece of together `bytes` bytes, none longer than `units` units and the bytes beside them; holdNanos: what a
// table of as many chunks would wait.
extern "C" int mfk_xcopy_pieces(const void *pieces, uint32_t count, uint64_t bytes, uint32_t units, void *mask, uint32_t maskValue,
                                void *stream, uint32_t holdNanos, void *event)
{
    using namespace mf;
    hipStream_t s = static_cast<hipStream_t>(stream);
    const int err = SubmitPieceList(pieces, count, bytes, units, holdNanos, 0, 0, s, static_cast<hipEvent_t>(event), nullptr, 0, nullptr);
    return err != 0 ? err : Signal(mask, maskValue, s);
}

// The same, in either form, with a word of pinned host memory that gets `value`: when what is in front of them in the stream has ended
// or, with a counter (kDoneCounterBytes of device memory, 0; not in windows), when they have been read.
extern "C" int mfk_xcopy_pieces_reported(const void *pieces, uint32_t count, uint64_t bytes, uint32_t units, uint32_t holdNanos,
                                         uint32_t windowMBps, uint32_t reading, void *word, uint32_t value, void *counter, void *stream)
{
    if (word == nullptr || (counter != nullptr && windowMBps != 0)) {
        return -1;
    }
    return mf::SubmitPieceList(pieces, count, bytes, units, holdNanos, windowMBps, reading, static_cast<hipStream_t>(stream), nullptr, word, value,
                               counter);
}

// The same of 4 KiB and their bytes beside; the last of them stores `value` in `word`.  counter: kDoneCounterBytes of device memory.
extern "C" int mfk_xcopy_pieces_done(const void *pieces, uint32_t count, void *word, uint32_t value, void *counter, void *stream)
{
    using namespace mf;
    if (!IsList(pieces, count) || word == nullptr || counter == nullptr) {
        return -1;
    }
    return Launch(XcopyPieceDoneKernel, (count + kPieceGroup - 1) / kPieceGroup * kPieceGroup, 64, 0, static_cast<hipStream_t>(stream), At(pieces),
                  count, At(word), At(counter), value);
}

// The same pieces, of up to kWindowUnits units, in windows cut for windowMBps.
extern "C" int mfk_xcopy_pieces_windowed(const void *pieces, uint32_t count, uint64_t bytes, uint32_t windowMBps, uint32_t reading, void *mask,
                                         uint32_t maskValue, void *stream, void *event)
{
    using namespace mf;
    hipStream_t s = static_cast<hipStream_t>(stream);
    const int err = windowMBps == 0 ? -1 : SubmitPieceList(pieces, count, bytes, kWindowUnits, 0, windowMBps, reading, s, static_cast<hipEvent_t>(event),
                                                            nullptr, 0, nullptr);
    return err != 0 ? err : Signal(mask, maskValue, s);
}

extern "C" int mfk_xcopy_table(const void *tablePlan, int route, uint32_t grid, void *mask, uint32_t maskValue, void *stream)
{
    const mf::TablePlan &plan = *static_cast<const mf::TablePlan *>(tablePlan);
    const mf::ChunkPattern &pat = plan.pattern;
    if (plan.nseg == 0 || grid == 0 || plan.triples == nullptr) {
        return -1;
    }
    if (pat.period == 0 && (plan.first == nullptr || plan.group == nullptr || plan.groupShift < mf::kGroupShiftMin ||
                            plan.groupShift > 31)) {
        return -1;
    }
    if (pat.period != 0 && (pat.period > mf::kMaxPeriod || pat.chunksPerPeriod == 0 || pat.start[0] != 0 ||
                            pat.start[pat.period] != pat.chunksPerPeriod || mf::PatternChunks(pat, plan.nseg) != plan.nchunk)) {
        return -1;
    }
    hipStream_t s = static_cast<hipStream_t>(stream);
    const int err = mf::WithPolicy(mf::PolicyOf(route), [&](auto ntLoad, auto store) {
        hipLaunchKernelGGL((mf::XcopyTableKernel<decltype(ntLoad)::value, decltype(store)::value>), dim3(grid),
                           dim3(mf::LanesFor(plan.units, route)), 0, s, plan);
        return static_cast<int>(hipGetLastError());
    });
    return err != 0 ? err : mf::Signal(mask, maskValue, s);
}

// rest: a RestList with room for `capacity` segments, its counts 0.
extern "C" int mfk_xcopy_direct(const void *triples, uint32_t nseg, uint32_t units, int route, uint32_t grid, uint32_t restGrid, void *rest,
                                uint32_t capacity, uint32_t windowMBps, void *mask, uint32_t maskValue, void *stream, void *event)
{
    using namespace mf;
    if (nseg == 0 || nseg > capacity || grid == 0 || restGrid == 0 || rest == nullptr) {
        return -1;
    }
    hipStream_t s = static_cast<hipStream_t>(stream);
    // (grid: the waves that are paced have to be there)
    const bool sampled = windowMBps != 0 && route == MFRT_ROUTE_HBM && nseg > kPlannedSegments && grid >= kHeldMaxPieces;
    const TablePace pace = sampled ? PaceOf(0, 0, windowMBps, true) : TablePace{};
    const int err = WithPolicy(PolicyOf(route), [&](auto ntLoad, auto store) {
        return LaunchDirect<decltype(ntLoad)::value, decltype(store)::value>(static_cast<const uint64_t *>(triples), nseg, units, grid, restGrid,
                                                                             LanesFor(units, route), static_cast<RestList *>(rest), capacity, s,
                                                                             static_cast<hipEvent_t>(event), sampled && pace.windowTicks != 0 ? &pace : nullptr);
    });
    return err != 0 ? err : Signal(mask, maskValue, s);
}

extern "C" int mfk_xcopy_planned(const void *triples, uint32_t nseg, uint32_t holdNanos, uint32_t holdMoreNanos, uint32_t windowMBps, void *mask,
                                 uint32_t maskValue, void *stream)
{
    using namespace mf;
    if (triples == nullptr || nseg == 0 || nseg > kPlannedSegments) {
        return -1;
    }
    hipStream_t s = static_cast<hipStream_t>(stream);
    const TablePace pace = PaceOf(holdNanos, holdMoreNanos, windowMBps, false);
    const int err = nseg <= 64 * kPlannedShortRun
                        ? Launch(XcopyPlannedKernel<1, kPlannedShortRun>, kWindowWaves, 64, PlannedLds(1, nseg), s, At(triples), nseg, pace)
                        : Launch(XcopyPlannedKernel<kPlannedWaves, kPlannedRun>, kWindowWaves / kPlannedWaves, 64 * kPlannedWaves,
                                 PlannedLds(kPlannedWaves, nseg), s, At(triples), nseg, pace);
    return err != 0 ? err : Signal(mask, maskValue, s);
}

// Makes `count` lists `stride` bytes apart empty.
extern "C" int mfk_xcopy_clear_lists(void *lists, uint32_t count, uint64_t stride, void *stream)
{
    using namespace mf;
    hipLaunchKernelGGL(XcopyClearListsKernel, dim3(count), dim3(64), 0, static_cast<hipStream_t>(stream), static_cast<uint8_t *>(lists), stride);
    return static_cast<int>(hipGetLastError());
}

// Every copy kernel once, on plans that hold nothing, so that a caller who captures a stream later finds the code of
// this file loaded and every kernel known to the runtime (a kernel's first launch is not capturable).
extern "C" int mfk_xcopy_prelaunch(void *stream)
{
    using namespace mf;
    hipStream_t s = static_cast<hipStream_t>(stream);
    InlinePlan empty{};
    for (uint32_t i = 0; i < kInlineSegs; ++i) {
        empty.first[i] = kNoChunk;
    }
    empty.units = kXcopyThreads;
    TablePlan none{};
    none.nseg = 1;
    none.units = kXcopyThreads;
    none.groupShift = kGroupShiftMin;
    // (the copies that store a word of their own are never captured: a blocking call cannot be)
    for (int route = MFRT_ROUTE_HBM; route <= MFRT_ROUTE_FROM_HOST; ++route) {
        (void)WithPolicy(PolicyOf(route), [&](auto ntLoad, auto store) {
            constexpr bool kNt = decltype(ntLoad)::value;
            constexpr int kSt = decltype(store)::value;
            hipLaunchKernelGGL((XcopyInlineKernel<kNt, kSt, kHoldNone>), dim3(1), dim3(64), 0, s, empty, 0u);
            hipLaunchKernelGGL((XcopySingleKernel<kNt, kSt, kHoldNone>), dim3(1), dim3(64), 0, s, 0ull, 0ull, 0u, 0u, kXcopyThreads, 0u, 64u, 1u, 0u);
            hipLaunchKernelGGL((XcopyTableKernel<kNt, kSt>), dim3(1), dim3(64), 0, s, none);
            if (route == MFRT_ROUTE_HBM) {
                hipLaunchKernelGGL((XcopyInlineKernel<kNt, kSt, kHoldShallow>), dim3(1), dim3(64), 0, s, empty, 1u);
                hipLaunchKernelGGL((XcopyInlineKernel<kNt, kSt, kHoldDeep>), dim3(1), dim3(64), 0, s, empty, 1u);
                hipLaunchKernelGGL((XcopySingleKernel<kNt, kSt, kHoldShallow>), dim3(1), dim3(64), 0, s, 0ull, 0ull, 0u, 0u, kXcopyThreads, 1u, 64u, 1u, 0u);
                (void)Launch(XcopySingleHeldKernel, 1, 64, 0, s, 0ull, 0ull, 0u, 1u);
                (void)Launch(XcopyPieceKernel<64, 4, false>, 1, 64, 0, s, 0, 0u, 0u, 0u, 0, 0);
                (void)Launch(XcopyPieceKernel<64, 4, true>, 1, 64, 0, s, 0, 0u, 0u, 0u, 0, 0);
                (void)Launch(XcopyPieceHeldKernel, 1, 64, 0, s, 0, 0u, 0u, 0u, 0, 0);
                (void)Launch(XcopyPieceKernel<128, 4, false>, 1, 128, 0, s, 0, 0u, 0u, 0u, 0, 0);
                (void)Launch(XcopyPieceKernel<128, 4, true>, 1, 128, 0, s, 0, 0u, 0u, 0u, 0, 0);
                (void)Launch(XcopyPieceKernel<256, 4, false>, 1, 256, 0, s, 0, 0u, 0u, 0u, 0, 0);
                (void)Launch(XcopyPieceDoneKernel, 1, 64, 0, s, 0, 0u, 0, 0, 0u);
                (void)Launch(XcopyPieceWindowKernel, 1, 64, 0, s, 0, 0u, 64u, 32u, NextWindowSeq(), 1u, 0u, 0);
                (void)Launch(XcopyPlannedKernel<1, kPlannedShortRun>, 1, 64, 64, s, 0, 0u, TablePace{});
                (void)Launch(XcopyPlannedKernel<kPlannedWaves, kPlannedRun>, 1, 64 * kPlannedWaves, 64, s, 0, 0u, TablePace{});
                (void)Launch(XcopySampledKernel, 1, 64, 0, s, 0, 0u, 0, 0u, TablePace{});
                hipLaunchKernelGGL(XcopyWindowKernel, dim3(1), dim3(64), 0, s, empty, 64u, NextWindowSeq());
            }
            return 0;
        });
    }
    return static_cast<int>(hipGetLastError());
}

// Calibration workloads, timed by events on `stream` (see XcopyEngine::Calibrate for what is chosen from them).
// out[0 .. 3]: microseconds per batch of 122 segments (61 x 128 KiB and 16 KiB in turn, 2196 chunks, 32 tables in turn
// inside 1 GiB of scratch) without a hold and held for holdNanos[0 .. 2]; out[4 .. 7]: microseconds per copy of 512 MiB by
// the kernel without windows and in windows cut for windowMBps[0 .. 2].  Batches: the fastest of three rounds of 128
// launches; copies: the fastest of six, each timed on its own.
extern "C" int mfk_xcopy_calibrate(void *stream, const uint32_t *holdNanos, const uint32_t *windowMBps, float *out)
{
    using namespace mf;
    hipStream_t s = static_cast<hipStream_t>(stream);
    const uint64_t half = 512ull << 20;
    char *scratchMem = nullptr;
    hipError_t err = hipMalloc(&scratchMem, 2 * half);
    if (err != hipSuccess) {
        return static_cast<int>(err);
    }
    hipEvent_t e0 = nullptr;
    hipEvent_t e1 = nullptr;
    auto release = [&](hipError_t code) {
        (void)hipStreamSynchronize(s);
        if (e0 != nullptr) {
            (void)hipEventDestroy(e0);
        }
        if (e1 != nullptr) {
            (void)hipEventDestroy(e1);
        }
        (void)hipFree(scratchMem);
        return static_cast<int>(code);
    };
    if ((err = hipMemsetAsync(scratchMem, 0x5A, 2 * half, s)) != hipSuccess || (err = hipEventCreate(&e0)) != hipSuccess ||
        (err = hipEventCreate(&e1)) != hipSuccess) {
        return release(err);
    }
    // 32 tables of K and V blocks, every block in a 128 KiB slot of its own: sources in the lower half, destinations in
    // the upper; together they touch 576 MB, more than the last-level cache holds, as a caller's batches do
    constexpr uint32_t kTables = 32;
    constexpr uint32_t kSlotsPerHalf = 4096;
    std::vector<InlinePlan> plans(kTables);
    const uint64_t base = reinterpret_cast<uint64_t>(scratchMem);
    for (uint32_t t = 0; t < kTables; ++t) {
        InlinePlan &plan = plans[t];
        uint32_t run = 0;
        for (uint32_t i = 0; i < kInlineSegs; ++i) {
            if (i < 122) {
                const uint32_t len = (i & 1u) != 0 ? 16384u : 131072u;
                const uint32_t at = t * 122 + i;
                plan.src[i] = base + static_cast<uint64_t>((at * 1103u + 17u) % kSlotsPerHalf) * (128u << 10);
                plan.dst[i] = base + half + static_cast<uint64_t>((at * 757u + 5u) % kSlotsPerHalf) * (128u << 10);
                plan.len[i] = len;
                plan.first[i] = run;
                run += len / 4096;
            } else {
                plan.src[i] = plan.dst[i] = 0;
                plan.len[i] = 0;
                plan.first[i] = kNoChunk;
            }
        }
        plan.nchunk = run;
        plan.units = kXcopyThreads;
    }
    InlinePlan big{};
    for (uint32_t i = 0; i < kInlineSegs; ++i) {
        big.first[i] = kNoChunk;
    }
    big.src[0] = base;
    big.dst[0] = base + half;
    big.len[0] = static_cast<uint32_t>(half);
    big.first[0] = 0;
    auto timed = [&](auto launch, int warm, int count, float &best) -> hipError_t {
        for (int i = 0; i < warm; ++i) {
            launch(i);
        }
        hipError_t code = hipEventRecord(e0, s);
        for (int i = 0; i < count && code == hipSuccess; ++i) {
            launch(i);
        }
        if (code == hipSuccess) {
            code = hipEventRecord(e1, s);
        }
        if (code == hipSuccess) {
            code = hipEventSynchronize(e1);
        }
        float ms = 0.0f;
        if (code == hipSuccess) {
            code = hipEventElapsedTime(&ms, e0, e1);
        }
        if (code == hipSuccess) {
            const float us = ms * 1000.0f / static_cast<float>(count);
            best = best == 0.0f || us < best ? us : best;
        }
        return code != hipSuccess ? code : hipGetLastError();
    };
    for (int i = 0; i < 8; ++i) {
        out[i] = 0.0f;
    }
    for (int round = 0; round < 3; ++round) {
        for (int v = 0; v < 4; ++v) {
            const uint32_t nanos = v == 0 ? 0u : holdNanos[v - 1];
            err = timed([&](int i) { (void)LaunchInline<true, kStoreStream>(plans[i % kTables], plans[0].nchunk, 64, s, false, nanos); }, 32, 128,
                        out[v]);
            if (err != hipSuccess) {
                return release(err);
            }
        }
    }
    // Every copy is timed on its own and the fastest of six counts: a windowed launch now and then loses its schedule part of
    // the way, at any rate, and the question here is whether this GPU holds the rate at all (two launches timed together,
    // three times, once gave 156.6 us for a rate whose launches otherwise take 148.4: one more such sample and the process
    // would have run at the lower rate for good).
    for (int round = 0; round < 6; ++round) {
        for (int v = 0; v < 4; ++v) {
            if (v == 0) {
                big.units = kXcopyThreads;
                big.nchunk = static_cast<uint32_t>(half / (kXcopyThreads * kUnitBytes));
                err = timed([&](int) { (void)LaunchInline<true, kStoreStream>(big, big.nchunk, 64, s, false, 0); }, round == 0 ? 1 : 0, 1, out[4]);
            } else {
                big.units = kWindowUnits;
                big.nchunk = static_cast<uint32_t>(half / (kWindowUnits * kUnitBytes));
                const uint32_t rate = windowMBps[v - 1];
                err = timed([&](int) { (void)LaunchWindowed(big, rate, s); }, round == 0 ? 1 : 0, 1,
                            out[4 + v]);
            }
            if (err != hipSuccess) {
                return release(err);
            }
        }
    }
    return release(hipSuccess);
}

#ifndef MF_RT_HIDDEN   // the plugin library has no entry point that needs it
// List of the entry point that allocates nothing (mfk_xcopy_table_static), with room for every segment of the longest table.  One copy per GPU, zero when its code is loaded and
// held until the process ends.  In host code the array's name is only a handle for hipGetSymbolAddress: kernels get the
// address that call returned for the current device, never the name.
constexpr uint32_t kStaticRestCapacity = MFK_STATIC_TABLE_SEGMENTS;
static __device__ __align__(256) uint32_t scratch[mf::RestListBytes(kStaticRestCapacity) / 4];

namespace {
constexpr int kMaxDevices = 64;
uint32_t *g_scratchOf[kMaxDevices] = {};   // device ordinal -> address of that device's copy of `scratch`
// Calls on one GPU share the array.  The host side keeps them apart where it can without allocating: an event made at
// set-up is recorded behind every call, and a call that comes on another stream than the one before first makes its
// stream wait for that event.  Calls under stream capture are outside this (an event recorded there belongs to the graph).
hipEvent_t g_staticDone[kMaxDevices] = {};
hipStream_t g_staticLast[kMaxDevices] = {};
bool g_staticUsed[kMaxDevices] = {};
std::mutex g_staticLock;
}  // namespace

extern "C" int mfk_xcopy_static_setup(void)
{
    int dev = -1;
    hipError_t err = hipGetDevice(&dev);
    if (err != hipSuccess) {
        return static_cast<int>(err);
    }
    if (dev < 0 || dev >= kMaxDevices) {
        return static_cast<int>(hipErrorInvalidDevice);
    }
    void *ptr = nullptr;
    err = hipGetSymbolAddress(&ptr, HIP_SYMBOL(scratch));
    if (err != hipSuccess) {
        return static_cast<int>(err);
    }
    g_scratchOf[dev] = static_cast<uint32_t *>(ptr);
    if (g_staticDone[dev] == nullptr && hipEventCreateWithFlags(&g_staticDone[dev], hipEventDisableTiming) != hipSuccess) {
        g_staticDone[dev] = nullptr;   // calls then go unguarded, as documented for callers that overlap them
        (void)hipGetLastError();
    }
    // The kernels of the device-table path once, on a table of no segments (what mfk_xcopy_prelaunch cannot do without device
    // memory): a caller may then capture its very first call.
    {
        using namespace mf;
        uint32_t *words = g_scratchOf[dev];
        RestList *rest = reinterpret_cast<RestList *>(words);
        const uint64_t *none = reinterpret_cast<const uint64_t *>(words);
        (void)Launch(XcopySignalKernel, 1, 64, 0, nullptr, At(rest->reserved), 0u);
        hipLaunchKernelGGL(XcopyClearListsKernel, dim3(1), dim3(64), 0, nullptr, reinterpret_cast<uint8_t *>(rest), 0ull);
        for (int route = MFRT_ROUTE_HBM; route <= MFRT_ROUTE_FROM_HOST; ++route) {
            (void)WithPolicy(PolicyOf(route), [&](auto ntLoad, auto store) {
                return LaunchDirect<decltype(ntLoad)::value, decltype(store)::value>(none, 0, kXcopyThreads, 1, 1, 64, rest,
                                                                                     kStaticRestCapacity, nullptr, nullptr);
            });
        }
        err = hipGetLastError();
        if (err == hipSuccess) {
            err = hipStreamSynchronize(nullptr);
        }
        if (err != hipSuccess) {
            return static_cast<int>(err);
        }
    }
    return 0;
}

extern "C" int mfk_xcopy_table_static(const void *triples, uint32_t nseg, uint32_t units, int route, uint32_t grid, uint32_t restGrid,
                                      void *stream)
{
    if (nseg == 0 || nseg > MFK_STATIC_TABLE_SEGMENTS || grid == 0) {
        return -1;
    }
    int dev = -1;
    if (hipGetDevice(&dev) != hipSuccess || dev < 0 || dev >= kMaxDevices || g_scratchOf[dev] == nullptr) {
        return -2;   // mfk_xcopy_static_setup has not run on this device
    }
    std::lock_guard<std::mutex> guard(g_staticLock);
    hipStream_t s = static_cast<hipStream_t>(stream);
    hipStreamCaptureStatus capture = hipStreamCaptureStatusNone;
    const bool capturing = hipStreamIsCapturing(s, &capture) == hipSuccess && capture != hipStreamCaptureStatusNone;
    const bool guarded = !capturing && g_staticDone[dev] != nullptr;
    if (guarded && g_staticUsed[dev] && g_staticLast[dev] != s && hipStreamWaitEvent(s, g_staticDone[dev], 0) != hipSuccess) {
        return static_cast<int>(hipGetLastError());
    }
    const int err = mfk_xcopy_direct(triples, nseg, units, route, grid, restGrid, g_scratchOf[dev], kStaticRestCapacity, 0, nullptr, 0, stream,
                                     nullptr);
    if (guarded && hipEventRecord(g_staticDone[dev], s) == hipSuccess) {
        g_staticLast[dev] = s;
        g_staticUsed[dev] = true;
    }
    return err;
}
#endif  // MF_RT_HIDDEN
