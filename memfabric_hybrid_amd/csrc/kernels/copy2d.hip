// Batched strided 2-D copy for gfx950: up to 64 rectangles per launch, work cut
// into groups of rows of about 16 KiB so that narrow rows (a few hundred bytes)
// still fill every lane with 128-bit accesses, or from 32 MiB on into chunks of
// the payload.  HBM bound, 2 bytes of traffic per payload byte; no LDS, no MFMA.
#include <hip/hip_runtime.h>
#include <stdint.h>

#include "../rt/mf_rt.h"
#include "copy2d_plan.h"
#include "launch.h"
#include "window_clock.h"

namespace mf {
namespace {

typedef uint32_t u32x4 __attribute__((ext_vector_type(4)));
#define MF_GLOBAL __attribute__((address_space(1)))

__device__ __forceinline__ uint64_t ReadLane64(uint64_t v, uint32_t lane)
{
    const uint32_t lo = __builtin_amdgcn_readlane(static_cast<uint32_t>(v), lane);
    const uint32_t hi = __builtin_amdgcn_readlane(static_cast<uint32_t>(v >> 32), lane);
    return (static_cast<uint64_t>(hi) << 32) | lo;
}

__global__ __launch_bounds__(kRectThreads) void Copy2dKernel(const RectPlan p)
{
    // the whole rectangle table in registers after one round trip, one row per lane
    const uint32_t lane = threadIdx.x & 63u;
    const uint32_t first = p.first[lane];
    const uint64_t src = p.src[lane];
    const uint64_t dst = p.dst[lane];
    const uint32_t sp = p.spitchUnits[lane];
    const uint32_t dp = p.dpitchUnits[lane];
    const uint32_t wu = p.widthUnits[lane];
    const uint32_t ht = p.height[lane];
    const uint32_t rpc = p.rowsPerChunk[lane];
    const uint32_t mg = p.magic[lane];
    const uint32_t mt = p.mate[lane];
    const uint32_t nchunk = p.nchunk;
    uint32_t c = blockIdx.x;
    do {
        // Two rectangles side by side in the destination take the chunks of their common range in turn, so that
        // workgroups launched together write both parts of the same destination rows.
        uint32_t r = __popcll(__ballot(first <= c)) - 1;
        uint32_t k = c - __builtin_amdgcn_readlane(first, r);
        const uint32_t m = __builtin_amdgcn_readlane(mt, r);
        if (m != 0) {
            const uint32_t r0 = r - (m - 1);
            const uint32_t both = c - __builtin_amdgcn_readlane(first, r0);
            r = r0 + (both & 1u);
            k = both >> 1;
        }
        const uint64_t rs = ReadLane64(src, r);
        const uint64_t rd = ReadLane64(dst, r);
        const uint32_t rsp = __builtin_amdgcn_readlane(sp, r);
        const uint32_t rdp = __builtin_amdgcn_readlane(dp, r);
        const uint32_t rwu = __builtin_amdgcn_readlane(wu, r);
        const uint32_t rht = __builtin_amdgcn_readlane(ht, r);
        const uint32_t rrpc = __builtin_amdgcn_readlane(rpc, r);
        const uint32_t rmg = __builtin_amdgcn_readlane(mg, r);
        const uint32_t row0 = k * rrpc;
        const uint32_t rows = rht - row0 < rrpc ? rht - row0 : rrpc;
        const uint32_t units = rows * rwu;
        const MF_GLOBAL u32x4 *s = reinterpret_cast<const MF_GLOBAL u32x4 *>(rs) + static_cast<uint64_t>(row0) * rsp;
        MF_GLOBAL u32x4 *d = reinterpret_cast<MF_GLOBAL u32x4 *>(rd) + static_cast<uint64_t>(row0) * rdp;
        for (uint32_t u0 = 0; u0 < units; u0 += 4 * kRectThreads) {
            u32x4 v[4];
            uint32_t row[4];
            uint32_t col[4];
#pragma unroll
            for (uint32_t j = 0; j < 4; ++j) {
                const uint32_t u = u0 + j * kRectThreads + threadIdx.x;
                RectRowCol(u, rwu, rrpc, rmg, row[j], col[j]);
                if (u < units) {
                    v[j] = __builtin_nontemporal_load(s + static_cast<uint64_t>(row[j]) * rsp + col[j]);
                }
            }
#pragma unroll
            for (uint32_t j = 0; j < 4; ++j) {
                const uint32_t u = u0 + j * kRectThreads + threadIdx.x;
                if (u < units) {
                    __builtin_nontemporal_store(v[j], d + static_cast<uint64_t>(row[j]) * rdp + col[j]);
                }
            }
        }
        c += gridDim.x;
    } while (c < nchunk);
}

// Rectangles in chunks of their payload (RectChunkPlan).  HBM bounds it.  A chunk of 4 KiB or 16 KiB of the payload is whole cache lines
// of the destination wherever its rows lie against one another, those of a pair included, where groups of whole rows, and the two
// halves of a pair's rows written by workgroups apart, end inside a line whenever the width is not a multiple of 128 bytes.
// us per launch, back to back on buffers that no cache holds, whole rows (Copy2dKernel) / 4 KiB chunks / in windows cut for 6.8 TB/s:
// pairs of 896 and 4736 bytes, 161 MB 57.5 / - / 51.4, 646 MB 215 / - / 200; of 480 and 2992, 107 MB 45.6 / 38.2 / 34.7, 213 MB 87.6 / - / 67.7; of
// 736 and 1888, 62 MB 27.0 / 23.7 / 21.3, 247 MB 99.3 / 81.4 / 77.2.  Single rectangles of 896 or 4736 bytes a row with strided source,
// strided destination or both, 40 MB 17.1 to 17.8 / 16.6 to 17.0 / 14.9 to 15.2, 400 MB 134 to 146 / 129 to 133 / 123 to 129; rows of 480, 2992 or
// 20 000 bytes, 400 MB 147 to 197 / 129 to 190 / 126 to 201: which rows go without windows is RectHolds.  Below 32 MiB whole rows are as fast or faster (24 MB
// 9.0 to 9.5 / 11.2 to 11.6 / 10.1 to 10.7).
// kPaced: sixteen loads per lane at the wave's offset into the read half of the period, the stores at the same offset into the
// write half, as XcopyWindowKernel does for long segments.  Rates of 7.1 TB/s and more fall apart for half of these geometries;
// uneven parts lose (a read part of 0.42 / 0.45 / 0.475 / 0.5 / 0.525 / 0.55 / 0.58 of a period at 7.0, 161 MB 56.2 / 54.5 / 51.4 / 50.8 / 51.0 / 54.1 / 59.4).
template <bool kPaced>
__global__ __launch_bounds__(64) __attribute__((amdgpu_waves_per_eu(kPaced ? 5 : 8))) void Copy2dChunkKernel(const RectChunkPlan p, uint32_t groups,
                                                                                                        uint32_t period, uint32_t seq)
{
    constexpr uint32_t kDepth = kPaced ? kRectWindowDepth : kRectChunkDepth;
    constexpr uint32_t kUnits = 64 * kDepth;
    // Only what the search needs stays in vector registers; the rectangle a chunk belongs to is read from the
    // argument block by scalar loads once it is known (a period is microseconds long, their latency does not show).
    const uint32_t lane = threadIdx.x & 63u;
    const uint32_t first = p.first[lane];
    const uint32_t nchunk = p.nchunk;
    const uint32_t half = period / 2;
    uint64_t slot = kPaced ? AgreedStart(seq) + static_cast<uint64_t>(blockIdx.x) * half / groups : 0;
    for (uint32_t c = blockIdx.x; c < nchunk; c += groups) {
        const uint32_t r = (__popcll(__ballot(first <= c)) - 1) & (kRectInline - 1);
        const uint32_t base = (c - __builtin_amdgcn_readlane(first, r)) * kUnits;
        const uint32_t sp = p.spitchUnits[r];
        const uint32_t dp = p.dpitchUnits[r];
        const uint32_t split = p.halfUnits[r];
        const uint32_t ru = p.rowUnits[r];
        const uint32_t mg = p.magic[r];
        const uint32_t left = p.height[r] * ru - base;
        const uint32_t n = left < kUnits ? left : kUnits;
        const uint32_t row0 = base / ru;
        const uint64_t down = static_cast<uint64_t>(row0) * sp;
        const MF_GLOBAL u32x4 *s = reinterpret_cast<const MF_GLOBAL u32x4 *>(p.src[r]) + down;
        const MF_GLOBAL u32x4 *o = reinterpret_cast<const MF_GLOBAL u32x4 *>(p.other[r]) + down - split;
        MF_GLOBAL u32x4 *d = reinterpret_cast<MF_GLOBAL u32x4 *>(p.dst[r]) + static_cast<uint64_t>(row0) * dp;
        // Row and column of a unit are worked out where its address is needed, before the loads and again before the
        // stores, from a lane offset the compiler cannot see through: kept across the waits (or worked out ahead of them,
        // as it prefers) sixteen rows or thirty-two addresses beside the data take the kernel past the registers at which
        // all kRectWindowWaves waves are resident together with room to spare, which the schedule needs.
        uint32_t x0 = base - row0 * ru + lane;
        auto load = [&](uint32_t j) -> u32x4 {
            uint32_t row;
            uint32_t col;
            RectWindowRowCol(x0 + j * 64, ru, mg, row, col);
            const MF_GLOBAL u32x4 *from = col < split ? s : o;
            return __builtin_nontemporal_load(from + (static_cast<uint64_t>(row) * sp + col));
        };
        auto store = [&](uint32_t j, u32x4 v) {
            uint32_t row;
            uint32_t col;
            RectWindowRowCol(x0 + j * 64, ru, mg, row, col);
            __builtin_nontemporal_store(v, d + (static_cast<uint64_t>(row) * dp + col));
        };
        auto between = [&] {
            if (kPaced) {
                asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
                WaitForClock(slot + half);
            }
            asm volatile("" : "+v"(x0));
        };
        u32x4 v[kDepth];
        if (kPaced) {
            WaitForClock(slot);
        }
        asm volatile("" : "+v"(x0));
        if (n == kUnits) {
#pragma unroll
            for (uint32_t j = 0; j < kDepth; ++j) {
                v[j] = load(j);
            }
            between();
#pragma unroll
            for (uint32_t j = 0; j < kDepth; ++j) {
                store(j, v[j]);
            }
        } else {
#pragma unroll
            for (uint32_t j = 0; j < kDepth; ++j) {
                if (j * 64 + lane < n) {
                    v[j] = load(j);
                }
            }
            between();
#pragma unroll
            for (uint32_t j = 0; j < kDepth; ++j) {
                if (j * 64 + lane < n) {
                    store(j, v[j]);
                }
            }
        }
        slot += period;
    }
}

}  // namespace
}  // namespace mf

// In windows cut for windowMBps over chunks of kRectWindowUnits units or, with 0, in chunks of kRectChunkDepth loads per lane.
extern "C" int mfk_copy2d_chunks(const void *rectChunkPlan, uint32_t windowMBps, void *stream)
{
    using namespace mf;
    const RectChunkPlan &plan = *static_cast<const RectChunkPlan *>(rectChunkPlan);
    hipStream_t s = static_cast<hipStream_t>(stream);
    if (plan.nchunk == 0) {
        return 0;
    }
    if (windowMBps == 0) {
        constexpr uint32_t kMost = (1u << 24) - 1;   // the grid size in lanes must stay below 2^32; workgroups loop over the rest
        const uint32_t grid = plan.nchunk < kMost ? plan.nchunk : kMost;
        return Launch(Copy2dChunkKernel<false>, grid, 64, 0, s, plan, grid, 0u, 0u);
    }
    const uint32_t grid = WindowGrid(plan.nchunk, kRectWindowWaves);
    const uint32_t ticks = WindowPeriodTicks(2ull * grid * kRectWindowUnits * 16u, windowMBps);
    if (ticks == 0) {
        return static_cast<int>(hipErrorInvalidValue);
    }
    return Launch(Copy2dChunkKernel<true>, grid, 64, 0, s, plan, grid, ticks, NextWindowSeq());
}

// Every kernel once on a plan that holds nothing: a kernel's first launch is not capturable.
extern "C" int mfk_copy2d_prelaunch(void *stream)
{
    mf::RectPlan empty{};
    for (uint32_t i = 0; i < mf::kRectInline; ++i) {
        empty.first[i] = 0xFFFFFFFFu;
        empty.rowsPerChunk[i] = 1;
    }
    hipLaunchKernelGGL(mf::Copy2dKernel, dim3(1), dim3(mf::kRectThreads), 0, static_cast<hipStream_t>(stream), empty);
    mf::RectChunkPlan none{};
    for (uint32_t i = 0; i < mf::kRectInline; ++i) {
        none.first[i] = 0xFFFFFFFFu;
    }
    (void)mf::Launch(mf::Copy2dChunkKernel<false>, 1, 64, 0, static_cast<hipStream_t>(stream), none, 1u, 0u, 0u);
    (void)mf::Launch(mf::Copy2dChunkKernel<true>, 1, 64, 0, static_cast<hipStream_t>(stream), none, 1u, 64u, mf::NextWindowSeq());
    return static_cast<int>(hipGetLastError());
}

extern "C" int mfk_copy2d(const void *rectPlan, uint32_t grid, void *stream)
{
    const mf::RectPlan &plan = *static_cast<const mf::RectPlan *>(rectPlan);
    if (plan.nchunk == 0) {
        return 0;
    }
    if (grid == 0 || grid > plan.nchunk) {
        grid = plan.nchunk;
    }
    if (grid > (1u << 24) - 1) {
        grid = (1u << 24) - 1;   // the grid size in lanes must stay below 2^32; workgroups loop over the rest
    }
    hipLaunchKernelGGL(mf::Copy2dKernel, dim3(grid), dim3(mf::kRectThreads), 0, static_cast<hipStream_t>(stream), plan);
    return static_cast<int>(hipGetLastError());
}
