// Copies between a ring of slots in pinned host memory and HBM that run while the CPU fills or empties the ring.
//
// A launch moves the chunks of 4 MiB, the launches of a copy follow one another without a gap.  Workgroup g takes the chunks g, g + groups, ...; chunk
// c uses slot c % slots.  Each side says in a word per slot, on a line of its own, which chunk it has finished there (base + c + 1).  On the
// way to HBM the GPU waits for the chunk to be filled; to the host it waits for nothing, the host launches no more chunks than there are slots free.
// The GPU's waits end after limitTicks of the constant-rate clock: a workgroup then leaves, the host finds that nothing of the
// launch is left and copies another way.
// Bound: the host link, 56 to 57 GB/s.  A launch a round of up to 8 MiB instead, filled or emptied by the CPU as a whole, waits for the CPU at one
// end of the copy, and for a launch and its completion word in every round.
#include <hip/hip_ext.h>
#include <hip/hip_runtime.h>
#include <stdint.h>

#include "../rt/mf_rt.h"
#include "launch.h"
#include "staging.h"
#include "through.h"

namespace mf {
namespace {

typedef uint32_t u32x4 __attribute__((ext_vector_type(4)));
#define MF_GLOBAL __attribute__((address_space(1)))

constexpr uint32_t kStreamThreads = 512;
constexpr uint32_t kStreamUnits = kStreamChunkBytes / (16 * kStreamThreads);     // 128-bit accesses per lane
// Few enough that a chunk is done soon after it was begun, which is what the CPU waits for at the end of a copy to it, or from its start on to
// the host; enough that the link always has some to move.  us with 8 / 12 / 16 / 24 / 32 groups, to the GPU 2 MiB 64 / 58 / 57 / 54 / 54, 16 MiB 375 / 369 / 338 /
// 344 / 354, 64 MiB 1415 / 1384 / 1264 / 1261 / 1269; to the host 2 MiB 56 / 56 / 59 / 65 / 68, 8 MiB in 20 parts 172 / 183 / 192 / 206 / 215.  Chunks of 32 KiB in workgroups of
// 256 lanes, the best of 4 to 96: 52, 344 and 1288; 56 and 175; of 16 KiB 54, 361 and 1415; of 64 KiB in 1024 lanes 64, 400 and 1517.
// As many on each of the eight XCDs: 64 MiB to the GPU with 16 / 20 / 32 1260 / 1304 / 1273.
constexpr uint32_t kStreamGroupsIn = 16;
constexpr uint32_t kStreamGroupsOut = 8;

__device__ __forceinline__ uint64_t ReadWord(uint64_t at)
{
    return __hip_atomic_load(Buffer<uint64_t>(at), __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_SYSTEM);
}

__device__ __forceinline__ void CopyByteThrough(uint64_t src, uint64_t dst)
{
    StoreThrough1(dst, *reinterpret_cast<const MF_GLOBAL uint8_t *>(src));
}

// `len` bytes between addresses that agree modulo kStreamLine, in units counted from the line they begin in; with what lies in front of
// them in that line they are at most kStreamChunkBytes.
__device__ __forceinline__ void CopyChunkThrough(uint64_t src, uint64_t dst, uint32_t len)
{
    const uint32_t skip = static_cast<uint32_t>(dst) & (kStreamLine - 1);
    const uint64_t s = src - skip;
    const uint64_t d = dst - skip;
    const uint32_t end = skip + len;
    const uint32_t first = (skip + 15) / 16;        // whole units [first, last)
    const uint32_t last = end / 16;
    if (first < last) {
        // what a lane past either end loads is the unit there
        u32x4 v[kStreamUnits];
#pragma unroll
        for (uint32_t j = 0; j < kStreamUnits; ++j) {
            const uint32_t u = j * kStreamThreads + threadIdx.x;
            const uint32_t upTo = u < last ? u : last - 1;
            v[j] = __builtin_nontemporal_load(reinterpret_cast<const MF_GLOBAL u32x4 *>(s + (upTo > first ? upTo : first) * 16));
        }
        asm volatile("" ::: "memory");      // all of them first: a load that moves to its store waits for the others
#pragma unroll
        for (uint32_t j = 0; j < kStreamUnits; ++j) {
            const uint32_t u = j * kStreamThreads + threadIdx.x;
            if (u >= first && u < last) {
                StoreThrough16(d + u * 16, v[j]);
            }
        }
    }
    // bytes in front of the first whole unit, and behind the last
    const uint32_t headEnd = first * 16 < end ? first * 16 : end;
    const uint32_t tailFrom = last * 16 > headEnd ? last * 16 : headEnd;
    if (threadIdx.x < 16 && skip + threadIdx.x < headEnd) {
        CopyByteThrough(s + skip + threadIdx.x, d + skip + threadIdx.x);
    }
    if (threadIdx.x < 16 && tailFrom + threadIdx.x < end) {
        CopyByteThrough(s + tailFrom + threadIdx.x, d + tailFrom + threadIdx.x);
    }
}

template <bool kToHost>
__global__ __launch_bounds__(kStreamThreads) void StreamChunksKernel(uint64_t ring, uint64_t chunks, uint64_t hostWords, uint64_t gpuWords,
                                                                     uint64_t base, uint32_t count, uint32_t slots, uint32_t groups,
                                                                     uint32_t limitTicks)
{
    __shared__ uint32_t ready;
    const MF_GLOBAL StreamChunk *list = reinterpret_cast<const MF_GLOBAL StreamChunk *>(chunks);
#pragma unroll 1
    for (uint32_t c = blockIdx.x; c < count; c += groups) {
        const uint32_t slot = c % slots;
        const uint64_t at = list[c].at;
        const uint32_t len = list[c].len;
        if (!kToHost) {
            if (threadIdx.x == 0) {
                const uint64_t wanted = base + c + 1;
                const uint64_t start = wall_clock64();
                uint64_t seen = ReadWord(hostWords + static_cast<uint64_t>(slot) * kStreamWordBytes);
                while (seen != wanted && wall_clock64() - start < limitTicks) {
                    __builtin_amdgcn_s_sleep(8);
                    seen = ReadWord(hostWords + static_cast<uint64_t>(slot) * kStreamWordBytes);
                }
                ready = seen == wanted ? 1 : 0;
            }
            __syncthreads();
            if (ready == 0) {
                return;
            }
            __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "");       // nothing of the slot from before, in whatever cache
        }
        const uint64_t there = ring + static_cast<uint64_t>(slot) * kStreamChunkBytes + (at & (kStreamLine - 1));
        if (kToHost) {
            CopyChunkThrough(at, there, len);
        } else {
            CopyChunkThrough(there, at, len);
        }
        asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
        __syncthreads();
        if (threadIdx.x == 0) {
            __hip_atomic_store(Buffer<uint64_t>(gpuWords + static_cast<uint64_t>(slot) * kStreamWordBytes), base + c + 1, __ATOMIC_RELAXED,
                               __HIP_MEMORY_SCOPE_SYSTEM);
        }
    }
}

}  // namespace
}  // namespace mf

// Both kernels once, on no chunks: what a first launch costs, this file's code has to be loaded for it, is not paid in a copy, whose helpers
// would wait for it.
extern "C" int mfk_stream_prelaunch(void *stream)
{
    using namespace mf;
    const int in = Launch(StreamChunksKernel<false>, 1, kStreamThreads, 0, static_cast<hipStream_t>(stream), 0, 0, 0, 0, 0, 0u, 1u, 1u, 1u);
    const int out = Launch(StreamChunksKernel<true>, 1, kStreamThreads, 0, static_cast<hipStream_t>(stream), 0, 0, 0, 0, 0, 0u, 1u, 1u, 1u);
    return in != 0 ? in : out;
}

static int LaunchChunks(bool beside, int toHost, void *ring, const void *chunks, void *hostWords, void *gpuWords, uint64_t base, uint32_t count,
                        uint32_t slots, uint32_t limitMillis, void *stream)
{
    using namespace mf;
    int dev = 0;
    int khz = 0;
    if (ring == nullptr || chunks == nullptr || hostWords == nullptr || gpuWords == nullptr || count == 0 || slots == 0 ||
        (toHost != 0 && count > slots) || limitMillis == 0 || limitMillis > kStreamMostMillis ||
        hipGetDevice(&dev) != hipSuccess || hipDeviceGetAttribute(&khz, hipDeviceAttributeWallClockRate, dev) != hipSuccess || khz <= 0 || khz > 1000000) {
        return -1;
    }
    const uint32_t most = toHost != 0 ? kStreamGroupsOut : kStreamGroupsIn;
    const uint32_t groups = count < most ? count : most;
    const uint32_t ticks = static_cast<uint32_t>(khz) * limitMillis;
    const auto kernel = toHost != 0 ? StreamChunksKernel<true> : StreamChunksKernel<false>;
    hipStream_t s = static_cast<hipStream_t>(stream);
    if (!beside) {
        return Launch(kernel, groups, kStreamThreads, 0, s, At(ring), At(chunks), At(hostWords), At(gpuWords), base, count, slots, groups, ticks);
    }
    hipExtLaunchKernelGGL(kernel, dim3(groups), dim3(kStreamThreads), 0, s, nullptr, nullptr, hipExtAnyOrderLaunch, At(ring), At(chunks),
                          At(hostWords), At(gpuWords), base, count, slots, groups, ticks);
    return static_cast<int>(hipGetLastError());
}

extern "C" int mfk_stream_chunks(int toHost, void *ring, const void *chunks, void *hostWords, void *gpuWords, uint64_t base, uint32_t count,
                                 uint32_t slots, uint32_t limitMillis, void *stream)
{
    return LaunchChunks(false, toHost, ring, chunks, hostWords, gpuWords, base, count, slots, limitMillis, stream);
}

extern "C" int mfk_stream_chunks_beside(int toHost, void *ring, const void *chunks, void *hostWords, void *gpuWords, uint64_t base, uint32_t count,
                                        uint32_t slots, uint32_t limitMillis, void *stream)
{
    return LaunchChunks(true, toHost, ring, chunks, hostWords, gpuWords, base, count, slots, limitMillis, stream);
}
