// Local MoE token dispatch / combine for gfx950.
//
// The reference has no counterpart (its only device code is the copy plugin,
// src/hybm/csrc/copy_extend/hybm_copy_kernel.cpp); the arithmetic these kernels
// are held to is the specification in the test oracle:
//   dispatch  entry i = t*K + k goes to row offsets[e] + #{j < i : topk[j] == e}
//             (a stable counting sort of the flat (t,k) order by expert id)
//   combine   y[t][h] = bf16_rne(fma(w[t][K-1], v[K-1], ... fma(w[t][0], v[0], 0)))
//
// One launch for a small dispatch (MoeDispatchSmallKernel, up to 4096 entries: every token ranks its own entries) and for one whose
// rows fit the last-level cache (MoeDispatchCountKernel, up to 49152 entries: every workgroup counts all entries).
// Three launches for a larger one (two when the entries fill few rank blocks), one for combine:
//   MoeHistKernel    per-block expert histograms (wave ballots + LDS); not launched for a few blocks,
//                    which count one another's entries inside the rank kernel
//   MoeRankKernel    cross-block scan, stable rank of every entry -> rowOf/srcOf, counts, offsets,
//                    and for the tile permute the rows of every step of entries in ascending order
//   the permute, one of
//   MoePermuteTileKernel  rows of whole cache lines, enough work: the output walked in runs of
//                    consecutive rows, in 2 KiB tiles, one stream of steps per XCD, token rows
//                    re-read from that XCD's L2 (HBM bound: H*2*(1+K) bytes per token)
//   MoePermuteLoopKernel  other wide rows: waves that walk the tokens, a row read once into
//                    registers and stored to its K destination rows
//   MoePermuteKernel other narrow rows: one workgroup per token
//   MoeCombineKernel one workgroup per token: K rows gathered, fp32 FMA chain in slot
//                    order, one rounding to bf16 (HBM bound: H*2*(K+1) bytes per token)
//   MoeCombineWindowKernel  the same arithmetic for wide rows and many tokens, by waves that
//                    stay for the whole launch and, chip-wide and by the clock, read for
//                    most of a period and write at its end
// Ranks come from ballots and prefix sums, never from atomics on a shared
// cursor (the only atomics add up plain counts), so the permutation is the same on
// every run and equals the CPU sort.
#include <hip/hip_runtime.h>
#include <stdint.h>

#include <atomic>

#include "../rt/mf_rt.h"
#include "launch.h"
#include "through.h"
#include "window_clock.h"

namespace mf {
namespace {

// A rank launch is a chain of steps that each wait (ids, ballots, LDS tables, scans), so a block has a wave per slice: with four
// waves of four slices each 1024 / 2048 tokens of 1024 elements at top-8 took 14.5 / 18.5 us per dispatch, so 12.4 / 15.3, 4096 of 7168
// 92.5 / 90.4.
constexpr uint32_t kRankThreads = 1024;                // 16 waves
constexpr uint32_t kRankRounds = 1;                    // entries per lane
constexpr uint32_t kRankBlock = kRankThreads * kRankRounds;  // 1024 entries per workgroup
constexpr uint32_t kRankSlices = kRankBlock / 64;      // 16 wave-sized slices, in entry order
constexpr uint32_t kMaxExperts = 512;
constexpr uint32_t kRowThreads = 256;
constexpr uint32_t kMaxTopK = 16;
constexpr uint32_t kCountingBlocks = 24;                // launches of up to this many rank blocks need no histogram kernel
constexpr uint32_t kCountingBatch = 8;                  // ... whose ids they request together
static_assert(kCountingBlocks * kRankBlock < 1u << 16, "counts of half a word");
constexpr uint32_t kHistPad = 32;                      // rows of the [expert][block] table are padded to this many blocks

typedef uint32_t u32x4 __attribute__((ext_vector_type(4)));
typedef int32_t i32x4a __attribute__((ext_vector_type(4), aligned(4)));
#define MF_GLOBAL __attribute__((address_space(1)))

// Lanes of the wave whose expert id equals mine (among lanes with valid == true).
__device__ __forceinline__ uint64_t PeersOf(uint32_t expert, bool valid, uint32_t bits)
{
    uint64_t peers = __ballot(valid);
    for (uint32_t b = 0; b < bits; ++b) {
        const bool bit = (expert >> b) & 1u;
        const uint64_t vote = __ballot(bit);
        peers &= bit ? vote : ~vote;
    }
    return peers;
}

__device__ __forceinline__ uint32_t BitsFor(uint32_t experts)
{
    return 32u - __builtin_clz(experts > 1 ? experts - 1 : 1u);
}

// Slice s of a block holds entries [block*1024 + s*64, +64), lane = offset in the slice.
// Wave w of the workgroup handles slice w.
// hist[s][e] = number of entries of slice s routed to expert e.
__device__ __forceinline__ void SliceHistograms(const int32_t *__restrict__ topk, uint32_t total, uint32_t experts,
                                                uint32_t blockBase, uint32_t *hist /* [kRankSlices][experts] in LDS */,
                                                uint32_t *myExpert, uint32_t *myRank, uint32_t *bad)
{
    const uint32_t lane = threadIdx.x & 63u;
    const uint32_t wave = threadIdx.x >> 6;
    const uint32_t bits = BitsFor(experts);
    // all expert ids of this lane are requested before anything waits on them
    int32_t ids[kRankRounds];
#pragma unroll
    for (uint32_t r = 0; r < kRankRounds; ++r) {
        const uint32_t idx = blockBase + (wave + r * (kRankThreads / 64)) * 64 + lane;
        ids[r] = idx < total ? topk[idx] : -1;
    }
    for (uint32_t i = threadIdx.x; i < kRankSlices * experts; i += kRankThreads) {
        hist[i] = 0;
    }
    __syncthreads();
#pragma unroll
    for (uint32_t r = 0; r < kRankRounds; ++r) {
        const uint32_t slice = wave + r * (kRankThreads / 64);
        const uint32_t idx = blockBase + slice * 64 + lane;
        const int32_t e = ids[r];
        const bool valid = e >= 0 && static_cast<uint32_t>(e) < experts;
        if (idx < total && !valid) {
            *bad = 1;
        }
        const uint64_t peers = PeersOf(static_cast<uint32_t>(e), valid, bits);
        const uint64_t below = peers & ((1ull << lane) - 1ull);
        myExpert[r] = valid ? static_cast<uint32_t>(e) : 0xFFFFFFFFu;
        myRank[r] = __popcll(below);
        if (valid && below == 0) {  // first lane of each group publishes the group's size
            hist[slice * experts + static_cast<uint32_t>(e)] = __popcll(peers);
        }
    }
    __syncthreads();
}

// The rank launches keep a quarter of the chip and no memory busy.  The workgroups behind theirs read the token rows, which
// leaves them in the last-level cache (256 MiB, in front of HBM) for the permute: it then streams its stores without
// the eleventh part of reads from HBM between them.  8192 tokens of 7168 elements at top-8, rows not in that cache before: dispatch
// 191 against 218 us; 16 384 tokens 375 against 413.  Rows that are there already gain nothing from it: dispatch and combine of the same
// 117 MB 352 against 350 us (dispatch alone 184 against 178).  128 workgroups of sixteen waves: with 64 / 32 of them dispatch takes 203 / 239 us,
// with 128 of four waves 195, with 128 of sixteen 189.
// Rows below kWarmMinBytes are the likelier to be there (94 us for 58 MB in turn with two others, 97 with this); beyond
// kWarmMaxBytes the first rows would be gone again before their turn.
constexpr uint64_t kWarmMinBytes = 80ull << 20;
constexpr uint64_t kWarmMaxBytes = 224ull << 20;
constexpr uint32_t kWarmGroups = 128;
constexpr uint32_t kWarmPieces = 8;                     // 128-bit loads in flight per lane
constexpr uint32_t kWarmHistPercent = 30;               // share of the shorter first launch
// Rows of so many bytes are read by all CUs that rank nothing, as long as those are many.  Dispatch with 128 groups and 30 % / so, us, four processes each in turn on one machine, each
// within 0.5: 8192 tokens of 7168 elements (117 MB) top-8 over 256 experts 180.6 / 176.5, over 8 169.4 / 164.9, top-6 144.8 / 140.8, top-4 112.2 / 108.0, top-2 73.9 / 73.4; 7168 of 7168 (103 MB)
// 155.3 / 153.5, 6144 of 10 240 (126 MB) 194.0 / 188.9, 8192 of 8192 and 4096 of 16 384 (134 MB) 204.5 / 202.6, 204.3 / 202.0; at top-4 over 64 8192 of 12 288 (201 MB) 208.5 / 194.1, 3584 of 28 672
// (206 MB) 213.7 / 211.0; but 84 MB, partly in that cache, 98.2 / 100.1.  Under a tracer, which sets the launches apart, the histograms, ranks and permute of the first take 8.7 + 18.8 + 157 / 9.1 +
// 14.5 + 162, at top-4 8.3 + 18.6 + 84.7 / 8.7 + 13.7 + 84.7.
constexpr uint64_t kWarmMoreBytes = 96ull << 20;
constexpr uint32_t kWarmMoreGroups = 192;
constexpr uint32_t kWarmMoreBlocks = 64;                // with which they are 256 (16 384 tokens of 4096 elements, 128 blocks, dispatch 208.3 / 210.0)
constexpr uint32_t kWarmMoreHistPercent = 40;

__device__ __forceinline__ void WarmRows(const u32x4 *rows, uint64_t units, uint32_t group, uint32_t groups)
{
    const MF_GLOBAL u32x4 *src = reinterpret_cast<const MF_GLOBAL u32x4 *>(reinterpret_cast<uint64_t>(rows));
    constexpr uint64_t kStep = kWarmPieces * kRankThreads;
    for (uint64_t u0 = group * kStep; u0 < units; u0 += groups * kStep) {
        u32x4 v[kWarmPieces];
#pragma unroll
        for (uint32_t j = 0; j < kWarmPieces; ++j) {
            const uint64_t u = u0 + j * kRankThreads + threadIdx.x;
            v[j] = src[u < units ? u : units - 1];
        }
#pragma unroll
        for (uint32_t j = 0; j < kWarmPieces; ++j) {
            asm volatile("" : : "v"(v[j]));             // the load is all that is wanted
        }
    }
}

__global__ __launch_bounds__(kRankThreads) void MoeHistKernel(const int32_t *__restrict__ topk, uint32_t total,
                                                              uint32_t experts, uint32_t *__restrict__ blockHist,
                                                              uint32_t histStride, uint32_t *__restrict__ blockBad,
                                                              uint32_t blocks, const u32x4 *__restrict__ warm, uint64_t warmUnits)
{
    if (blockIdx.x >= blocks) {
        WarmRows(warm, warmUnits, blockIdx.x - blocks, gridDim.x - blocks);
        return;
    }
    extern __shared__ uint32_t hist[];
    uint32_t e[kRankRounds];
    uint32_t r[kRankRounds];
    uint32_t bad = 0;
    SliceHistograms(topk, total, experts, blockIdx.x * kRankBlock, hist, e, r, &bad);
    for (uint32_t x = threadIdx.x; x < experts; x += kRankThreads) {
        uint32_t sum = 0;
        for (uint32_t s = 0; s < kRankSlices; ++s) {
            sum += hist[s * experts + x];
        }
        blockHist[static_cast<uint64_t>(x) * histStride + blockIdx.x] = sum;  // [expert][block], rows padded to kHistPad
        if (blockIdx.x == 0) {
            for (uint32_t pad = blocks; pad < histStride; ++pad) {
                blockHist[static_cast<uint64_t>(x) * histStride + pad] = 0;
            }
        }
    }
    // every block reports, so the flags need no clearing between calls
    const uint32_t anyBad = __syncthreads_or(static_cast<int>(bad)) != 0 ? 1u : 0u;
    if (threadIdx.x == 0) {
        blockBad[blockIdx.x] = anyBad;
    }
}

__global__ __launch_bounds__(kRankThreads) void MoeRankKernel(const int32_t *__restrict__ topk, uint32_t total,
                                                              uint32_t experts, const uint32_t *__restrict__ blockHist,
                                                              uint32_t histStride, int32_t *__restrict__ counts, int32_t *__restrict__ offsets,
                                                              int32_t *__restrict__ rowOf, int32_t *__restrict__ srcOf,
                                                              const uint32_t *__restrict__ blockBad,
                                                              uint32_t *__restrict__ status, uint32_t topK,
                                                              int2 *__restrict__ runOrder, uint32_t restSlices,
                                                              uint32_t together, uint32_t blocksTogether, uint32_t blocksWhole,
                                                              uint32_t blocks, const u32x4 *__restrict__ warm, uint64_t warmUnits)
{
    if (blockIdx.x >= blocks) {
        WarmRows(warm, warmUnits, blockIdx.x - blocks, gridDim.x - blocks);
        return;
    }
    extern __shared__ uint32_t lds[];
    uint32_t *hist = lds;                                 // [kRankSlices][experts]
    uint32_t *base = lds + kRankSlices * experts;         // [experts] first row of this block's entries per expert
    uint32_t *scan = base + experts;                      // [kRankThreads] scratch of the block scan
    uint32_t *stepValid = scan + kRankThreads;            // [kRankSlices] entries with a row in each step of the block
    uint32_t *cum = stepValid + kRankSlices;              // [steps][experts] entries of the step with a smaller expert id
    uint32_t myExpert[kRankRounds];
    uint32_t myRank[kRankRounds];
    uint32_t bad = 0;
    // blockHist == nullptr: no histogram kernel ran before this launch.  Its few blocks count the entries of the other
    // blocks themselves, each for itself: per expert, the entries of all other blocks and those of the blocks before it
    // (plain counts, so LDS atomics give the same result every time).
    const bool tabled = blockHist != nullptr;
    const bool counting = !tabled;
    const uint32_t stepSlices = blockIdx.x < blocksWhole ? kRankSlices : restSlices;
    const uint32_t steps = runOrder != nullptr ? kRankSlices / stepSlices : 0;
    uint32_t *others = cum + steps * experts;             // [experts], counting only
    const bool grouped = blockIdx.x < blocksTogether;     // a step is `together` blocks, from groupFirst on
    const uint32_t groupFirst = grouped ? blockIdx.x / together * together : blockIdx.x;
    uint32_t *groupBefore = cum + steps * experts;        // [experts] entries of the step's blocks before this one, grouped only
    for (uint32_t i = threadIdx.x; counting && i < experts; i += kRankThreads) {
        others[i] = 0;
    }
    SliceHistograms(topk, total, experts, blockIdx.x * kRankBlock, hist, myExpert, myRank, &bad);
    if (counting) {
        // One word per expert, entries of the blocks before this one above entries of all others (kCountingBlocks * kRankBlock
        // fit 16 bits).  The ids of eight blocks are requested before the first is counted: with a round trip per block, 1024 tokens
        // took 15.9 us per dispatch, so 14.5.
        for (uint32_t from = 0; from < blocks; from += kCountingBatch) {
            int32_t id[kCountingBatch];
#pragma unroll
            for (uint32_t q = 0; q < kCountingBatch; ++q) {
                const uint32_t at = (from + q) * kRankBlock + threadIdx.x;
                id[q] = at < total ? topk[at] : 0;
            }
#pragma unroll
            for (uint32_t q = 0; q < kCountingBatch; ++q) {
                if (from + q != blockIdx.x && (from + q) * kRankBlock + threadIdx.x < total) {
                    if (static_cast<uint32_t>(id[q]) < experts) {
                        atomicAdd(&others[id[q]], from + q < blockIdx.x ? 0x10001u : 1u);
                    } else {
                        bad = 1;
                    }
                }
            }
        }
        __syncthreads();
    }
    if (blockIdx.x == 0) {
        uint32_t any = tabled ? 0 : bad;
        for (uint32_t blk = threadIdx.x; tabled && blk < blocks; blk += kRankThreads) {
            any |= blockBad[blk];
        }
        any = __syncthreads_or(static_cast<int>(any)) != 0 ? 1u : 0u;
        if (threadIdx.x == 0) {
            status[0] = any;  // 1: some expert id was outside [0, experts); those entries got row -1
        }
    }
    // totals and "entries of earlier blocks" per expert
    uint32_t tot[(kMaxExperts + kRankThreads - 1) / kRankThreads];
    uint32_t before[(kMaxExperts + kRankThreads - 1) / kRankThreads];
    uint32_t mine = 0;
#pragma unroll
    for (uint32_t j = 0; j < (kMaxExperts + kRankThreads - 1) / kRankThreads; ++j) {
        // thread t owns the contiguous experts t*per .. t*per+per-1 so that a scan over threads is a scan over experts
        tot[j] = 0;
        before[j] = 0;
    }
    const uint32_t per = (experts + kRankThreads - 1) / kRankThreads;
    for (uint32_t j = 0; j < per; ++j) {
        const uint32_t x = threadIdx.x * per + j;
        if (x < experts) {
            // one contiguous row of the [expert][block] table per expert, fetched 16 bytes at a time
            const uint32_t *rowHist = blockHist + static_cast<uint64_t>(x) * histStride;
            uint32_t t = 0;
            uint32_t b = 0;
            uint32_t g = 0;
            uint32_t gb = 0;
            if (counting) {
#pragma unroll
                for (uint32_t sl = 0; sl < kRankSlices; ++sl) {
                    t += hist[sl * experts + x];
                }
                t += others[x] & 0xFFFFu;
                b = others[x] >> 16;
            }
            // kHistPad blocks per step, all their loads requested before the first is used (with one load per step the
            // loop waited a round trip per four blocks)
            for (uint32_t blk = 0; tabled && blk < blocks; blk += kHistPad) {
                u32x4 v[kHistPad / 4];
#pragma unroll
                for (uint32_t q = 0; q < kHistPad / 4; ++q) {
                    v[q] = *reinterpret_cast<const u32x4 *>(rowHist + blk + 4 * q);  // rows are padded with zeros up to histStride
                }
#pragma unroll
                for (uint32_t q = 0; q < kHistPad / 4; ++q) {
#pragma unroll
                    for (uint32_t i = 0; i < 4; ++i) {
                        t += v[q][i];
                        b += blk + 4 * q + i < blockIdx.x ? v[q][i] : 0u;
                    }
                }
                if (grouped && blk == groupFirst / kHistPad * kHistPad) {       // a step's blocks lie in one
#pragma unroll
                    for (uint32_t q = 0; q < kHistPad / 4; ++q) {
#pragma unroll
                        for (uint32_t i = 0; i < 4; ++i) {
                            const uint32_t after = blk + 4 * q + i - groupFirst;    // wraps in front of it
                            g += after < together ? v[q][i] : 0u;
                            gb += after < blockIdx.x - groupFirst ? v[q][i] : 0u;
                        }
                    }
                }
            }
            tot[j] = t;
            before[j] = b;
            mine += t;
            if (grouped) {
                cum[x] = g;
                groupBefore[x] = gb;
            }
        }
    }
    // exclusive scan of `mine` over the threads: shuffles inside each wave, LDS across the waves
    uint32_t incl = mine;
#pragma unroll
    for (uint32_t step = 1; step < 64; step <<= 1) {
        const uint32_t up = __shfl_up(incl, step, 64);
        incl += (threadIdx.x & 63u) >= step ? up : 0u;
    }
    if ((threadIdx.x & 63u) == 63u) {
        scan[threadIdx.x >> 6] = incl;
    }
    __syncthreads();
    uint32_t waveBase = 0;
    for (uint32_t wv = 0; wv < (threadIdx.x >> 6); ++wv) {
        waveBase += scan[wv];
    }
    incl += waveBase;
    uint32_t run = incl - mine;
    for (uint32_t j = 0; j < per; ++j) {
        const uint32_t x = threadIdx.x * per + j;
        if (x < experts) {
            if (blockIdx.x == 0) {
                counts[x] = static_cast<int32_t>(tot[j]);
                offsets[x] = static_cast<int32_t>(run);
            }
            base[x] = run + before[j];
            run += tot[j];
        }
    }
    __syncthreads();
    // Turn slice histograms into exclusive prefixes over the slices of this block.  For the run-ordered list the
    // block is cut into steps of stepSlices slices (the tile permute works through one step at a time); the
    // entries per (step, expert) are what the prefix gains over a step.  (Those of a step of several blocks are in cum already.)
    for (uint32_t x = threadIdx.x; x < experts; x += kRankThreads) {
        uint32_t acc = base[x];
        uint32_t stepStart = acc;
        uint32_t v[kRankSlices];                          // all read before the first is replaced
#pragma unroll
        for (uint32_t s = 0; s < kRankSlices; ++s) {
            v[s] = hist[s * experts + x];
        }
#pragma unroll
        for (uint32_t s = 0; s < kRankSlices; ++s) {
            hist[s * experts + x] = acc;
            acc += v[s];
            if (steps != 0 && !grouped && (s + 1) % stepSlices == 0) {
                cum[(s / stepSlices) * experts + x] = acc - stepStart;
                stepStart = acc;
            }
        }
    }
    __syncthreads();
    const uint32_t lane = threadIdx.x & 63u;
    const uint32_t wave = threadIdx.x >> 6;
    if (steps != 0) {
        // cum[j][x]: entries of step j routed to an expert below x, i.e. where the rows of expert x start in the list
        // of the step's rows in ascending order; behind them those of the step's blocks before this one.  One wave per step; a lane scans experts/64 neighbours itself.
        const uint32_t perLane = (experts + 63) / 64;     // at most kMaxExperts / 64
        for (uint32_t j = wave; j < steps; j += kRankThreads / 64) {
            uint32_t mineOf[kMaxExperts / 64];
            uint32_t sum = 0;
#pragma unroll
            for (uint32_t i = 0; i < kMaxExperts / 64; ++i) {
                const uint32_t x = lane * perLane + i;
                mineOf[i] = i < perLane && x < experts ? cum[j * experts + x] : 0u;
                sum += mineOf[i];
            }
            uint32_t incl2 = sum;
#pragma unroll
            for (uint32_t step = 1; step < 64; step <<= 1) {
                const uint32_t up = __shfl_up(incl2, step, 64);
                incl2 += lane >= step ? up : 0u;
            }
            uint32_t at = incl2 - sum;
#pragma unroll
            for (uint32_t i = 0; i < kMaxExperts / 64; ++i) {
                const uint32_t x = lane * perLane + i;
                if (i < perLane && x < experts) {
                    cum[j * experts + x] = at + (grouped ? groupBefore[x] : 0u);
                    at += mineOf[i];
                }
            }
            if (lane == 63) {
                stepValid[j] = incl2;
            }
        }
        __syncthreads();
    }
#pragma unroll
    for (uint32_t r = 0; r < kRankRounds; ++r) {
        const uint32_t slice = wave + r * (kRankThreads / 64);
        const uint32_t idx = blockIdx.x * kRankBlock + slice * 64 + lane;
        if (idx < total) {
            int32_t row = -1;
            if (myExpert[r] != 0xFFFFFFFFu) {
                row = static_cast<int32_t>(hist[slice * experts + myExpert[r]] + myRank[r]);
                if (srcOf != nullptr) {
                    srcOf[row] = static_cast<int32_t>(idx);
                }
                if (runOrder != nullptr) {
                    const uint32_t j = slice / stepSlices;
                    const uint32_t firstOfStep = hist[j * stepSlices * experts + myExpert[r]];
                    const uint32_t at = cum[j * experts + myExpert[r]] + (static_cast<uint32_t>(row) - firstOfStep);
                    runOrder[static_cast<uint64_t>(groupFirst) * kRankBlock + j * stepSlices * 64 + at] =
                        make_int2(row, static_cast<int32_t>(idx / topK));
                }
            }
            rowOf[idx] = row;
        }
    }
    if (runOrder != nullptr) {
        // slots past a step's valid entries (ids out of range, the tail of the last block) name no row
        const uint32_t stepEntries = stepSlices * 64;
        for (uint32_t slot = threadIdx.x; slot < kRankBlock; slot += kRankThreads) {
            const uint32_t j = slot / stepEntries;
            if (slot - j * stepEntries + (blockIdx.x - groupFirst) * kRankBlock >= stepValid[j]) {
                runOrder[static_cast<uint64_t>(blockIdx.x) * kRankBlock + slot] = make_int2(-1, 0);
            }
        }
    }
}

template <int kMode>
__device__ __forceinline__ void RowStore(MF_GLOBAL u32x4 *p, u32x4 v)
{
    if (kMode == 2) {
        StoreThrough16(reinterpret_cast<uint64_t>(p), v);
    } else if (kMode == 1) {
        __builtin_nontemporal_store(v, p);
    } else {
        *p = v;
    }
}

// One workgroup per token.  unitsPerRow = H*2/16.  Each lane keeps up to kHold 128-bit pieces of
// the token's row in registers and stores them to the token's K destination rows.
template <uint32_t kThreads, uint32_t kHold, int kMode>
__global__ __launch_bounds__(kThreads) void MoePermuteKernel(const u32x4 *__restrict__ x,
                                                             const int32_t *__restrict__ rowOf, uint32_t topK,
                                                             uint32_t unitsPerRow, uint32_t parts, u32x4 *__restrict__ out)
{
    const uint32_t token = blockIdx.x / parts;
    const uint32_t part = blockIdx.x - token * parts;
    const uint32_t perPart = (unitsPerRow + parts - 1) / parts;
    const uint32_t begin = part * perPart;
    const uint32_t end = begin + perPart < unitsPerRow ? begin + perPart : unitsPerRow;
    const MF_GLOBAL u32x4 *src = reinterpret_cast<const MF_GLOBAL u32x4 *>(reinterpret_cast<uint64_t>(x)) +
                                 static_cast<uint64_t>(token) * unitsPerRow;
    int32_t rows[kMaxTopK];
#pragma unroll
    for (uint32_t k = 0; k < kMaxTopK; ++k) {
        rows[k] = k < topK ? rowOf[static_cast<uint64_t>(token) * topK + k] : -1;
    }
    for (uint32_t u0 = begin; u0 < end; u0 += kHold * kThreads) {
        u32x4 v[kHold];
#pragma unroll
        for (uint32_t j = 0; j < kHold; ++j) {
            const uint32_t u = u0 + j * kThreads + threadIdx.x;
            if (u < end) {
                v[j] = __builtin_nontemporal_load(src + u);
            }
        }
#pragma unroll
        for (uint32_t k = 0; k < kMaxTopK; ++k) {
            if (k < topK && rows[k] >= 0) {
                MF_GLOBAL u32x4 *dst = reinterpret_cast<MF_GLOBAL u32x4 *>(reinterpret_cast<uint64_t>(out)) +
                                       static_cast<uint64_t>(rows[k]) * unitsPerRow;
#pragma unroll
                for (uint32_t j = 0; j < kHold; ++j) {
                    const uint32_t u = u0 + j * kThreads + threadIdx.x;
                    if (u < end) {
                        RowStore<kMode>(dst + u, v[j]);
                    }
                }
            }
        }
    }
}

// Single-wave workgroups that walk items (token, part) with stride gridDim.x and fetch the next
// item's pieces before they store the current one's: after the first item of every wave, reads of
// x overlap the eight-fold stores instead of preceding them.
template <uint32_t kHold>
__global__ __launch_bounds__(64) void MoePermuteLoopKernel(const u32x4 *__restrict__ x, const int32_t *__restrict__ rowOf,
                                                           uint32_t topK, uint32_t unitsPerRow, uint32_t parts,
                                                           uint32_t items, u32x4 *__restrict__ out)
{
    const uint32_t perPart = (unitsPerRow + parts - 1) / parts;
    const MF_GLOBAL u32x4 *xg = reinterpret_cast<const MF_GLOBAL u32x4 *>(reinterpret_cast<uint64_t>(x));
    MF_GLOBAL u32x4 *og = reinterpret_cast<MF_GLOBAL u32x4 *>(reinterpret_cast<uint64_t>(out));
    auto fetch = [&](uint32_t item, u32x4(&v)[kHold], int32_t(&rows)[kMaxTopK]) {
        const uint32_t token = item / parts;
        const uint32_t begin = (item - token * parts) * perPart;
        const uint32_t end = begin + perPart < unitsPerRow ? begin + perPart : unitsPerRow;
#pragma unroll
        for (uint32_t k = 0; k < kMaxTopK; ++k) {
            rows[k] = k < topK ? rowOf[static_cast<uint64_t>(token) * topK + k] : -1;
        }
#pragma unroll
        for (uint32_t j = 0; j < kHold; ++j) {
            const uint32_t u = begin + j * 64 + threadIdx.x;
            if (u < end) {
                v[j] = __builtin_nontemporal_load(xg + static_cast<uint64_t>(token) * unitsPerRow + u);
            }
        }
    };
    auto spread = [&](uint32_t item, const u32x4(&v)[kHold], const int32_t(&rows)[kMaxTopK]) {
        const uint32_t token = item / parts;
        const uint32_t begin = (item - token * parts) * perPart;
        const uint32_t end = begin + perPart < unitsPerRow ? begin + perPart : unitsPerRow;
#pragma unroll
        for (uint32_t k = 0; k < kMaxTopK; ++k) {
            if (k < topK && rows[k] >= 0) {
                MF_GLOBAL u32x4 *dst = og + static_cast<uint64_t>(rows[k]) * unitsPerRow;
#pragma unroll
                for (uint32_t j = 0; j < kHold; ++j) {
                    const uint32_t u = begin + j * 64 + threadIdx.x;
                    if (u < end) {
                        dst[u] = v[j];
                    }
                }
            }
        }
    };
    // two register sets, a and b, alternate between "being fetched" and "being stored"
    uint32_t ia = blockIdx.x;
    if (ia >= items) {
        return;
    }
    u32x4 a[kHold];
    u32x4 b[kHold];
    int32_t ra[kMaxTopK];
    int32_t rb[kMaxTopK];
    fetch(ia, a, ra);
    while (true) {
        const uint32_t ib = ia + gridDim.x;
        const bool hasB = ib < items;
        if (hasB) {
            fetch(ib, b, rb);
        }
        spread(ia, a, ra);
        if (!hasB) {
            break;
        }
        ia = ib + gridDim.x;
        const bool hasA = ia < items;
        if (hasA) {
            fetch(ia, a, ra);
        }
        spread(ib, b, rb);
        if (!hasA) {
            break;
        }
    }
}

// The permute of wide rows when a block of kRankBlock entries holds no more of x than an XCD's L2 keeps:
// output-ordered, in tiles.  runOrder lists, step by step (a step is a block of kRankBlock entries, several or a power-of-two
// part of one, chosen so that the token rows of a step fit), the step's output rows in ascending
// order (runs of consecutive rows per expert) with the token each row is a copy of.  Workgroup i, a single
// wave, belongs to stream i % 8 (the dispatcher deals consecutive workgroups to the eight XCDs in turn);
// stream s takes the steps s, s + 8, ... one after the other and walks a step's rows in list order, a row in
// tiles of 128 units (2 KiB).  So an XCD writes runs of consecutive rows front to back, two stores per wave,
// the store pattern this part takes fastest, and the K reads of a token row all come from the same XCD within
// the time it spends on the block: the first from HBM, the others from its L2 (plain loads), which stores that
// are written through pass without evicting x.  8192 x 7168, top-8, 256 experts, one block a step: 163-166 us against 192 us for
// the token-ordered loop kernel; streams that do not follow the XCDs 283 us.
constexpr uint32_t kTileUnits = 128;
constexpr uint32_t kTileStreams = 8;
// The longer a step's runs the better HBM takes them, as long as its token rows stay in the L2: kTileStepBytes of them, all of it (8192 x 7168 in steps of
// four blocks, 7.3 MB, 227 us and not 193).  So a step has several blocks, as many as make runs of kTileRunBytes, and blocks that their rows cut in two are
// whole again from four slots on.  Dispatch, us, one block a step / so, top-8, 256 experts: 8192 x 7168 193 / 185, 16 384 382 / 368, 4100 110 / 96, 7300 x 5120 134 / 119,
// 6200 x 4096 96.5 / 83.5, 16 384 232 / 213, 30 000 x 2048 233 / 214, 6200 56.0 / 51.1; 512 experts 8192 x 7168 204 / 194, x 2048 70.4 / 62.7.  128 experts have runs twice
// as long as they are: 8192 x 7168 183 / 179, 6400 148 / 138, but x 2048 58.0 / 58.8, x 4096 99.9 / 100.0, hence kTileLongRowBytes; 64 lose (x 7168 174.0 / 174.7, x 5120
// 120.9 / 123.2).  Rows of one tile lose with two and four blocks (7300 x 1024 38.4 / 39.4), and so do four slots, whose rows are read less often from the
// L2 (9999 x 4096 77.2 / 78.5).
// Steps that the streams do not divide leave XCDs idle at the end, 4 of 56 the half of them for a seventh of the time: what is left of the last round
// is cut until they do (6900 x 7168 over 8 experts 148 / 144, 6500 at top-4 88.1 / 84.8, 7000 over 64 at top-6 127 / 122.5, 6300 x 1024 33.0 / 31.6; it is
// most of what 4100, 6200 and 6400 tokens above gain).
constexpr uint64_t kTileStepBytes = 4ull << 20;
constexpr uint64_t kTileRunBytes = 128ull << 10;
constexpr uint32_t kTileMostTogether = 8;
constexpr uint32_t kTileFewExperts = 128;
constexpr uint32_t kTileLongRowBytes = 12288;
constexpr uint32_t kTileTogetherRowBytes = 4096;
constexpr uint32_t kTileWholeSlots = 4;                 // the fewest for whole blocks of more than half of kTileStepBytes, and too few for several
static_assert(kHistPad % kTileMostTogether == 0, "the counts of a step's blocks are fetched together");

// Steps of longEntries entries first, then of kRankBlock, then of restEntries: rounds of a step for every stream, the last one what is left.
struct TilePlan {
    uint32_t entries;           // of the list, whole blocks
    uint32_t longEntries;
    uint32_t longRounds;
    uint32_t wholeRounds;
    uint32_t restEntries;
};

__global__ __launch_bounds__(64) void MoePermuteTileKernel(const u32x4 *__restrict__ x, const int2 *__restrict__ runOrder,
                                                           uint32_t unitsPerRow, uint32_t tilesPerRow, TilePlan plan, u32x4 *__restrict__ out)
{
    const uint32_t stream = blockIdx.x % kTileStreams;
    uint32_t q = blockIdx.x / kTileStreams;
    const uint32_t tilesLong = plan.longRounds * plan.longEntries * tilesPerRow;
    const uint32_t tilesWhole = plan.wholeRounds * kRankBlock * tilesPerRow;
    uint32_t each = plan.longEntries;
    uint32_t from = 0;
    if (q >= tilesLong) {
        q -= tilesLong;
        from = plan.longRounds * kTileStreams * plan.longEntries;
        each = kRankBlock;
        if (q >= tilesWhole) {
            q -= tilesWhole;
            from += plan.wholeRounds * kTileStreams * kRankBlock;
            each = plan.restEntries;
        }
    }
    const uint32_t tilesPerStep = each * tilesPerRow;
    const uint32_t round = q / tilesPerStep;
    const uint32_t within = q - round * tilesPerStep;
    const uint32_t entry = within / tilesPerRow;
    const uint32_t first = from + (round * kTileStreams + stream) * each;
    if (first >= plan.entries) {
        return;
    }
    const int2 rowAndToken = runOrder[static_cast<uint64_t>(first) + entry];
    if (rowAndToken.x < 0) {
        return;
    }
    const uint32_t begin = (within - entry * tilesPerRow) * kTileUnits;
    const MF_GLOBAL u32x4 *src = reinterpret_cast<const MF_GLOBAL u32x4 *>(reinterpret_cast<uint64_t>(x)) +
                                 static_cast<uint64_t>(rowAndToken.y) * unitsPerRow;
    MF_GLOBAL u32x4 *dst = reinterpret_cast<MF_GLOBAL u32x4 *>(reinterpret_cast<uint64_t>(out)) +
                           static_cast<uint64_t>(rowAndToken.x) * unitsPerRow;
    u32x4 v[kTileUnits / 64];
#pragma unroll
    for (uint32_t j = 0; j < kTileUnits / 64; ++j) {
        const uint32_t u = begin + j * 64 + threadIdx.x;
        if (u < unitsPerRow) {
            v[j] = src[u];
        }
    }
#pragma unroll
    for (uint32_t j = 0; j < kTileUnits / 64; ++j) {
        const uint32_t u = begin + j * 64 + threadIdx.x;
        if (u < unitsPerRow) {
            RowStore<2>(dst + u, v[j]);
        }
    }
}

// The whole dispatch of a small call in one launch: workgroup (token, part of the row) ranks the token's entries
// itself, against all the others, and stores its part of the row to the K rows; the last workgroup counts the experts.
// An entry's row is the number of entries that come before it by (expert, index), so every id is compared, as one
// word with its index, with the words of the token's K entries, and a wave adds its lanes up by counting the bits of
// the comparison.  Nothing is exchanged between workgroups.
// What bounds it: the chain of a launch and of its memory round trips (kernel arguments; the ids and the row, side by side; the
// stores), not bytes, as long as the comparisons stay few: with all parts they grow with tokens * entries.  Dispatch
// alone, with the rank launch and the permute launch / in one (both with plain stores, see below): 16 tokens of 7168 elements at
// top-8 over 256 experts 12.0 / 4.3 us, 64: 12.3 / 4.9, 128: 13.6 / 6.1, 256: 15.3 / 9.3; 2000 tokens of 1024 elements at top-2 12.1 / 7.1.  Then its
// loads were put side by side: ids, the token's own ids and the row were waited for one after the other.  Dispatch / dispatch and combine, before /
// so, 256 experts: 64 tokens of 7168 elements at top-8 4.4, 9.3 / 3.9, 8.5; 200 8.1, 13.7 / 6.7, 12.2; 400 at top-4 7.5, 13.3 / 6.5, 12.3; 1000 of 2048 at
// top-4 over 128 6.6, 12.1 / 5.3, 10.7; 2000 of 1024 at top-2 6.4, 10.3 / 5.5, 9.4.
// It ends where counting is the quicker (MoeDispatchCountKernel): at 4096 entries (1500 tokens of 1024 elements at top-4 7.3, 11.2 here and 5.8, 10.2 there,
// 3000 at top-2 9.6, 14.1 and 6.9, 11.4), and at 20480 comparisons per part (at top-8 260 of 4096 elements over 8 experts 5.7, 11.2 and 6.9, 12.0, 300 of 2048 5.0,
// 10.3 and 5.8, 10.8, 320 of 7168 9.2, 16.5 and 9.9, 17.2, but 400 11.4, 20.0 and 11.2, 19.8; at top-6 500 of 4096 7.4, 13.1 and 7.9, 13.6, but 600 9.1, 15.4 and 8.8,
// 15.1), with more than eight slots at 16384 (128 of 4096 at top-12 5.6, 13.1 and 6.1, 12.4).  Plain stores leave the rows in
// the caches, where the experts' kernel finds them (dispatch and combine in turn, 256 tokens of 7168 elements: 15.1 us), and up to kQuickBytes
// nontemporal ones do not wait for the launch's end: dispatch / both with plain stores and so, 8 tokens 4.4 / 7.0, 3.9 / 6.4, 64 5.1 / 9.9, 4.5 /
// 9.2, 160 7.7 / 12.7, 6.5 / 12.1; 300 at top-2 4.5 / 8.6, 3.5 / 8.2, 500 5.5 / 10.2, 4.3 / 10.4.
constexpr uint32_t kSmallThreads = 256;
constexpr uint32_t kSmallHold = 2;                      // 128-bit pieces of the row per lane: a part is 512 units at most
constexpr uint32_t kSmallEntries = 4096;                // the largest such call
constexpr uint32_t kSmallCompares = 20480;              // entries times slots: what a part of a token compares
constexpr uint32_t kSmallManyCompares = 16384;          // with more than eight slots
constexpr uint32_t kSmallGroups = 256;                  // rows are cut until there are so many workgroups, one per CU
constexpr uint32_t kSmallBatch = 4;                     // ids per lane requested together by the counting workgroup
static_assert(kSmallEntries <= 1u << 16 && kMaxExperts <= 1u << 16, "an entry's expert and index share a word");

// (expert, index) in one word; an id out of range comes behind every entry.
__device__ __forceinline__ uint32_t SmallKey(int32_t id, uint32_t index, uint32_t experts)
{
    return static_cast<uint32_t>(id) < experts ? static_cast<uint32_t>(id) << 16 | index : 0xFFFFFFFFu;
}

template <uint32_t kSlots, int kMode>
__global__ __launch_bounds__(kSmallThreads) void MoeDispatchSmallKernel(uint64_t x, uint64_t topkAt, uint32_t total, uint32_t topK,
                                                                        uint32_t experts, uint32_t unitsPerRow, uint32_t parts,
                                                                        uint32_t perPart, uint32_t groups, uint64_t out,
                                                                        uint64_t countsAt, uint64_t offsetsAt, uint64_t rowOfAt,
                                                                        uint64_t srcOfAt, uint64_t statusAt)
{
    const int32_t *const topk = Buffer<const int32_t>(topkAt);
    int32_t *const counts = Buffer<int32_t>(countsAt);
    int32_t *const offsets = Buffer<int32_t>(offsetsAt);
    int32_t *const rowOf = Buffer<int32_t>(rowOfAt);
    int32_t *const srcOf = Buffer<int32_t>(srcOfAt);
    __shared__ uint32_t lds[kMaxExperts + kSmallThreads / 64];
    __shared__ uint32_t anyBad;
    const uint32_t lane = threadIdx.x & 63u;
    const uint32_t wave = threadIdx.x >> 6;
    if (blockIdx.x == groups - 1) {
        uint32_t *perWave = lds + kMaxExperts;
        for (uint32_t e = threadIdx.x; e < kMaxExperts; e += kSmallThreads) {
            lds[e] = 0;
        }
        if (threadIdx.x == 0) {
            anyBad = 0;
        }
        __syncthreads();
        uint32_t bad = 0;
        for (uint32_t i0 = threadIdx.x; i0 < total; i0 += kSmallBatch * kSmallThreads) {
            int32_t id[kSmallBatch];
#pragma unroll
            for (uint32_t q = 0; q < kSmallBatch; ++q) {
                id[q] = i0 + q * kSmallThreads < total ? topk[i0 + q * kSmallThreads] : 0;
            }
#pragma unroll
            for (uint32_t q = 0; q < kSmallBatch; ++q) {
                if (i0 + q * kSmallThreads < total) {
                    if (static_cast<uint32_t>(id[q]) < experts) {
                        atomicAdd(&lds[id[q]], 1u);     // plain counts: the same whatever the order
                    } else {
                        bad = 1;
                    }
                }
            }
        }
        if (bad != 0) {
            anyBad = 1;
        }
        __syncthreads();
        constexpr uint32_t kPer = kMaxExperts / kSmallThreads;   // neighbouring experts per thread
        uint32_t mine[kPer];
        uint32_t incl = 0;
#pragma unroll
        for (uint32_t j = 0; j < kPer; ++j) {
            mine[j] = lds[threadIdx.x * kPer + j];
            incl += mine[j];
        }
        const uint32_t sum = incl;
#pragma unroll
        for (uint32_t step = 1; step < 64; step <<= 1) {
            const uint32_t up = __shfl_up(incl, step, 64);
            incl += lane >= step ? up : 0u;
        }
        if (lane == 63) {
            perWave[wave] = incl;
        }
        __syncthreads();
        uint32_t run = incl - sum;
        for (uint32_t w = 0; w < wave; ++w) {
            run += perWave[w];
        }
#pragma unroll
        for (uint32_t j = 0; j < kPer; ++j) {
            const uint32_t e = threadIdx.x * kPer + j;
            if (e < experts) {
                counts[e] = static_cast<int32_t>(mine[j]);
                offsets[e] = static_cast<int32_t>(run);
            }
            run += mine[j];
        }
        if (threadIdx.x == 0) {
            *Buffer<uint32_t>(statusAt) = anyBad;
        }
        return;
    }
    const uint32_t token = blockIdx.x / parts;
    const uint32_t part = blockIdx.x - token * parts;
    const uint32_t begin = part * perPart;
    const uint32_t end = begin + perPart < unitsPerRow ? begin + perPart : unitsPerRow;
    MF_GLOBAL u32x4 *dst = reinterpret_cast<MF_GLOBAL u32x4 *>(out);
    // An entry as one word, expert above index: what comes before the token's slots is what compares below their words.
    // Every wave looks at a quarter of the ids, for all slots.  Loads return in the order of their requests, and a load that some path
    // skips is waited for with all behind it: so the ids are requested in front of the row, and every lane requests the same number of
    // loads, those past the end what is there already.  The ranks are then known when the row has come.
    const uint32_t first = token * topK;
    const int32_t idOfLane = topk[first + (lane < topK ? lane : 0)];
    constexpr uint32_t kRound = 4 * kSmallThreads;
    const uint32_t mineAt = wave * 256 + lane * 4;
    const uint32_t lastAt = total >= 4 ? total - 4 : 0;
    const auto idsAt = [&](uint32_t at) {
        i32x4a id;
        if (total >= 4) {
            id = *reinterpret_cast<const i32x4a *>(topk + (at < lastAt ? at : lastAt));
        } else {
#pragma unroll
            for (uint32_t i = 0; i < 4; ++i) {
                id[i] = i < total ? topk[i] : -1;
            }
        }
        return id;
    };
    i32x4a id = idsAt(mineAt);
    i32x4a second = {-1, -1, -1, -1};
    if (total > kRound) {
        second = idsAt(mineAt + kRound);
    }
    const bool rows = perPart != 0;
    const MF_GLOBAL u32x4 *src = reinterpret_cast<const MF_GLOBAL u32x4 *>(rows ? x + static_cast<uint64_t>(token) * unitsPerRow * sizeof(u32x4)
                                                                                : topkAt & ~static_cast<uint64_t>(sizeof(u32x4) - 1));
    const uint32_t lastUnit = rows ? end - 1 : 0;
    u32x4 v[kSmallHold];
#pragma unroll
    for (uint32_t j = 0; j < kSmallHold; ++j) {
        const uint32_t u = begin + j * kSmallThreads + threadIdx.x;
        v[j] = src[u < lastUnit ? u : lastUnit];
    }
    const uint32_t keyOfLane = lane < topK ? SmallKey(idOfLane, first + lane, experts) : 0u;
    uint32_t own[kSlots];
    uint32_t before[kSlots];
#pragma unroll
    for (uint32_t k = 0; k < kSlots; ++k) {
        own[k] = __builtin_amdgcn_readlane(keyOfLane, k);
        before[k] = 0;
    }
    const auto compare = [&](const i32x4a &ids, uint32_t at) {
        const uint32_t from = at < lastAt ? at : lastAt;
        const uint32_t skip = at - from;                // of these, what another lane has
#pragma unroll
        for (uint32_t i = 0; i < 4; ++i) {
            const uint32_t key = i >= skip ? SmallKey(ids[i], from + i, experts) : 0xFFFFFFFFu;
#pragma unroll
            for (uint32_t k = 0; k < kSlots; ++k) {
                before[k] += __popcll(__ballot(key < own[k]));
            }
        }
    };
    compare(id, mineAt);
    if (total > kRound) {
        compare(second, mineAt + kRound);
        for (uint32_t at = mineAt + 2 * kRound; at - mineAt < total; at += kRound) {
            compare(idsAt(at), at);
        }
    }
    uint32_t mine = 0;
#pragma unroll
    for (uint32_t k = 0; k < kSlots; ++k) {
        mine = lane == k ? before[k] : mine;
    }
    if (lane < kSlots) {
        lds[kMaxTopK * (1 + wave) + lane] = mine;
    }
    __syncthreads();
    // every wave adds them up for itself, a slot a lane
    uint32_t rowOfLane = 0;
#pragma unroll
    for (uint32_t w = 0; w < kSmallThreads / 64; ++w) {
        rowOfLane += lds[kMaxTopK * (1 + w) + (lane < kSlots ? lane : 0)];
    }
    rowOfLane = static_cast<uint32_t>(idOfLane) < experts ? rowOfLane : 0xFFFFFFFFu;
    if (part == 0 && threadIdx.x < topK) {
        const int32_t row = static_cast<int32_t>(rowOfLane);
        rowOf[first + threadIdx.x] = row;
        if (srcOfAt != 0 && row >= 0) {
            srcOf[row] = static_cast<int32_t>(first + threadIdx.x);
        }
    }
#pragma unroll 1
    for (uint32_t k = 0; k < topK; ++k) {
        const uint32_t row = __builtin_amdgcn_readlane(rowOfLane, k);
        if (row != 0xFFFFFFFFu) {
#pragma unroll
            for (uint32_t j = 0; j < kSmallHold; ++j) {
                const uint32_t u = begin + j * kSmallThreads + threadIdx.x;
                if (u < end) {
                    RowStore<kMode>(dst + static_cast<uint64_t>(row) * unitsPerRow + u, v[j]);
                }
            }
        }
    }
}

// A dispatch in one launch whose entries are too many to compare with one another: a workgroup per CU takes neighbouring tokens,
// counts all ids for itself, in LDS, an id before its own entries in the upper half of the word too, and so knows where its
// own entries of every expert begin without a word from the others.  Their ranks inside the workgroup come from ballots, slice by slice.
// The rows wait in registers meanwhile, and every wave stores its pieces of 64 units K-fold.
// What bounds it: up to about 8000 entries of 2048 elements the chain of a launch (ids, counts, scan, rows, stores), beyond
// its stores.  Two launches and what lies between them went, as did the second read of the index tables.  Dispatch / dispatch and
// combine in turn, with the rank launch and the permute in front of this / with it, us: 700 tokens of 2048 elements at top-8 over 256 experts
// 13.1, 19.6 / 8.6, 13.9; 1500 17.3, 28.4 / 12.7, 21.8; 3000 26.4, 46.3 / 23.1, 38.5; 1500 of 5120 at top-6 over 128 28.3, 47.5 /
// 21.1, 35.5; 4000 of 2048 at top-2 over 8 16.3, 26.3 / 10.9, 18.4; and with every token against every entry in front of it:
// 400 of 2048 at top-8 8.6, 13.4 / 6.6, 10.7; 512 of 7168 15.4, 25.9 / 13.0, 23.4.
// A thread per id and 1024 of them: two workgroups of 512 threads took 0.1 to 1 us more, one 1 us more.
// Counts that fall on the same word wait for each other, so an expert has several words, side by side, the fewer experts the more,
// and a lane adds to its own: 16 us with four of them over 8 experts, where 64 take 7.
constexpr uint32_t kCountThreads = 1024;
constexpr uint32_t kCountWaves = kCountThreads / 64;
constexpr uint32_t kCountBatch = 4;                     // 128-bit loads of ids per lane in flight
constexpr uint32_t kCountEntries = 48u << 10;           // the largest such call: every workgroup counts all of them
constexpr uint32_t kCountLeastGroups = 128;             // so that a workgroup's own entries are fewer than its threads
static_assert(kCountEntries < 1u << 16, "counts of half a word");
static_assert(kCountEntries / kCountLeastGroups + kMaxTopK <= kCountThreads && kMaxExperts <= kCountThreads, "one per thread");

__host__ __device__ constexpr uint32_t CountCopiesLog(uint32_t experts)
{
    return experts <= 16 ? 6 : experts <= 64 ? 4 : 2;
}

// [experts][copies] counts, [experts] first rows, a sum per wave, whether an id is out of range, the rows of the own entries, [slices][experts] of those
constexpr uint32_t CountLdsWords(uint32_t experts, uint32_t ownMost)
{
    return (experts << CountCopiesLog(experts)) + experts + kCountWaves + 1 + ownMost + (ownMost + 63) / 64 * experts;
}

// The lines lie where the token rows and the stored rows together, in bytes, change what a store should do.
// Up to kQuickBytes nontemporal stores: they are on their way at once, where plain ones wait in an XCD's L2 for the end of
// the launch (dispatch and combine in turn, 400 tokens of 2048 elements at top-8: 10.7 us, 11.4 with plain ones).  Beyond, plain
// stores leave the rows in the last-level cache, where the next kernel finds them (1000 of 5120 at top-8: 31.2, 35.5 with
// nontemporal ones; 1500 of 2048 21.8, 23.6).  From kCountNearBytes on nontemporal loads and twice as many of them ahead keep the token rows
// from taking turns with them (2400 of 7168 at top-2: dispatch 19.4, 25.9 without; before kCountNearBytes the longer code
// costs 0.5).  Calls of few slots read most: from kCountDeepBytes on plain stores cost them more than the next kernel
// gains (4096 of 7168 at top-2, dispatch / both: nontemporal 28.6 / 57.4, plain 36.5 / 56.0).
// What fits the last-level cache (256 MiB) too little goes to the tiles: they are the quicker dispatch from about 300 MiB on, but pass that cache with their
// stores, where this leaves a part of the rows for the next kernel.  The line follows the whole: dispatch, a kernel that reads the rows and writes
// others of their size, and the combine of those.  Dispatch / all three with the tiles and so, us, three sets of buffers in turn, 7168 elements: top-8 over
// 256 experts, 262 MiB 60.9 / 191, 53.7 / 180; 310 65.1 / 222, 64.3 / 211; 350 67.3 / 246, 75.6 / 240; 400 84.7 / 289, 86.6 / 274; 430 85.4 / 304, 93.3 / 297, but of 4096
// elements over 64 72.5 / 292, 94.6 / 295.  Top-6 310 58.2 / 215, 66.9 / 206; 366 69.9 / 261, 80.4 / 246.  Top-4 290 59.6 / 199, 51.3 / 196; 310 60.4 / 211, 54.3 / 208; 334
// 61.4 / 225, 58.6 / 227.  Top-2 270 59.2 / 164, 58.9 / 164.  64 and 128 experts as 256; over 8 the next kernel finds the rows of the tiles better: top-8 270
// 62.1 / 185, 56.7 / 180, 310 62.8 / 204, 65.2 / 206, 350 63.2 / 225, 75.8 / 234; top-4 270 50.0 / 173, 48.4 / 178.  Rows that are not whole cache lines are always
// stored plainly: two waves share a line.
constexpr uint64_t kQuickBytes = 24ull << 20;            // also of the dispatch above
constexpr uint64_t kQuickFewBytes = 16ull << 20;         // with up to two slots, whose next kernel reads the rows sooner
constexpr uint64_t kCountNearBytes = 96ull << 20;
constexpr uint64_t kCountDeepBytes = 150ull << 20;
constexpr uint32_t kCountFewExperts = 64;                // below
constexpr uint64_t CountBytes(uint32_t topK, uint32_t experts, bool lines)
{
    return (topK <= 2 || experts < kCountFewExperts || !lines ? 256ull : topK <= 4 ? 320ull : topK <= 6 ? 368ull : 400ull) << 20;
}

template <bool kNt>
__device__ __forceinline__ u32x4 RowLoad(const MF_GLOBAL u32x4 *p)
{
    return kNt ? __builtin_nontemporal_load(p) : *p;
}

template <uint32_t kAhead, int kMode, bool kNtLoad>
__global__ __launch_bounds__(kCountThreads) void MoeDispatchCountKernel(uint64_t x, uint64_t topkAt, uint32_t total, uint32_t topK,
                                                                        uint32_t experts, uint32_t unitsPerRow, uint32_t perGroup,
                                                                        uint64_t out, uint64_t countsAt, uint64_t offsetsAt,
                                                                        uint64_t rowOfAt, uint64_t srcOfAt, uint64_t statusAt)
{
    const int32_t *const topk = Buffer<const int32_t>(topkAt);
    int32_t *const counts = Buffer<int32_t>(countsAt);
    int32_t *const offsets = Buffer<int32_t>(offsetsAt);
    int32_t *const rowOf = Buffer<int32_t>(rowOfAt);
    int32_t *const srcOf = Buffer<int32_t>(srcOfAt);
    extern __shared__ uint32_t lds[];
    const uint32_t lane = threadIdx.x & 63u;
    const uint32_t wave = threadIdx.x >> 6;
    const uint32_t copiesLog = CountCopiesLog(experts);
    const uint32_t ownMost = perGroup * topK;
    const uint32_t slices = (ownMost + 63) / 64;
    uint32_t *count = lds;
    uint32_t *base = count + (experts << copiesLog);
    uint32_t *scan = base + experts;
    uint32_t *rows = scan + kCountWaves + 1;
    uint32_t *anyBad = scan + kCountWaves;
    uint32_t *hist = rows + ownMost;
    const uint32_t begin = blockIdx.x * ownMost;
    const uint32_t end = begin + ownMost < total ? begin + ownMost : total;
    // the ids before the rows: everything waits for them.  The last vector ends with the last id.
    i32x4a id[kCountBatch];
#pragma unroll
    for (uint32_t q = 0; q < kCountBatch; ++q) {
        const uint32_t at = (q * kCountThreads + threadIdx.x) * 4;
        id[q] = *reinterpret_cast<const i32x4a *>(topk + (at + 3 < total ? at : total - 4));
    }
    const uint32_t own = begin + threadIdx.x;
    const int32_t ownId = own < end ? topk[own] : -1;
    const uint32_t tokens = (end - begin) / topK;
    const uint32_t parts = (unitsPerRow + 63) / 64;     // pieces of 64 units
    const uint32_t items = x != 0 ? tokens * parts : 0;
    const MF_GLOBAL u32x4 *src = reinterpret_cast<const MF_GLOBAL u32x4 *>(x) +
                                 static_cast<uint64_t>(blockIdx.x) * perGroup * unitsPerRow;
    MF_GLOBAL u32x4 *dst = reinterpret_cast<MF_GLOBAL u32x4 *>(out);
    u32x4 v[kAhead];
#pragma unroll
    for (uint32_t j = 0; j < kAhead; ++j) {
        const uint32_t item = wave + j * kCountWaves;
        if (item < items) {
            const uint32_t token = item / parts;
            const uint32_t u = (item - token * parts) * 64 + lane;
            if (u < unitsPerRow) {
                v[j] = RowLoad<kNtLoad>(src + static_cast<uint64_t>(token) * unitsPerRow + u);
            }
        }
    }
    for (uint32_t i = threadIdx.x; i < experts << copiesLog; i += kCountThreads) {
        count[i] = 0;
    }
    for (uint32_t i = threadIdx.x; i < slices * experts; i += kCountThreads) {
        hist[i] = 0;
    }
    if (threadIdx.x == 0) {
        *anyBad = 0;
    }
    __syncthreads();
    uint32_t bad = 0;
    uint32_t *counting = count + (lane & ((1u << copiesLog) - 1u));
    for (uint32_t from = 0; from < total; from += kCountBatch * kCountThreads * 4) {
#pragma unroll
        for (uint32_t q = 0; q < kCountBatch; ++q) {
            if (from + q * kCountThreads * 4 >= total) {
                break;
            }
            const uint32_t at = from + (q * kCountThreads + threadIdx.x) * 4;
#pragma unroll
            for (uint32_t i = 0; i < 4; ++i) {
                const uint32_t index = at + 3 < total ? at + i : total - 4 + i;
                if (index >= at) {
                    const uint32_t e = static_cast<uint32_t>(id[q][i]);
                    if (e < experts) {
                        atomicAdd(&counting[e << copiesLog], index < begin ? 0x10001u : 1u);   // plain counts: the same whatever the order
                    } else {
                        bad = 1;
                    }
                }
            }
        }
        if (from + kCountBatch * kCountThreads * 4 < total) {
#pragma unroll
            for (uint32_t q = 0; q < kCountBatch; ++q) {
                const uint32_t at = from + ((kCountBatch + q) * kCountThreads + threadIdx.x) * 4;
                id[q] = *reinterpret_cast<const i32x4a *>(topk + (at + 3 < total ? at : total - 4));
            }
        }
    }
    uint32_t rank = 0;
    const bool valid = static_cast<uint32_t>(ownId) < experts;
    if (wave < slices) {
        const uint64_t peers = PeersOf(static_cast<uint32_t>(ownId), valid, BitsFor(experts));
        const uint64_t below = peers & ((1ull << lane) - 1ull);
        rank = __popcll(below);
        if (valid && below == 0) {
            hist[wave * experts + static_cast<uint32_t>(ownId)] = __popcll(peers);
        }
    }
    if (bad != 0) {
        *anyBad = 1;
    }
    __syncthreads();
    uint32_t all = 0;
    uint32_t before = 0;
    if (threadIdx.x < experts) {
        for (uint32_t c = 0; c < 1u << copiesLog; c += 4) {
            const u32x4 w = *reinterpret_cast<const u32x4 *>(&count[(threadIdx.x << copiesLog) + c]);
#pragma unroll
            for (uint32_t i = 0; i < 4; ++i) {
                all += w[i] & 0xFFFFu;
                before += w[i] >> 16;
            }
        }
    }
    uint32_t incl = all;
#pragma unroll
    for (uint32_t step = 1; step < 64; step <<= 1) {
        const uint32_t up = __shfl_up(incl, step, 64);
        incl += lane >= step ? up : 0u;
    }
    if (lane == 63) {
        scan[wave] = incl;                              // experts of a wave: the sums in front of theirs are added by who asks
    }
    if (threadIdx.x < experts) {
        base[threadIdx.x] = incl - all + before;
    }
    __syncthreads();
    if (blockIdx.x == 0) {
        if (threadIdx.x < experts) {
            uint32_t run = incl - all;
            for (uint32_t w = 0; w < wave; ++w) {
                run += scan[w];
            }
            counts[threadIdx.x] = static_cast<int32_t>(all);
            offsets[threadIdx.x] = static_cast<int32_t>(run);
        }
        if (threadIdx.x == 0) {
            *Buffer<uint32_t>(statusAt) = *anyBad;
        }
    }
    if (own < end) {
        uint32_t row = 0xFFFFFFFFu;
        if (valid) {
            const uint32_t e = static_cast<uint32_t>(ownId);
            row = base[e] + rank;
            for (uint32_t w = 0; w < e >> 6; ++w) {
                row += scan[w];
            }
            for (uint32_t s = 0; s < wave; ++s) {
                row += hist[s * experts + e];
            }
            if (srcOfAt != 0) {
                srcOf[row] = static_cast<int32_t>(own);
            }
        }
        rows[threadIdx.x] = row;
        rowOf[own] = static_cast<int32_t>(row);
    }
    __syncthreads();
    // the next piece is requested into the registers of the one that was stored
    for (uint32_t first = wave; first < items; first += kAhead * kCountWaves) {
#pragma unroll
        for (uint32_t j = 0; j < kAhead; ++j) {
            const uint32_t item = first + j * kCountWaves;
            if (item < items) {
                const uint32_t token = item / parts;
                const uint32_t u = (item - token * parts) * 64 + lane;
                for (uint32_t k = 0; k < topK; ++k) {
                    const uint32_t row = __builtin_amdgcn_readfirstlane(rows[token * topK + k]);
                    if (row != 0xFFFFFFFFu && u < unitsPerRow) {
                        RowStore<kMode>(dst + static_cast<uint64_t>(row) * unitsPerRow + u, v[j]);
                    }
                }
                const uint32_t next = item + kAhead * kCountWaves;
                if (next < items) {
                    const uint32_t nextToken = next / parts;
                    const uint32_t nextU = (next - nextToken * parts) * 64 + lane;
                    if (nextU < unitsPerRow) {
                        v[j] = RowLoad<kNtLoad>(src + static_cast<uint64_t>(nextToken) * unitsPerRow + nextU);
                    }
                }
            }
        }
    }
}

__device__ __forceinline__ float Bf16Lo(uint32_t w)
{
    return __uint_as_float(w << 16);
}

__device__ __forceinline__ float Bf16Hi(uint32_t w)
{
    return __uint_as_float(w & 0xFFFF0000u);
}

// Two results in one word, each rounded to nearest even; NaN stays a quiet NaN, subnormal numbers stay what they are: one
// v_cvt_pk_bf16_f32, which gives what the eight integer operations per value that it replaces gave, for all 2^32 inputs.
typedef float f32x2 __attribute__((ext_vector_type(2)));
typedef __bf16 bf16x2 __attribute__((ext_vector_type(2)));
__device__ __forceinline__ uint32_t ToBf16Pair(float lo, float hi)
{
    return __builtin_bit_cast(uint32_t, __builtin_convertvector(f32x2{lo, hi}, bf16x2));
}

// The columns [begin, end) of one token.  kAllLive: every slot has a row, which is the usual case and needs no
// branch per slot.
template <uint32_t kTopK, uint32_t kThreads, bool kNtLoad, uint32_t kBatch, bool kAllLive, uint32_t kSlots = kTopK != 0 ? kTopK : kMaxTopK>
__device__ __forceinline__ void CombineColumns(const MF_GLOBAL u32x4 *in, MF_GLOBAL u32x4 *dst, const uint64_t (&rowBase)[kSlots],
                                               const float (&w)[kSlots], uint32_t live, uint32_t begin, uint32_t end)
{
    // kBatch column positions per lane are requested together (kBatch * K loads in flight per lane)
    // before any of them is consumed.
    for (uint32_t u0 = begin + threadIdx.x; u0 < end; u0 += kBatch * kThreads) {
        u32x4 v[kBatch][kSlots];
#pragma unroll
        for (uint32_t b = 0; b < kBatch; ++b) {
            const uint32_t u = u0 + b * kThreads;
#pragma unroll
            for (uint32_t k = 0; k < kSlots; ++k) {
                if ((kAllLive || ((live >> k) & 1u) != 0) && u < end) {
                    v[b][k] = kNtLoad ? __builtin_nontemporal_load(in + rowBase[k] + u) : in[rowBase[k] + u];
                }
            }
        }
#pragma unroll
        for (uint32_t b = 0; b < kBatch; ++b) {
            const uint32_t u = u0 + b * kThreads;
            if (u >= end) {
                break;
            }
            float acc[8];
#pragma unroll
            for (uint32_t i = 0; i < 8; ++i) {
                acc[i] = 0.0f;
            }
#pragma unroll
            for (uint32_t k = 0; k < kSlots; ++k) {
                if (kAllLive || ((live >> k) & 1u) != 0) {
#pragma unroll
                    for (uint32_t i = 0; i < 4; ++i) {
                        acc[2 * i] = __builtin_fmaf(w[k], Bf16Lo(v[b][k][i]), acc[2 * i]);
                        acc[2 * i + 1] = __builtin_fmaf(w[k], Bf16Hi(v[b][k][i]), acc[2 * i + 1]);
                    }
                }
            }
            u32x4 o;
#pragma unroll
            for (uint32_t i = 0; i < 4; ++i) {
                o[i] = ToBf16Pair(acc[2 * i], acc[2 * i + 1]);
            }
            __builtin_nontemporal_store(o, dst + u);
        }
    }
}

// Calls whose dispatch is one launch and whose buffers, this much together, stay in the last-level cache (256 MiB, used by others
// too) find the rows there: plain loads, and one column position per lane, so that twice as many waves each do half as much.
// What bounds those calls is the chain of one wave; before, a test per slot stood between any two loads and each result took
// sixteen integer operations to round, code that is fetched anew in every launch.  Dispatch and combine in turn, of 7168
// elements at top-8 (before / all slots tested at once and the rounding in one instruction / this): 16 tokens 11.0 / 8.2 / 7.1 us,
// 64 12.4 / 10.4 / 10.1, 256 16.2 / 15.9 / 14.7, 512 26.2 / 30.5 / 25.2; combine alone 64 tokens 5.7 / 3.7 / 3.1.  Beyond, plain loads
// lose: 2048 tokens at top-2, 117 MB, 27.5 us without and 30.1 with them, 1000 at top-8 52.8 and 61.2.  Larger calls gain from the shorter
// code alone: 1500 tokens 76.8 -> 74.3 us.
constexpr uint64_t kCombineCachedBytes = 80ull << 20;
constexpr uint32_t kCombineCachedEntries = 4096;        // measured with rows that were stored past the caches; rows in them change nothing (29 shapes)

template <uint32_t kTopK, uint32_t kThreads, bool kNtLoad, uint32_t kBatch = 1>
__global__ __launch_bounds__(kThreads) void MoeCombineKernel(uint64_t rowsIn, uint64_t rowOfAt, uint64_t weightsAt, uint32_t topK,
                                                             uint32_t unitsPerRow, uint32_t parts, uint64_t y)
{
    const int32_t *const rowOf = Buffer<const int32_t>(rowOfAt);
    const float *const weights = Buffer<const float>(weightsAt);
    const uint32_t token = blockIdx.x / parts;
    const uint32_t part = blockIdx.x - token * parts;
    const uint32_t perPart = (unitsPerRow + parts - 1) / parts;
    const uint32_t begin = part * perPart;
    const uint32_t end = begin + perPart < unitsPerRow ? begin + perPart : unitsPerRow;
    const uint32_t nk = kTopK != 0 ? kTopK : topK;
    constexpr uint32_t kSlots = kTopK != 0 ? kTopK : kMaxTopK;
    uint64_t rowBase[kSlots];
    float w[kSlots];
    // Slots without a row (an expert id that dispatch flagged) are skipped: neither loaded nor
    // multiplied, so whatever lies in row 0 (an infinity, a NaN) cannot reach y through 0 * x.
    // The mask is the same for every lane of the workgroup.
    uint32_t live = 0;
#pragma unroll
    for (uint32_t k = 0; k < kSlots; ++k) {
        if (k < nk) {
            const int32_t row = rowOf[static_cast<uint64_t>(token) * nk + k];
            rowBase[k] = static_cast<uint64_t>(row < 0 ? 0 : row) * unitsPerRow;
            w[k] = weights[static_cast<uint64_t>(token) * nk + k];
            live |= row < 0 ? 0u : 1u << k;
        } else {
            rowBase[k] = 0;
            w[k] = 0.0f;
        }
    }
    const MF_GLOBAL u32x4 *in = reinterpret_cast<const MF_GLOBAL u32x4 *>(rowsIn);
    MF_GLOBAL u32x4 *dst = reinterpret_cast<MF_GLOBAL u32x4 *>(y) +
                           static_cast<uint64_t>(token) * unitsPerRow;
    if (kTopK != 0 && live == (1u << nk) - 1u) {
        CombineColumns<kTopK, kThreads, kNtLoad, kBatch, true>(in, dst, rowBase, w, live, begin, end);
    } else {
        CombineColumns<kTopK, kThreads, kNtLoad, kBatch, false>(in, dst, rowBase, w, live, begin, end);
    }
}

// The combine of wide rows when there are many tokens: gridDim.x single-wave workgroups, all
// resident at once, walk the items (token, 128-unit slice of the row) with stride gridDim.x.
// HBM streams reads at 7.0 TB/s and the combine's mix of eight reads to one write at 6.0, so
// the two are kept apart in time: a period is kItems read parts and one write part.  In read
// part j a wave requests the 16 pieces of its j-th item of the period (eight rows, two column
// positions per lane) at its own offset of the part, reduces them when they have arrived and
// keeps the result in LDS; in the write part it stores the kItems results at
// its own offset of that part (top-6: six rows, twelve pieces).  The start of the first period is agreed through
// AgreedStart(); after that every wave goes by the constant-rate clock alone.  8192 tokens of 7168
// elements at top-8: 162 us against 177-181 us for one workgroup per item.  Read parts are paced at 6.8 TB/s, write parts at 6.5.
// HBM is the bound.  Results in registers, four an item (116 of them), left room for 4096 waves: 5120 have a quarter more time for loads that come late in as
// much longer parts.  Combine, and dispatch and combine, us, 4096 waves at 6.8 and 6.2 / 5120 at 6.8 and 6.5: 8192 tokens of 7168 elements at top-8 over 256 experts 165.8 / 161.5, 352.7 / 349.6, over
// 8 166.1 / 163.1, 336.2 / 334.3, at top-6 129.9 / 126.0, 275.8 / 271.1, of 5120 117.9 / 116.0, 245.3 / 243.9, of 4096, two whole periods before and now an eighth more, 92.9 / 93.6, 190.5 / 190.7;
// 3600 of 7168 74.5 / 73.2, 155.4 / 154.2 (five processes each in turn, within 0.5).  Reads at 6.85 make the waves fall behind behind a
// dispatch, whose rows are still on their way out of the last-level cache (350).  Not taken: 6144 waves (80 registers spill), four results (LDS for 18 waves, 346).
// Arithmetic and the rule for slots without a row are MoeCombineKernel's.
constexpr uint32_t kCombineItems = 3;                  // of which the results, 2 KiB each, wait in LDS
constexpr uint32_t kCombineWavesPerSimd = 5;           // 90 registers
constexpr uint32_t kCombineWavesPerCu = 4 * kCombineWavesPerSimd;
constexpr uint32_t kCombineSliceUnits = 128;           // two column positions per lane
constexpr uint32_t kCombineMinItemsPerCu = 96;

template <uint32_t kItems, uint32_t kSlots>
__global__ __launch_bounds__(64) __attribute__((amdgpu_waves_per_eu(kCombineWavesPerSimd, kCombineWavesPerSimd))) void MoeCombineWindowKernel(const u32x4 *__restrict__ rowsIn,
                                                             const int32_t *__restrict__ rowOf,
                                                             const float *__restrict__ weights, uint32_t unitsPerRow,
                                                             uint32_t parts, uint32_t items, u32x4 *__restrict__ y,
                                                             uint32_t readTicks, uint32_t writeTicks, uint32_t seq)
{
    constexpr uint32_t kBatch = kCombineSliceUnits / 64;
    const uint64_t start = AgreedStart(seq);
    const uint32_t period = kItems * readTicks + writeTicks;
    const uint32_t readOffset = static_cast<uint32_t>(static_cast<uint64_t>(blockIdx.x) * readTicks / gridDim.x);
    const uint32_t writeOffset = static_cast<uint32_t>(static_cast<uint64_t>(blockIdx.x) * writeTicks / gridDim.x);
    const uint32_t perPart = (unitsPerRow + parts - 1) / parts;
    const MF_GLOBAL u32x4 *in = reinterpret_cast<const MF_GLOBAL u32x4 *>(reinterpret_cast<uint64_t>(rowsIn));
    MF_GLOBAL u32x4 *out = reinterpret_cast<MF_GLOBAL u32x4 *>(reinterpret_cast<uint64_t>(y));
    __shared__ u32x4 o[kItems][kBatch][64];
    uint64_t t0 = start;
    for (uint32_t base = 0; base < items; base += kItems * gridDim.x, t0 += period) {
        if (base + blockIdx.x >= items) {
            break;                                     // nothing left for this wave
        }
        // The last period holds as many read parts as it has items per wave, and its last read part lasts as long
        // as the waves that still have an item need to request it (both the same for every wave).
        const uint32_t remaining = items - base;
        const uint32_t left = (remaining + gridDim.x - 1) / gridDim.x;
        const uint32_t readParts = left < kItems ? left : kItems;
        const uint32_t inLastPart = remaining - (readParts - 1) * gridDim.x;       // >= 1
        const uint32_t lastPartTicks = inLastPart >= gridDim.x ? readTicks
            : static_cast<uint32_t>(static_cast<uint64_t>(inLastPart) * readTicks / gridDim.x);
        const uint32_t readEnd = (readParts - 1) * readTicks + lastPartTicks;
#pragma unroll
        for (uint32_t j = 0; j < kItems; ++j) {
            const uint32_t item = base + j * gridDim.x + blockIdx.x;
            if (j < readParts && item < items) {
                const uint32_t token = item / parts;
                const uint32_t begin = (item - token * parts) * perPart;
                const uint32_t end = begin + perPart < unitsPerRow ? begin + perPart : unitsPerRow;
                // No branch on a slot without a row (rowOf < 0): its pieces are read from the token's own row
                // of y, which is memory this launch owns, masked to zero and multiplied by -0.0f, and
                // fma(-0.0f, 0.0f, acc) is acc for every acc, so the slot contributes nothing, as if skipped.
                const MF_GLOBAL u32x4 *rowPtr[kSlots];
                float w[kSlots];
                uint32_t keep[kSlots];
#pragma unroll
                for (uint32_t k = 0; k < kSlots; ++k) {
                    const int32_t row = rowOf[static_cast<uint64_t>(token) * kSlots + k];
                    const float weight = weights[static_cast<uint64_t>(token) * kSlots + k];
                    rowPtr[k] = row < 0 ? out + static_cast<uint64_t>(token) * unitsPerRow
                                        : in + static_cast<uint64_t>(row) * unitsPerRow;
                    w[k] = row < 0 ? -0.0f : weight;
                    keep[k] = row < 0 ? 0u : 0xFFFFFFFFu;
                }
                WaitForClock(t0 + j * readTicks + readOffset);
                u32x4 v[kBatch][kSlots];
#pragma unroll
                for (uint32_t b = 0; b < kBatch; ++b) {
                    const uint32_t u = begin + b * 64 + threadIdx.x;
                    if (u < end) {
#pragma unroll
                        for (uint32_t k = 0; k < kSlots; ++k) {
                            v[b][k] = __builtin_nontemporal_load(rowPtr[k] + u);
                        }
                    }
                }
#pragma unroll
                for (uint32_t b = 0; b < kBatch; ++b) {
                    float acc[8];
                    u32x4 sum;
#pragma unroll
                    for (uint32_t i = 0; i < 8; ++i) {
                        acc[i] = 0.0f;
                    }
#pragma unroll
                    for (uint32_t k = 0; k < kSlots; ++k) {
#pragma unroll
                        for (uint32_t i = 0; i < 4; ++i) {
                            const uint32_t word = v[b][k][i] & keep[k];
                            acc[2 * i] = __builtin_fmaf(w[k], Bf16Lo(word), acc[2 * i]);
                            acc[2 * i + 1] = __builtin_fmaf(w[k], Bf16Hi(word), acc[2 * i + 1]);
                        }
                    }
#pragma unroll
                    for (uint32_t i = 0; i < 4; ++i) {
                        sum[i] = ToBf16Pair(acc[2 * i], acc[2 * i + 1]);
                    }
                    o[j][b][threadIdx.x] = sum;
                }
            }
        }
        WaitForClock(t0 + readEnd + writeOffset);
#pragma unroll
        for (uint32_t j = 0; j < kItems; ++j) {
            const uint32_t item = base + j * gridDim.x + blockIdx.x;
            if (j < readParts && item < items) {
                const uint32_t token = item / parts;
                const uint32_t begin = (item - token * parts) * perPart;
                const uint32_t end = begin + perPart < unitsPerRow ? begin + perPart : unitsPerRow;
#pragma unroll
                for (uint32_t b = 0; b < kBatch; ++b) {
                    const uint32_t u = begin + b * 64 + threadIdx.x;
                    if (u < end) {
                        __builtin_nontemporal_store(o[j][b][threadIdx.x], out + static_cast<uint64_t>(token) * unitsPerRow + u);
                    }
                }
            }
        }
    }
}

// Which XCD a wave runs on (XCC_ID, hardware register 20, bits 3:0), for mfk_moe_setup().
__global__ void XcdProbeKernel(uint32_t *__restrict__ ids)
{
    if (threadIdx.x == 0) {
        ids[blockIdx.x] = static_cast<uint32_t>(__builtin_amdgcn_s_getreg((3 << 11) | 20)) & 0xFu;
    }
}

// 1 once mfk_moe_setup() has seen consecutive workgroups go to kTileStreams different XCDs in turn, which is what the
// streams of MoePermuteTileKernel stand on; 0 (the loop kernel is used) before that and where the GPU deals them
// otherwise (a partition of one XCD, for instance).
std::atomic<int> g_xcdStreams{0};

// Pace of the windowed combine, MB/s of HBM traffic in the read parts and in the write parts; 0 = never windowed.
std::atomic<uint32_t> g_combineReadMBps{6800000};
std::atomic<uint32_t> g_combineWriteMBps{6500000};

uint32_t CombineWaves()
{
    return static_cast<uint32_t>(mfrt_cu_count() > 0 ? mfrt_cu_count() : 256) * kCombineWavesPerCu;
}

// The dispatch in one launch that counts: where the lines lie, see those.
bool DispatchCounts(uint64_t entries, uint64_t moved, uint32_t topK, uint32_t experts, bool lines)
{
    return entries <= kCountEntries && moved <= CountBytes(topK, experts, lines);
}

// The dispatch in one launch that compares: where the lines lie, see MoeDispatchSmallKernel.
bool DispatchCompares(uint64_t entries, uint32_t topK)
{
    return entries <= kSmallEntries && entries * topK <= (topK <= 8 ? kSmallCompares : kSmallManyCompares);
}

// Whether waves that stay and keep reads and writes apart in time combine rows of at least 256 units: from 96 slices per CU on (top-8, 16 800 items
// on 4096 waves of 16 a CU 51.4 us, one workgroup per item 50.5; 19 200 the same; 25 200 74.4 / 76.7), below which the first read part and the last write part, in
// which the chip only reads or only writes for want of work, cost what the separation gains; and where the last-level cache does not hold the rows that
// the kernel before has just written.  Rows written by an elementwise kernel and combined, with windows from three items on / from six on / in rows
// that a dispatch leaves there, us: top-8 3.6 to 5.9 items of 2048 elements a row, 262 MiB of rows and tokens 125.1 / 119.4, 310 146.3 / 141.2, 430 201.7 / 196.9; top-6
// 290 MiB 132.7 / 127.9; and 6.2 items of 7168 elements at top-6, 350 MiB - / 163.8 / 159.8, 366 - / 171.1 / 166.5.  (Directly behind a dispatch
// whose stores pass that cache windows gain 2 to 3 % from three items on; a program's experts lie between.)
// Top-6 gains as top-8 does (8192 x 7168: 131-133 against 138-140 us); top-4 gains nothing (98 against 97 us)
// and top-2 loses (16 384 x 4096: 79 against 66 us): their read parts are too short for the switch to pay.
bool CombineInWindows(uint32_t tokens, uint32_t hidden, uint32_t topK, uint32_t &readTicks, uint32_t &writeTicks)
{
    const uint32_t upr = hidden / 8;
    const uint32_t parts = (upr + kCombineSliceUnits - 1) / kCombineSliceUnits;
    const uint32_t perPart = (upr + parts - 1) / parts;
    const uint64_t items = static_cast<uint64_t>(tokens) * parts;
    const uint64_t entries = static_cast<uint64_t>(tokens) * topK;
    const uint32_t waves = CombineWaves();
    if ((topK != 6 && topK != 8) || upr < 256 || items < static_cast<uint64_t>(waves / kCombineWavesPerCu) * kCombineMinItemsPerCu || items >= 0x40000000ull ||
        DispatchCounts(entries, (entries + tokens) * upr * 16, topK, kMaxExperts, hidden % 64 == 0)) {
        return false;
    }
    readTicks = WindowPeriodTicks(static_cast<uint64_t>(waves) * topK * perPart * 16, g_combineReadMBps.load(std::memory_order_relaxed));
    writeTicks = WindowPeriodTicks(static_cast<uint64_t>(waves) * kCombineItems * perPart * 16,
                                   g_combineWriteMBps.load(std::memory_order_relaxed));
    return readTicks != 0 && writeTicks != 0;
}

}  // namespace
}  // namespace mf

extern "C" uint64_t mfk_moe_workspace_bytes(uint32_t tokens, uint32_t topK, uint32_t experts)
{
    const uint64_t total = static_cast<uint64_t>(tokens) * topK;
    const uint64_t blocks = (total + mf::kRankBlock - 1) / mf::kRankBlock;
    const uint64_t stride = (blocks + mf::kHistPad - 1) / mf::kHistPad * mf::kHistPad;
    // status words, per-block flags, the [expert][block] histogram, the run-ordered row list (8 bytes per entry slot)
    const uint64_t tables = 256 + stride * sizeof(uint32_t) + stride * experts * sizeof(uint32_t);
    return (tables + 15) / 16 * 16 + blocks * mf::kRankBlock * sizeof(int2);
}

extern "C" int mfk_moe_dispatch(const void *x, const void *topk, uint32_t tokens, uint32_t hidden, uint32_t topK,
                                uint32_t experts, void *out, void *counts, void *offsets, void *rowOf, void *srcOf,
                                void *workspace, void *stream)
{
    using namespace mf;
    const uint64_t total64 = static_cast<uint64_t>(tokens) * topK;
    if (total64 == 0 || total64 > 0x7FFFFFFFull || experts == 0 || experts > kMaxExperts || topK > kMaxTopK ||
        (static_cast<uint64_t>(hidden) * 2) % 16 != 0) {
        return -1;
    }
    const uint32_t total = static_cast<uint32_t>(total64);
    const uint32_t blocks = (total + kRankBlock - 1) / kRankBlock;
    hipStream_t s = static_cast<hipStream_t>(stream);
    uint32_t *status = static_cast<uint32_t *>(workspace);
    const uint32_t histStride = (blocks + kHistPad - 1) / kHistPad * kHistPad;   // rows of the [expert][block] table
    uint32_t *blockBad = status + 64;
    uint32_t *blockHist = blockBad + histStride;
    const size_t histLds = static_cast<size_t>(kRankSlices) * experts * sizeof(uint32_t);
    const uint32_t upr = hidden / 8;
    const bool rows = x != nullptr && out != nullptr && hidden != 0;
    const uint64_t moved = rows ? (static_cast<uint64_t>(tokens) + total) * upr * 16 : 0;
    const bool lines = hidden % 64 == 0;                // rows of whole cache lines
    const bool quick = lines && moved <= (topK <= 2 ? kQuickFewBytes : kQuickBytes);
    if (DispatchCompares(total, topK)) {
        const uint32_t least = (upr + kSmallHold * kSmallThreads - 1) / (kSmallHold * kSmallThreads);
        const uint32_t most = (upr + 63) / 64;
        uint32_t parts = (kSmallGroups + tokens - 1) / tokens;
        parts = parts < least ? least : parts > most ? most : parts;
        const uint32_t perPart = rows ? ((upr + parts - 1) / parts + 7) / 8 * 8 : 0;   // whole cache lines
        parts = rows ? (upr + perPart - 1) / perPart : 1;
#define MF_DISPATCH_SMALL(SLOTS)                                                                                       \
    return Launch(quick ? MoeDispatchSmallKernel<SLOTS, 1> : MoeDispatchSmallKernel<SLOTS, 0>, tokens * parts + 1, kSmallThreads, 0, s, At(x), \
                  At(topk), total, topK, experts, upr, parts, perPart, tokens * parts + 1, At(out), At(counts), At(offsets), At(rowOf),          \
                  At(srcOf), At(workspace))
        if (topK <= 2) {
            MF_DISPATCH_SMALL(2);
        } else if (topK <= 4) {
            MF_DISPATCH_SMALL(4);
        } else if (topK <= 8) {
            MF_DISPATCH_SMALL(8);
        } else {
            MF_DISPATCH_SMALL(16);
        }
#undef MF_DISPATCH_SMALL
    }
    if (DispatchCounts(total, moved, topK, experts, lines)) {
        const uint32_t cus = static_cast<uint32_t>(mfrt_cu_count() > 0 ? mfrt_cu_count() : 256);
        const uint32_t most = cus < kCountLeastGroups ? kCountLeastGroups : cus;
        const uint32_t perGroup = (tokens + most - 1) / most;
        const uint32_t lds = CountLdsWords(experts, perGroup * topK) * sizeof(uint32_t);
#define MF_DISPATCH_COUNT(AHEAD, MODE, NT)                                                                             \
    return Launch(MoeDispatchCountKernel<AHEAD, MODE, NT>, (tokens + perGroup - 1) / perGroup, kCountThreads, lds, s, rows ? At(x) : 0, \
                  At(topk), total, topK, experts, upr, perGroup, At(out), At(counts), At(offsets), At(rowOf), At(srcOf), At(workspace))
        if (quick || (lines && topK <= 4 && moved > kCountDeepBytes)) {
            MF_DISPATCH_COUNT(4, 1, false);
        } else if (moved <= kCountNearBytes) {
            MF_DISPATCH_COUNT(4, 0, false);
        } else {
            MF_DISPATCH_COUNT(8, 0, true);
        }
#undef MF_DISPATCH_COUNT
    }
    // The output-ordered tile permute needs the token rows of one step (a block of kRankBlock entries, or a half, a
    // quarter ... down to one slice of 64 entries: stepEntries / topK tokens) to stay in an XCD's 4 MiB L2 while the
    // step's rows are written, and enough steps for the eight streams.  It wins on every shape of whole cache lines
    // that was measured (8192 tokens, top-8, 256 experts, 7168 elements: 174 against 208 us with the loop kernel;
    // 1024 elements: 44 against 49 us with one workgroup per token).  Rows that are not whole cache lines
    // (10 000 elements) lose, whatever the step: every tile then begins and ends inside a line; they keep the loop kernel.
    // Where steps of whole blocks and of several lie, and why: see kTileStepBytes.
    uint32_t restSlices = kRankSlices;
    while (restSlices > 1 && static_cast<uint64_t>(restSlices * 64 / topK + 1) * hidden * 2 > 2200000ull) {
        restSlices /= 2;
    }
    // a call of few blocks is cut finer, so that every XCD gets steps to work on
    while (restSlices > 1 && static_cast<uint64_t>(blocks) * (kRankSlices / restSlices) < 2 * kTileStreams) {
        restSlices /= 2;
    }
    const uint32_t tilesPerRow = (upr + kTileUnits - 1) / kTileUnits;
    const auto tileGridOf = [&](uint32_t longBlocks, uint32_t slices) {     // longBlocks: whole rounds of them
        const uint64_t restSteps = static_cast<uint64_t>(blocks - longBlocks) * (kRankSlices / slices);
        return (static_cast<uint64_t>(longBlocks) * kRankBlock + (restSteps + kTileStreams - 1) / kTileStreams * kTileStreams * slices * 64) * tilesPerRow;
    };
    const bool tiles = g_xcdStreams.load(std::memory_order_relaxed) != 0 && x != nullptr && out != nullptr && upr >= kTileUnits &&
                       hidden % 64 == 0 && static_cast<uint64_t>(restSlices * 64 / topK + 1) * hidden * 2 <= 2200000ull &&
                       kRankSlices / restSlices * experts <= 4096 && tileGridOf(0, restSlices) <= 0x7FFFFFFFull;
    // Up to kCountingBlocks blocks rank without a histogram launch in front of them: every block counts the entries
    // of the others itself.  Dispatch of rows of 1024 elements, with the launch / so: 2200 tokens at top-8 over 256 experts (18 blocks)
    // 20.1 / 17.6 us, 3000 (24) 19.7 / 18.3, 4096 (32) 22.2 / 22.0 (of 7168 elements 90.3 / 90.6).  The counts of a wave land on few LDS
    // words when the experts are few: over 64, 12 blocks 15.7 / 13.8, 16 34.5 / 34.0, 24 63.6 / 63.9 (longer rows); over 8, 16 blocks
    // 19.7 / 20.2.  (The short ones of these have one launch by now.)
    const bool counting = blocks <= (experts >= 128 ? kCountingBlocks : experts >= 64 ? 16u : 8u);
    uint32_t together = 1;
    const auto stepFits = [&](uint32_t m) { return static_cast<uint64_t>(kRankBlock / topK) * m * hidden * 2 <= kTileStepBytes; };
    if (tiles && !counting && topK > kTileWholeSlots && hidden * 2 >= kTileTogetherRowBytes &&
        (experts > kTileFewExperts || (experts == kTileFewExperts && hidden * 2 >= kTileLongRowBytes))) {
        while (static_cast<uint64_t>(kRankBlock) * together * hidden * 2 < kTileRunBytes * experts && stepFits(2 * together) &&
               2 * together <= kTileMostTogether && blocks >= 2 * together * kTileStreams) {
            together *= 2;
        }
    }
    const uint32_t longRounds = together > 1 ? blocks / (together * kTileStreams) : 0;
    const uint32_t blocksTogether = longRounds * together * kTileStreams;
    uint32_t wholeRounds = 0;
    if (tiles && (restSlices == kRankSlices || (topK >= kTileWholeSlots && stepFits(1))) && blocks >= 2 * kTileStreams) {
        wholeRounds = (blocks - blocksTogether) / kTileStreams;
    }
    const uint32_t blocksWhole = blocksTogether + wholeRounds * kTileStreams;
    if (wholeRounds != 0 || blocksTogether != 0) {
        while ((blocks - blocksWhole) * (kRankSlices / restSlices) % kTileStreams != 0 &&
               kRankSlices / restSlices * 2 * experts <= 4096) {
            restSlices /= 2;
        }
    }
    const uint32_t stepsPerBlock = kRankSlices / restSlices;
    const size_t rankLds = histLds + (experts + kRankThreads + kRankSlices + (tiles ? stepsPerBlock * experts : 0) +
                                      (counting || blocksTogether != 0 ? experts : 0)) * sizeof(uint32_t);
    const uint64_t tableBytes = 256 + histStride * sizeof(uint32_t) + static_cast<uint64_t>(histStride) * experts * sizeof(uint32_t);
    int2 *runOrder = tiles ? reinterpret_cast<int2 *>(static_cast<char *>(workspace) + (tableBytes + 15) / 16 * 16) : nullptr;
    const uint64_t rowBytes = static_cast<uint64_t>(upr) * 16;
    const bool warms = tiles && tokens * rowBytes >= kWarmMinBytes;
    const uint64_t warmUnits = !warms ? 0 : (tokens * rowBytes < kWarmMaxBytes ? tokens * rowBytes : kWarmMaxBytes) / 16;
    const bool warmsMore = warmUnits * 16 >= kWarmMoreBytes && blocks <= kWarmMoreBlocks;
    const uint64_t warmFirst = counting ? 0 : warmUnits * (warmsMore ? kWarmMoreHistPercent : kWarmHistPercent) / 100;
    const uint32_t warmGroups = !warms ? 0 : warmsMore ? kWarmMoreGroups : kWarmGroups;
    const u32x4 *warm = static_cast<const u32x4 *>(x);
    if (counting) {
        blockHist = nullptr;
    } else {
        hipLaunchKernelGGL(MoeHistKernel, dim3(blocks + warmGroups), dim3(kRankThreads), histLds, s, static_cast<const int32_t *>(topk),
                           total, experts, blockHist, histStride, blockBad, blocks, warm, warmFirst);
    }
    hipLaunchKernelGGL(MoeRankKernel, dim3(blocks + warmGroups), dim3(kRankThreads), rankLds, s, static_cast<const int32_t *>(topk),
                       total, experts, blockHist, histStride, static_cast<int32_t *>(counts), static_cast<int32_t *>(offsets),
                       static_cast<int32_t *>(rowOf), static_cast<int32_t *>(srcOf), blockBad, status, topK, runOrder, restSlices,
                       together, blocksTogether, blocksWhole, blocks, warm + warmFirst, warmUnits - warmFirst);
    if (x != nullptr && out != nullptr && hidden != 0) {
        const u32x4 *xi = static_cast<const u32x4 *>(x);
        const int32_t *ro = static_cast<const int32_t *>(rowOf);
        u32x4 *oo = static_cast<u32x4 *>(out);
        if (tiles) {
            const TilePlan plan{blocks * kRankBlock, together * kRankBlock, longRounds, wholeRounds, restSlices * 64};
            hipLaunchKernelGGL(MoePermuteTileKernel, dim3(static_cast<uint32_t>(tileGridOf(blocksWhole, restSlices))), dim3(64), 0, s, xi, runOrder,
                               upr, tilesPerRow, plan, oo);
        } else if (upr >= 512) {
            // Wide rows: single-wave workgroups that hold up to 14 pieces per lane (a whole 7168-element
            // row) and write them with plain stores; sixteen waves per CU that each take several tokens and
            // fetch the next row while they store the current one (207 us for 8192 x 7168 at top-8; staging in
            // LDS, two waves per row, nontemporal stores and the destination-side form were all slower).
            // 123 vector registers per lane: four waves per SIMD, sixteen per CU, all resident at once
            const uint32_t wideParts = (upr + 64 * 14 - 1) / (64 * 14);
            const uint32_t items = tokens * wideParts;
            const uint32_t waves = static_cast<uint32_t>(mfrt_cu_count() > 0 ? mfrt_cu_count() : 256) * 16u;
            hipLaunchKernelGGL((MoePermuteLoopKernel<14>), dim3(items < waves ? items : waves), dim3(64), 0, s, xi, ro, topK, upr,
                               wideParts, items, oo);
        } else {
            // Narrow rows: one four-wave workgroup per token.
            hipLaunchKernelGGL((MoePermuteKernel<256, 4, 1>), dim3(tokens), dim3(256), 0, s, xi, ro, topK, upr, 1u, oo);
        }
    }
    return static_cast<int>(hipGetLastError());
}

extern "C" int mfk_moe_combine(const void *rows, const void *rowOf, const void *weights, uint32_t tokens,
                               uint32_t hidden, uint32_t topK, void *y, void *stream, int paced)
{
    using namespace mf;
    if (tokens == 0 || topK == 0 || topK > kMaxTopK || hidden == 0 || (static_cast<uint64_t>(hidden) * 2) % 16 != 0) {
        return -1;
    }
    hipStream_t s = static_cast<hipStream_t>(stream);
    const u32x4 *in = static_cast<const u32x4 *>(rows);
    const int32_t *ro = static_cast<const int32_t *>(rowOf);
    const float *w = static_cast<const float *>(weights);
    u32x4 *o = static_cast<u32x4 *>(y);
    const uint32_t upr = hidden / 8;
    const uint64_t traffic = static_cast<uint64_t>(tokens) * (topK + 2) * upr * 16;   // the rows, the tokens they came from, the result
    const bool fanIn = topK == 2 || topK == 4 || topK == 6 || topK == 8;
    if (upr >= 256 && fanIn && static_cast<uint64_t>(tokens) * topK <= kCombineCachedEntries && traffic <= kCombineCachedBytes) {
        // One column position per lane and plain loads: where the line lies, see kCombineCachedBytes.
        const uint32_t parts = (upr + 63) / 64;
#define MF_COMBINE_CACHED(K) return Launch(MoeCombineKernel<K, 64, false, 1>, tokens * parts, 64, 0, s, At(rows), At(rowOf), At(weights), topK, upr, parts, At(y))
        if (topK == 2) {
            MF_COMBINE_CACHED(2);
        } else if (topK == 4) {
            MF_COMBINE_CACHED(4);
        } else if (topK == 6) {
            MF_COMBINE_CACHED(6);
        } else {
            MF_COMBINE_CACHED(8);
        }
#undef MF_COMBINE_CACHED
    } else if (upr >= 256 && fanIn) {
        // Wide rows: single-wave workgroups, each on a 128-unit slice of the row with two column positions per
        // lane in flight (2 x topK loads), the fastest shape measured on 7168-element rows at top-8 (178 us; one
        // four-wave workgroup per token 188 us; plain instead of nontemporal loads 194 us).  Compiled for the common
        // fan-ins, so that all of a lane's loads are in flight together: top-2 16 384 x 4096 65 against 74 us,
        // top-4 8192 x 7168 96 against 106 us, top-6 139 against 152 us (against the kernel that walks a run-time
        // number of slots).
        const uint32_t parts = (upr + kCombineSliceUnits - 1) / kCombineSliceUnits;
        const uint64_t items = static_cast<uint64_t>(tokens) * parts;
        const uint32_t waves = CombineWaves();
        uint32_t readTicks = 0;
        uint32_t writeTicks = 0;
        const bool windows = paced != 0 && CombineInWindows(tokens, hidden, topK, readTicks, writeTicks);
        const uint32_t grid = windows ? waves : tokens * parts;
#define MF_COMBINE_SLICES(K)                                                                                           \
    return Launch(MoeCombineKernel<K, 64, true, 2>, grid, 64, 0, s, At(rows), At(rowOf), At(weights), topK, upr, parts, At(y))
#define MF_COMBINE_WINDOWS(K)                                                                                          \
    hipLaunchKernelGGL((MoeCombineWindowKernel<kCombineItems, K>), dim3(grid), dim3(64), 0, s, in, ro, w, upr, parts,        \
                       static_cast<uint32_t>(items), o, readTicks, writeTicks, NextWindowSeq())
        if (topK == 2) {
            MF_COMBINE_SLICES(2);
        } else if (topK == 4) {
            MF_COMBINE_SLICES(4);
        } else if (topK == 6) {
            if (windows) {
                MF_COMBINE_WINDOWS(6);
            } else {
                MF_COMBINE_SLICES(6);
            }
        } else if (windows) {
            MF_COMBINE_WINDOWS(8);
        } else {
            MF_COMBINE_SLICES(8);
        }
#undef MF_COMBINE_SLICES
#undef MF_COMBINE_WINDOWS
    } else {
        // Narrow rows: one four-wave workgroup per token, compiled for the common fan-ins too, whose loads are then in flight together.
#define MF_COMBINE_TOKEN(K) return Launch(MoeCombineKernel<K, 256, true, 1>, tokens, 256, 0, s, At(rows), At(rowOf), At(weights), topK, upr, 1u, At(y))
        if (topK == 2) {
            MF_COMBINE_TOKEN(2);
        } else if (topK == 4) {
            MF_COMBINE_TOKEN(4);
        } else if (topK == 6) {
            MF_COMBINE_TOKEN(6);
        } else if (topK == 8) {
            MF_COMBINE_TOKEN(8);
        } else {
            MF_COMBINE_TOKEN(0);
        }
#undef MF_COMBINE_TOKEN
    }
    return static_cast<int>(hipGetLastError());
}

extern "C" int mfk_moe_dispatch_counts(uint32_t tokens, uint32_t hidden, uint32_t topK, uint32_t experts)
{
    const uint64_t entries = static_cast<uint64_t>(tokens) * topK;
    return !mf::DispatchCompares(entries, topK) && mf::DispatchCounts(entries, (entries + tokens) * (hidden / 8) * 16, topK, experts, hidden % 64 == 0) ? 1 : 0;
}

extern "C" int mfk_moe_combine_stays(uint32_t tokens, uint32_t hidden, uint32_t topK)
{
    uint32_t readTicks = 0;
    uint32_t writeTicks = 0;
    return mf::CombineInWindows(tokens, hidden, topK, readTicks, writeTicks) ? 1 : 0;
}

extern "C" void mfk_moe_combine_windows(uint32_t readMBps, uint32_t writeMBps)
{
    mf::g_combineReadMBps.store(readMBps, std::memory_order_relaxed);
    mf::g_combineWriteMBps.store(writeMBps, std::memory_order_relaxed);
}

// Once per process, after the GPU has been bound and outside any stream capture (it waits for a small kernel):
// checks that workgroup i of a launch runs on XCD i mod 8.
extern "C" int mfk_moe_setup(void)
{
    constexpr uint32_t kProbe = 256;
    uint32_t *dev = nullptr;
    hipError_t err = hipMalloc(reinterpret_cast<void **>(&dev), kProbe * sizeof(uint32_t));
    if (err != hipSuccess) {
        return static_cast<int>(err);
    }
    uint32_t ids[kProbe];
    hipLaunchKernelGGL(mf::XcdProbeKernel, dim3(kProbe), dim3(64), 0, nullptr, dev);
    err = hipMemcpy(ids, dev, sizeof(ids), hipMemcpyDeviceToHost);
    (void)hipFree(dev);
    if (err != hipSuccess) {
        return static_cast<int>(err);
    }
    bool inTurn = true;
    for (uint32_t i = 0; i < kProbe; ++i) {
        inTurn = inTurn && ids[i] == ids[i % mf::kTileStreams];
    }
    for (uint32_t a = 0; a < mf::kTileStreams; ++a) {
        for (uint32_t b = a + 1; b < mf::kTileStreams; ++b) {
            inTurn = inTurn && ids[a] != ids[b];
        }
    }
    mf::g_xcdStreams.store(inTurn ? 1 : 0, std::memory_order_relaxed);
    return 0;
}

extern "C" int mfk_moe_xcd_streams(void)
{
    return mf::g_xcdStreams.load(std::memory_order_relaxed);
}
