// Work decomposition shared by the host planner and the xcopy kernels.
//
// A batch is a list of segments {src, dst, len} (the reference's uint64
// triples, src/hybm/csrc/data_operation/host/hybm_data_op_sdma.cpp:520-528).
// Each segment is cut into "chunks", the unit one workgroup copies in one
// loop iteration, so that work is proportional to bytes and not to segment
// count (the reference's kernel gives every core count/32 whole segments,
// src/hybm/csrc/copy_extend/hybm_copy_kernel.cpp:102-104).
//
// Geometry of one segment (all derived from dst, len and the chunk size):
//   head  = bytes until dst reaches a 16-byte boundary (capped at len)
//   body  = the following floor((len-head)/16) 16-byte units; stores are aligned
//   tail  = the remaining (len-head) % 16 bytes
//   chunk k covers body units [k*U, min((k+1)*U, body)); chunk 0 also copies
//   the head, the last chunk also copies the tail.  A segment of len > 0 has
//   max(1, ceil(body/U)) chunks, a segment of len 0 has none.
//
// This header is plain C++ (no HIP types) so the host planner and its CPU
// tests can include it.
#ifndef MF_XCOPY_PLAN_H
#define MF_XCOPY_PLAN_H

#include <stdint.h>

namespace mf {

constexpr uint32_t kXcopyThreads = 256;       // most lanes a copy workgroup has (4 wave64); 4 KiB chunks get one wave
constexpr uint32_t kUnitBytes = 16;           // one 128-bit access
constexpr uint32_t kInlineSegs = 128;         // segments that fit in the kernel-argument block: 2 table rows per lane of a wave64
constexpr uint32_t kNoChunk = 0xFFFFFFFFu;    // sentinel prefix for unused slots

#if defined(__HIPCC__)
#define MF_HD __host__ __device__
#else
#define MF_HD
#endif

struct SegGeom {
    uint32_t head;     // 0..15
    uint32_t tail;     // 0..15
    uint64_t body;     // 16-byte units
};

MF_HD inline SegGeom SegmentGeometry(uint64_t dst, uint64_t len)
{
    SegGeom g;
    uint64_t h = (0 - dst) & (kUnitBytes - 1);
    if (h > len) {
        h = len;
    }
    g.head = static_cast<uint32_t>(h);
    g.body = (len - h) / kUnitBytes;
    g.tail = static_cast<uint32_t>((len - h) % kUnitBytes);
    return g;
}

// Chunks of a segment for `units` 16-byte units per chunk.
MF_HD inline uint64_t SegmentChunks(uint64_t dst, uint64_t len, uint32_t units)
{
    if (len == 0) {
        return 0;
    }
    SegGeom g = SegmentGeometry(dst, len);
    uint64_t n = (g.body + units - 1) / units;
    return n == 0 ? 1 : n;
}

// The same with its cuts where the destination reaches a multiple of kLineBytes: the first chunk is shorter by what the
// destination lies behind one, and no two chunks write one cache line.
constexpr uint32_t kLineBytes = 128;
MF_HD inline uint64_t LineChunks(uint64_t dst, uint64_t len, uint32_t units)
{
    const uint64_t each = static_cast<uint64_t>(units) * kUnitBytes;
    return len == 0 ? 0 : ((dst & (kLineBytes - 1)) + len + each - 1) / each;
}

// Bytes [begin, end) of such a segment that chunk k < LineChunks() holds.
struct LineSpan {
    uint64_t begin;
    uint64_t end;
};
MF_HD inline LineSpan LineChunk(uint64_t dst, uint64_t len, uint64_t k, uint32_t units)
{
    const uint64_t each = static_cast<uint64_t>(units) * kUnitBytes;
    const uint64_t skip = dst & (kLineBytes - 1);
    const uint64_t end = (k + 1) * each - skip;
    return LineSpan{k == 0 ? 0 : k * each - skip, end < len ? end : len};
}

// Everything a launch of up to kInlineSegs segments needs, passed by value in
// the kernel-argument block (3080 bytes of the 4096 available): no table
// upload, no extra dependent memory round trip before the first data load.
struct InlinePlan {
    uint64_t src[kInlineSegs];
    uint64_t dst[kInlineSegs];
    uint32_t len[kInlineSegs];          // inline path carries segments < 4 GiB only
    uint32_t first[kInlineSegs];        // exclusive prefix of chunk counts, kNoChunk past the end
    uint32_t nchunk;
    uint32_t units;                     // 16-byte units per chunk, a multiple of 64
};

// Stores held back: how long after its start a wave of the inline kernel waits before it stores.
//
// A launch of a few thousand single-chunk waves has every load in flight within two microseconds and
// would store as the data trickle in, so HBM sees reads and writes mixed.  When every wave keeps its four
// loaded registers until the loads of the whole launch are out, the reads run as one burst and the
// writes as another: a 2196-chunk batch takes 4.5 instead of 5.3 us.  The wait is counted from the start
// of the wave, is the same for every wave, and grows with the number of waves the dispatcher has to start
// (a line fitted to sweeps over 976 ... 7076 chunks; it aims 50 to 100 ns long, because falling 200 ns short
// loses the gain while each 100 ns beyond costs 0.1 us).  It pays only while every wave of the launch is
// resident at once (up to 24 single-wave workgroups per CU) and only for launches that do not overlap
// others on purpose.  A single segment has no table to fetch and gets a line of its own.
constexpr uint32_t kHoldMinChunks = 960;        // table in the kernel arguments
constexpr uint32_t kHoldKneeChunks = 3904;
constexpr uint32_t kHoldMinChunksSingle = 1400; // one segment
constexpr uint32_t kHoldMaxChunks = 6144;
constexpr uint32_t kHoldSharedMaxChunks = 4096; // the limit while several threads submit on streams of their own
// Beyond kHoldMaxChunks chunks of 4 KiB the waves of a launch are no longer resident together.  Batches of up to
// kDeepMaxChunks chunks of kDeepUnits units (16 KiB, sixteen loads per lane in flight: 64 MiB in 4096 waves, 16 per CU)
// are, and hold their stores the same way.
constexpr uint32_t kDeepUnits = 1024;
constexpr uint32_t kDeepMaxChunks = 4096;
constexpr uint64_t kDeepMinBytes = static_cast<uint64_t>(kHoldMaxChunks) * kXcopyThreads * kUnitBytes;   // 24 MiB
constexpr uint64_t kDeepMaxBytes = static_cast<uint64_t>(kDeepMaxChunks) * kDeepUnits * kUnitBytes;      // 64 MiB
constexpr uint32_t kHeldMaxPieces = 7168;          // waves of XcopyPieceHeldKernel that are resident together, 28 per CU
constexpr uint64_t kHeldSingleBytes = static_cast<uint64_t>(kHeldMaxPieces) * kDeepUnits * kUnitBytes - kLineBytes;   // wherever its lines begin
constexpr uint32_t kHoldMaxNanos = 20000;
constexpr uint64_t kDeepMinSegmentBytes = 32768;   // on average: short segments make chunks that are not whole
inline uint32_t DeepRuleNanos(uint32_t count)
{
    return 600 + count * 215 / 100;
}
inline uint32_t HoldNanosFor(uint32_t nchunk, uint32_t grid, uint32_t units, bool single)
{
    if (units == kDeepUnits && grid == nchunk && nchunk <= (single ? kHeldMaxPieces : kDeepMaxChunks)) {
        // fitted to sweeps over 1664 ... 4096 waves (26 to 64 MiB in 32 segments, one segment, 100 ragged ones): the best wait is
        // 600 ns and 2.15 ns per 16 KiB, a read rate of 7.6 TB/s; up to 10 % beyond costs 1 to 3 %, 10 % short loses half the gain
        // (a single segment's waves know their chunk at once, so the reads are over sooner: best waits of 26 to 117 MB in steps of
        // 500 ns 500 to 1000 shorter, 500 where source and destination differ modulo 16; that much more costs 2 to 4 %)
        return nchunk < kHoldMinChunks / 4 ? 0 : DeepRuleNanos(nchunk) - (single ? 500 : 0);
    }
    if (units != kXcopyThreads || grid != nchunk || nchunk > kHoldMaxChunks) {
        return 0;   // only launches of one chunk per single-wave workgroup were measured
    }
    if (single) {
        return nchunk < kHoldMinChunksSingle ? 0 : 100 + nchunk * 57 / 100;
    }
    if (nchunk < kHoldMinChunks) {
        return 0;
    }
    if (nchunk <= kHoldKneeChunks) {
        return 640 + nchunk * 6 / 10;
    }
    return 640 + kHoldKneeChunks * 6 / 10 + (nchunk - kHoldKneeChunks) * 33 / 100;
}

// Counters of the workgroups of a launch that says itself when it is done: one, and beyond kDoneFewGroups workgroups
// kDoneCounters more, on lines of their own, in front of it.
constexpr uint32_t kDoneFewGroups = 64;
constexpr uint32_t kDoneCounters = 32;
constexpr uint32_t kDoneCounterWords = 32;
constexpr uint64_t kDoneCounterBytes = (1 + kDoneCounters) * kDoneCounterWords * sizeof(uint32_t);

// On top of HoldNanosFor's rule where the waves of a launch have to look their descriptors up outside the kernel arguments, a
// round trip across the host link before their loads, and the same on 16 KiB chunks: sixteen loads per lane take longer to leave.
constexpr int32_t kHoldLookupExtraNanos = 1600;
constexpr int32_t kHoldLookupDeepExtraNanos = 2000;

// Wait of a launch of pieces of 16 KiB beyond kDeepMinBytes.  Best waits in steps of 400 ns, us: 28 / 40 / 56 / 72 / 88 / 104 MB of pages or blocks
// gathered and scattered 4.9 / 6.4 to 6.9 / 8.9 / 11.2 / 13.5 / 15.8, a read rate of 6.9 TB/s; where segments are cut into pieces that are not full
// 0.7 ns less for each that is missing, up to a thousand (88 MB in segments of 100 000 bytes 12.7); half as much less at odd addresses, where a piece reads
// lines at both ends that others read too (70 MB in segments of up to 70 000 bytes 25.7 us without, 25.4 so, 66 / 92 MB of up to 128 KiB 23.7 / 23.6, 32.8 /
// 32.5; two launches of 48 / 59 MB 36.1 / 36.4, 44.4 / 44.7), and nothing less where a segment is a piece (28 /
// 36 MB in segments of 5120 bytes 4.5 / 5.8, 45 / 58 MB of 8 KiB 7.3 / 9.2).  400 ns more or less cost 1 to 2 %.
inline uint32_t PieceMissing(uint32_t count, uint64_t bytes)
{
    const uint64_t full = bytes / (kDeepUnits * kUnitBytes);
    return count > full ? count - static_cast<uint32_t>(full) : 0;
}
constexpr uint32_t kPieceLessMissing = 1000;
inline uint64_t PieceDeepNanos(uint32_t count, uint64_t bytes)
{
    const uint64_t wait = 830 + bytes / 6930;
    const uint64_t missing = PieceMissing(count, bytes);
    const uint64_t less = missing < kPieceLessMissing ? missing * 7 / 10 : kPieceLessMissing * 7 / 10;
    return wait > less ? wait - less : 0;
}
inline uint32_t PieceWholeNanos(uint32_t count, uint64_t bytes)
{
    const uint32_t missing = PieceMissing(count, bytes);
    return (missing < kPieceLessMissing ? missing * 7 / 10 : kPieceLessMissing * 7 / 10) + missing / 10;
}

// What a launch of `count` pieces waits of the time a table of as many chunks would.  Its descriptors arrive eight to a line, and
// kPieceLeadNanos sooner than three words per wave did; and ragged pieces are not full, so that the reads are over sooner: by
// the rate of the rule above for the bytes that are not there.  Best waits beyond HoldNanosFor(count): K and V blocks of 10 / 18 /
// 24 MB +400 / 200 / 400 ns; ragged segments of 14 / 21 MB 0.
// Pieces of 8 and 16 KiB of a batch of up to kDeepMinBytes wait as its chunks of 4 KiB would, but for the knee of that rule: best
// waits beyond it with K and V blocks of 18 / 20 / 22 MB 0 / 40 / 250 ns, 23 MB of pages 300, on 8 KiB 8 / 16 / 25 MB of pages 200 / -100 / 300.
// Of 16 KiB beyond, PieceDeepNanos.
constexpr uint32_t kPieceLeadNanos = 1400;
constexpr uint64_t kPieceKneeBytes = 18000000;
inline uint32_t PieceLessNanos(uint32_t count, uint64_t bytes, uint32_t units)
{
    if (units != kXcopyThreads && bytes <= kDeepMinBytes) {
        return kPieceLeadNanos - (bytes > kPieceKneeBytes ? static_cast<uint32_t>((bytes - kPieceKneeBytes) * 7 / 100000) : 0);
    }
    if (units == kDeepUnits && count <= kHeldMaxPieces) {
        const uint64_t rule = DeepRuleNanos(count) + kHoldLookupDeepExtraNanos;
        const uint64_t wait = PieceDeepNanos(count, bytes);
        return rule > wait ? static_cast<uint32_t>(rule - wait) : 0;
    }
    const uint64_t full = static_cast<uint64_t>(count) * units * kUnitBytes;
    const uint64_t missing = full > bytes ? (full - bytes) / kUnitBytes : 0;                 // units
    return static_cast<uint32_t>(kPieceLeadNanos + missing * (units != kXcopyThreads ? 215 : 180) / (100ull * kDeepUnits));
}
inline uint32_t PieceHoldNanos(uint32_t holdNanos, uint32_t count, uint64_t bytes, uint32_t units)
{
    const uint32_t less = PieceLessNanos(count, bytes, units);
    return holdNanos > less ? holdNanos - less : 0;
}

// The start of a windowed launch's first period travels between its waves as the low kEpochClockBits bits of a
// clock value (2^40 ticks of 10 ns: three hours) under a sequence number; NearClock restores the full value: the
// one with those low bits that is nearest to `now`.
constexpr uint32_t kEpochClockBits = 40;
MF_HD inline uint64_t NearClock(uint64_t now, uint64_t low)
{
    const uint64_t mask = (1ull << kEpochClockBits) - 1;
    uint64_t t = (now & ~mask) | low;
    if (t > now && t - now > (mask >> 1)) {
        t -= mask + 1;
    } else if (t < now && now - t > (mask >> 1)) {
        t += mask + 1;
    }
    return t;
}

// Chunk counts that repeat with a short period: pages of one size (period 1), K and V blocks
// taking turns (period 2), ...  With such a pattern the owner of a chunk follows from a division
// and at most kMaxPeriod comparisons, and no chunk prefix is needed.
constexpr uint32_t kMaxPeriod = 8;

struct ChunkPattern {
    uint32_t period;                    // 0: no pattern, the chunk prefix is searched
    uint32_t chunksPerPeriod;
    uint32_t start[kMaxPeriod + 1];     // exclusive prefix of the counts inside one period; start[period] == chunksPerPeriod
};

// Segment and chunk-in-segment of global chunk c under a pattern.  Every start[] is read at a fixed index, so
// that a kernel keeps the pattern in scalar registers (the member that owns r is the last one whose start
// is <= r, and starts never decrease, so the hits form a prefix and the last hit's start is the owner's).
MF_HD inline void PatternOwner(const ChunkPattern &p, uint32_t c, uint32_t &seg, uint32_t &k)
{
    const uint32_t group = c / p.chunksPerPeriod;
    const uint32_t r = c - group * p.chunksPerPeriod;
    uint32_t j = 0;
    uint32_t base = 0;
    for (uint32_t i = 1; i < kMaxPeriod; ++i) {
        const bool hit = i < p.period && p.start[i] <= r;
        j += hit ? 1u : 0u;
        base = hit ? p.start[i] : base;
    }
    seg = group * p.period + j;
    k = r - base;
}

// Chunks of the first nseg segments under a pattern.
MF_HD inline uint64_t PatternChunks(const ChunkPattern &p, uint32_t nseg)
{
    return static_cast<uint64_t>(nseg / p.period) * p.chunksPerPeriod + p.start[nseg % p.period];
}

// Group map of a table without a pattern.  The chunks are taken in groups of 2^shift; group[g] is the
// segment that owns chunk g << shift, and one more entry names the segment that owns the last chunk.
// The owner of chunk c then lies in [group[g], group[g + 1]] with g = c >> shift, a range the 64 lanes
// of a wave probe in one round whenever it spans at most 64 segments: the lookup is two dependent loads
// instead of a search over the whole prefix.  A group of 2^shift chunks touches at most 2^shift + 1
// segments that are not empty, so groups of 32 chunks always resolve in that one round (groups of 64
// would need a second one for a run of 65 single-chunk segments).  The shift grows until the map fits
// the room there is for it.
constexpr uint32_t kGroupShiftMin = 5;

MF_HD constexpr inline uint32_t GroupCount(uint64_t nchunk, uint32_t shift)
{
    return static_cast<uint32_t>((nchunk + (1ull << shift) - 1) >> shift);
}

// Smallest shift from kGroupShiftMin on whose map (GroupCount + 1 entries) fits `capacity` entries.
MF_HD constexpr inline uint32_t GroupShiftFor(uint64_t nchunk, uint32_t capacity)
{
    uint32_t shift = kGroupShiftMin;
    while (shift < 32 && static_cast<uint64_t>(GroupCount(nchunk, shift)) + 1 > capacity) {
        ++shift;
    }
    return shift;
}

// Room the engine gives the map of a table of nseg segments: the finest groups for every table whose chunks
// number up to 32 times that (2 M chunks, 8 GiB in 4 KiB chunks, at the least), coarser ones beyond.
MF_HD constexpr inline uint32_t GroupCapacityFor(uint32_t nseg)
{
    return (nseg > 65536u ? nseg : 65536u) + 1u;
}

// Host-side build of the map from a finished prefix (first[0 .. nseg], first[nseg] == nchunk != 0); returns the shift.
// group: room for `capacity` entries.
inline uint32_t BuildGroupMap(const uint32_t *first, uint32_t nseg, uint32_t *group, uint32_t capacity)
{
    const uint32_t nchunk = first[nseg];
    const uint32_t shift = GroupShiftFor(nchunk, capacity);
    const uint32_t ngroups = GroupCount(nchunk, shift);
    uint32_t last = 0;
    for (uint32_t i = 0; i < nseg; ++i) {
        const uint32_t f = first[i];
        const uint32_t cnt = first[i + 1] - f;
        if (cnt == 0) {
            continue;
        }
        last = i;
        const uint32_t gLo = static_cast<uint32_t>((static_cast<uint64_t>(f) + (1ull << shift) - 1) >> shift);
        const uint32_t gHi = (f + cnt - 1) >> shift;
        for (uint64_t g = gLo; g <= gHi; ++g) {
            group[g] = i;
        }
    }
    group[ngroups] = last;
    return shift;
}

// A batch of more than kInlineSegs segments between HBM addresses, cut up by the host: one piece, one workgroup, one step.
// A piece is 16 bytes in pinned host memory, addresses of 56 bits and a length of 16 in the bytes above them.  Inside a segment
// pieces end where the destination reaches a multiple of kPieceAlign, so that no two workgroups write one cache line; all but
// the last are of one length.
constexpr uint32_t kPieceAlign = 128;
constexpr uint32_t kPieceGroup = 64;
constexpr uint32_t kPieceMaxCount = 1u << 23;      // below 2^32 lanes in a launch
struct Piece {
    uint64_t src;
    uint64_t dst;
};
static_assert(sizeof(Piece) == 16, "eight pieces make a line");
constexpr uint64_t kPieceAddress = (1ull << 56) - 1;
MF_HD inline Piece MakePiece(uint64_t src, uint64_t dst, uint32_t len)
{
    return Piece{(src & kPieceAddress) | static_cast<uint64_t>(len & 0xFFu) << 56, (dst & kPieceAddress) | static_cast<uint64_t>(len >> 8) << 56};
}
MF_HD inline uint32_t PieceLength(uint64_t src, uint64_t dst)
{
    return static_cast<uint32_t>(src >> 56) | static_cast<uint32_t>(dst >> 56) << 8;
}
// Which piece a workgroup copies.  Consecutive workgroups go to the eight XCDs in turn, and an XCD fetches descriptors over the
// host link by lines of eight: the eight of a line go to one XCD, which is then the only one to fetch it (4096 pages of 32 KiB in
// pieces of 4 KiB: 45.8 us, 101 with the pieces dealt out in their order), and 64 workgroups still copy 64 consecutive pieces
// (with an eighth of the whole list for each XCD: 51.6).
MF_HD inline uint32_t PieceOf(uint32_t workgroup)
{
    return (workgroup & ~(kPieceGroup - 1)) | (workgroup & 7u) << 3 | (workgroup >> 3 & 7u);
}

// A table that only the GPU can read, copied without a plan.  Its launch takes `parts` items per segment, part j of a segment
// copying the chunks j, j + parts, ... of it: right for every table, whatever `parts` is, and evenly spread where `parts` is near
// the chunk count of the usual segment.  That is taken from the first kDirectSample segments, by every wave for itself.
// A part copies kDirectRounds chunks at most; a segment that holds more than parts * kDirectRounds chunks is listed for a second
// launch, which cuts what is left of the listed segments into pieces, so that no wave is left with a long segment.
constexpr uint32_t kDirectSample = 8;
constexpr uint32_t kDirectMaxParts = 64;
constexpr uint32_t kDirectRounds = 4;
constexpr uint64_t kRestPieceBytes = 64ull << 10;
constexpr uint32_t kRestShare = 16;                   // pieces side by side whose workgroups take their chunks in turn
constexpr uint32_t kRestLanes = 512;                  // of a workgroup of the second launch between HBM addresses

// A table of up to kPlannedSegments segments between HBM addresses is planned by every workgroup of its one launch for itself: one
// wave, or sixteen for more than 512 segments, whose lanes take a run of them each.  Up to kPlannedShallowChunks chunks of 4 KiB it is
// cut into those, else into 16 KiB, whose stores are held up to kPlannedHeldChunks of 4 KiB.
constexpr uint32_t kPlannedShortRun = 8;
constexpr uint32_t kPlannedWaves = 16;
constexpr uint32_t kPlannedRun = 4;
constexpr uint32_t kPlannedSegments = 64 * kPlannedWaves * kPlannedRun;
constexpr uint32_t kPlannedFullPercent = 85;          // pieces of 16 KiB that are less full gain nothing from windows,
constexpr uint32_t kPlannedLoosePercent = 94;         // and those that are less full than this hold a higher rate wherever they lie
constexpr uint64_t kWindowLongBlockBytes = 64ull << 10;   // blocks of one length from here on, at multiples of it, hold a higher rate in any order
constexpr uint64_t kSampledMostBytes = 1ull << 20;         // of a segment of a longer table that goes by what its first ones are: fewer than 2^32 chunks
constexpr uint32_t kPlannedShallowChunks = 1024;
constexpr uint32_t kPlannedHeldChunks = 16384;
// What the last piece of 16 KiB of a segment lacks, in 256 bytes, and the payload of `deep` such pieces that lack `spare`, in 4 KiB.
// A sum over what is missing stays small where one over the lengths would pass 32 bits, however long the segments are.  (Lanes that
// counted 512 MiB at the most took longer segments for pieces that are not full: 8 of 1 GiB 3.26 to 3.33 ms without windows, 2.87
// in windows; 3 of 2 GiB 2.43 to 2.48 and 2.15.)
MF_HD inline uint32_t PlannedSpare(uint64_t len)
{
    return (((0u - static_cast<uint32_t>(len)) & 16383u) + 255u) >> 8;
}
MF_HD inline uint32_t PlannedTotal(uint32_t deep, uint32_t spare)
{
    return deep * 4 - (spare + 15) / 16;
}
MF_HD inline bool PlannedFull(uint32_t total, uint32_t deep)
{
    return static_cast<uint64_t>(total) * 100 >= static_cast<uint64_t>(deep) * (4 * kPlannedFullPercent);
}
constexpr uint32_t PlannedLds(uint32_t waves, uint32_t nseg)          // bytes: the prefix, and four words of each wave
{
    return (nseg + 1 + 4 * waves) * 4;
}
constexpr int32_t kTableHoldNanos = 2000;             // held stores of device tables: the wait,
constexpr uint32_t kTableHoldMoreNanos = 8800;        // and what more for 64 MiB (K and V blocks of 32, 48, 62 MB want 600 to 1200 less, ragged ones at odd addresses 300 more);
constexpr int32_t kTableEqualNanos = 850;             // of tables of segments of one length, whose waves load that much sooner: best
constexpr uint32_t kTableEqualMoreNanos = 9850;       // waits in steps of 400 ns 5.6 to 5.9 us at 33 MB, 10.2 to 10.6 at 62 to 65 MB

struct RestSegment {                                  // what is left of a long segment
    uint64_t first;                                   // pieces of those listed before
    uint64_t src;
    uint64_t dst;
    uint64_t len;
};
struct RestCount {                                    // on a line of its own
    uint64_t count;
    uint64_t reserved[15];
};
constexpr uint32_t kRestGroups = 16;
// One entry a segment, however long: a list with room for a table's segments holds what any table of them leaves.  All counts are 0
// between calls.  `taken` counts entries and pieces in one word, which makes `first` ascend with the entries.
struct RestList {
    uint64_t taken;                                   // entries * kRestEntry + pieces
    uint64_t reserved[15];
    RestCount done[kRestGroups + 1];                  // workgroups of the second launch that are done with it, by group, and groups
    RestSegment entry[1];                             // as many as the list has room for
};
constexpr uint64_t kRestHeadBytes = sizeof(RestList) - sizeof(RestSegment);
constexpr uint64_t kRestEntry = 1ull << 40;           // pieces of 64 KiB: 2^56 bytes
constexpr uint32_t kRestCapacity = 65536;             // 2 MiB; a longer table goes in several pairs of launches
constexpr uint32_t kRestGraphCapacity = 16384;        // of the lists for calls recorded into a graph
constexpr uint64_t RestListBytes(uint32_t capacity)
{
    return sizeof(RestList) + static_cast<uint64_t>(capacity - 1) * sizeof(RestSegment);
}
MF_HD inline uint64_t RestPieces(uint64_t left)
{
    return (left + kRestPieceBytes - 1) / kRestPieceBytes;
}

// A table-driven launch: triples, prefix and group map live in device memory (under a pattern the
// triples may sit in pinned host memory and the other two are not read).
struct TablePlan {
    const uint64_t *triples;            // {src,dst,len} * nseg
    const uint32_t *first;              // nseg + 1 entries, first[nseg] == nchunk
    const uint32_t *group;              // GroupCount(nchunk, groupShift) + 1 entries
    uint32_t nseg;
    uint32_t nchunk;
    uint32_t groupShift;
    uint32_t units;
    ChunkPattern pattern;
};

}  // namespace mf

#endif  // MF_XCOPY_PLAN_H
