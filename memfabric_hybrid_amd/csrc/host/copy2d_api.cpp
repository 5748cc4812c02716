// Native C entry point of the batched strided 2-D copy (declared in
// include/mf_hip_dataplane.h).  Rectangles whose addresses, pitches and width
// are all multiples of 16 go to the 2-D kernel; anything else is expanded into
// one segment per row and takes the ordinary batch path.
#include <algorithm>
#include <vector>

#include "../../../include/mf_hip_dataplane_internal.h"
#include "../../../include/mf_xcopy_types.h"
#include "../kernels/copy2d_plan.h"
#include "../rt/mf_rt.h"
#include "mf_log.h"
#include "xcopy_engine.h"

using namespace mf;

#define MF_EXPORT extern "C" __attribute__((visibility("default")))

namespace {

bool Aligned16(const mf_copy2d_desc &d)
{
    return RectFitsPlan(d.src, d.dst, d.width, d.height, d.spitch, d.dpitch);
}

// Rows of whole cache lines.
bool OnLines(const mf_copy2d_desc &d)
{
    return ((d.src | d.dst | d.width | d.spitch | d.dpitch) & (kWindowAlignBytes - 1)) == 0;
}

// Two rectangles that are one entry of a RectChunkPlan.
bool RectsPair(const mf_copy2d_desc &a, const mf_copy2d_desc &b)
{
    return RectsSideBySide(a.dst, b.dst, a.width, b.width, a.height, b.height, a.dpitch, b.dpitch) && a.spitch == b.spitch &&
           RectPayloadChunks(2 * (a.width / 16), a.height, 1) != 0;
}

struct RectRun {
    uint32_t rects = 0;            // of the list, from its front
    uint32_t entries = 0;
    uint64_t bytes = 0;
    uint64_t looseBytes = 0;       // of what does not hold a schedule: see RectHolds
    uint64_t shortBytes = 0;       // of that, of what does in short launches
    uint64_t linesBytes = 0;       // of rows of whole cache lines that lie against one another in the destination
    uint64_t againstBytes = 0;     // of other pairs whose rows do
};

// Whether a rectangle, or a pair with rows of `row` bytes, holds a schedule: where the destination's rows lie against one another (a pair), or begin and end on
// 64 bytes, and where lines that are only touched in part are few.  600 MB, us, in windows cut for 6.8 TB/s / in 4 KiB chunks without: pairs of 2736 bytes 182.7 /
// 194.1, 16 bytes between their rows 235 / 212, of 896 and 16 246 / 218, of 896 and 896 184 / 195; single ones of 896, 5120, 4736 bytes read from
// rows 16 bytes longer 184 / 194, 185 / 191, 185 / 191, of 480, 2736 and 20 000 185 / 198, 199 / 194, 186 / 195 but at 900 MB 345 / 309, 336 / 304, 334 / 305; of 64
// bytes 64 apart 308 / 264, of 192 read from rows of 256 281 / 243.  Pairs hold it in short launches whatever their rows: 40 MB of 2736 and 16 16.2 / 18.4 as whole rows.
enum class Holds { kAlways, kShort, kNever };
Holds RectHolds(const mf_copy2d_desc &d, bool pair)
{
    const uint64_t row = pair ? 2 * d.width : d.width;
    const bool against = d.dpitch == row;
    const bool on64 = ((d.dst | d.dpitch | row) & 63) == 0;
    const bool dstLines = ((d.dst | d.dpitch | row) & (kWindowAlignBytes - 1)) == 0;
    const bool srcLines = ((d.src | d.spitch | d.width) & (kWindowAlignBytes - 1)) == 0;
    const uint64_t dstPart = against || dstLines ? 0 : std::min(d.dpitch - row, kWindowAlignBytes);
    const uint64_t srcPart = d.spitch == d.width || srcLines ? 0 : std::min(d.spitch - d.width, kWindowAlignBytes);
    if ((on64 || (pair && against)) && dstPart * 5 <= row && srcPart * 10 <= d.width) {
        return Holds::kAlways;
    }
    return pair && dstPart * 3 <= row && srcPart * 3 <= d.width ? Holds::kShort : Holds::kNever;
}

// As many rectangles as the entries of a plan hold, or as make `target` bytes; none of 2^32 units.
RectRun FillRectChunks(const mf_copy2d_desc *rects, size_t n, uint64_t target, RectChunkPlan &plan)
{
    RectRun run;
    while (run.rects < n && run.entries < kRectInline && run.bytes < target) {
        const mf_copy2d_desc &d = rects[run.rects];
        const bool pair = run.rects + 1 < n && RectsPair(d, rects[run.rects + 1]);
        const uint32_t half = static_cast<uint32_t>(d.width / 16);
        const uint64_t row = pair ? 2ull * half : half;
        if (RectPayloadChunks(row, d.height, 1) == 0) {
            break;
        }
        const uint32_t e = run.entries++;
        plan.src[e] = d.src;
        plan.other[e] = pair ? rects[run.rects + 1].src : d.src;
        plan.dst[e] = d.dst;
        plan.spitchUnits[e] = static_cast<uint32_t>(d.spitch / 16);
        plan.dpitchUnits[e] = static_cast<uint32_t>(d.dpitch / 16);
        plan.halfUnits[e] = half;
        plan.rowUnits[e] = static_cast<uint32_t>(row);
        plan.height[e] = static_cast<uint32_t>(d.height);
        plan.magic[e] = RectMagic(plan.rowUnits[e]);
        run.rects += pair ? 2 : 1;
        run.bytes += row * 16 * d.height;
        const Holds holds = RectHolds(d, pair);
        run.looseBytes += holds == Holds::kAlways ? 0 : row * 16 * d.height;
        run.shortBytes += holds == Holds::kShort ? row * 16 * d.height : 0;
        const bool against = d.dpitch == row * 16;
        const bool lines = against && OnLines(d) && (!pair || OnLines(rects[run.rects - 1]));
        run.linesBytes += lines ? row * 16 * d.height : 0;
        run.againstBytes += !lines && pair && against ? row * 16 * d.height : 0;
    }
    return run;
}

// Whether the launch goes in windows.
bool RectsHold(const RectRun &run)
{
    return run.looseBytes - (run.bytes < kRectShortBytes ? run.shortBytes : 0) <= run.bytes / 4;
}

// Rows of whole cache lines that lie against one another in the destination hold more than segments at any place, whose rate the tuning is, and other pairs whose
// rows do a little more.  Rectangles of a reshard cut for
// 6.8 / 6.9 / 7.0 / 7.1 TB/s, us, the same to 1 % in three processes: on lines 161 MB 51.8 / 51.7 / 50.8 / 50.7, 419 MB 133 / 131 / 130.4 / 128.6, 969 MB 305 / 302 / 299 / 315,
// 4.5 GB 1405 / 1390 / 1369 / 1353; not on lines 248 MB 78.7 / 77.5 / 77.1 / 80.8, 344 MB 108.2 / 108.1 / 111.7 / 120.7, 363 MB 113.7 / 112.7 / 114.3 / 122, 963 MB
// 300 / 297 / 292 / 290.  With room between their rows they fall apart above the tuning's: 600 MB of single ones of 896, 4736 and 5120 bytes, as much apart, 186.5 /
// 186.3 / 186.7 at 6.8, 209.5 / 199.6 / 212.8 at 7.0, of pairs of 256 and of 128 bytes, as much apart, 189.5 / 190.3 and 222 / 208.
// Where no higher rate than windowMBps is in force (this GPU did not hold it, or a caller has set one for all), windowMBps it is.
uint32_t RectRate(const RectRun &run, const XcopyTuning &tuning)
{
    if (tuning.windowAlignedMBps <= tuning.windowMBps) {
        return tuning.windowMBps;
    }
    if (run.linesBytes == run.bytes) {
        return std::min(tuning.windowMBps / 34 * 35, tuning.windowAlignedMBps);
    }
    return run.linesBytes + run.againstBytes >= run.bytes / 4 * 3 ? tuning.windowMBps / 68 * 69 : tuning.windowMBps;
}

// The chunk prefix; false for a launch of 2^32 chunks.
bool CountRectChunks(const RectRun &run, uint32_t units, RectChunkPlan &plan)
{
    uint64_t chunks = 0;
    for (uint32_t i = 0; i < kRectInline; ++i) {
        plan.first[i] = i < run.entries ? static_cast<uint32_t>(chunks) : 0xFFFFFFFFu;
        chunks += i < run.entries ? RectPayloadChunks(plan.rowUnits[i], plan.height[i], units) : 0;
        if (chunks >= 0xFFFFFFFFull) {
            return false;
        }
    }
    plan.nchunk = static_cast<uint32_t>(chunks);
    return true;
}

// The first rectangles of the list in groups of whole rows, one launch; `taken` of them.
int LaunchRectRows(const mf_copy2d_desc *rects, size_t n, uint32_t gridCap, void *stream, uint32_t &taken)
{
    RectPlan plan;
    uint64_t run = 0;
    uint32_t used = 0;
    while (used < n && used < kRectInline) {
        const mf_copy2d_desc &d = rects[used];
        const uint32_t rows = RectRowsPerChunk(d.width);
        const uint64_t chunks = (d.height + rows - 1) / rows;
        if (used != 0 && run + chunks >= 0xFFFFFFFFull) {
            break;
        }
        plan.src[used] = d.src;
        plan.dst[used] = d.dst;
        plan.spitchUnits[used] = static_cast<uint32_t>(d.spitch / 16);
        plan.dpitchUnits[used] = static_cast<uint32_t>(d.dpitch / 16);
        plan.widthUnits[used] = static_cast<uint32_t>(d.width / 16);
        plan.height[used] = static_cast<uint32_t>(d.height);
        plan.rowsPerChunk[used] = rows;
        plan.magic[used] = RectMagic(plan.widthUnits[used]);
        plan.first[used] = static_cast<uint32_t>(run);
        plan.mate[used] = 0;
        if (used > 0 && plan.mate[used - 1] == 0) {
            const mf_copy2d_desc &a = rects[used - 1];
            if (RectsSideBySide(a.dst, d.dst, a.width, d.width, a.height, d.height, a.dpitch, d.dpitch)) {
                plan.mate[used - 1] = 1;
                plan.mate[used] = 2;
            }
        }
        run += chunks;
        ++used;
    }
    for (uint32_t i = used; i < kRectInline; ++i) {
        plan.src[i] = plan.dst[i] = 0;
        plan.spitchUnits[i] = plan.dpitchUnits[i] = plan.widthUnits[i] = plan.height[i] = 0;
        plan.rowsPerChunk[i] = 1;
        plan.magic[i] = 0;
        plan.first[i] = 0xFFFFFFFFu;
        plan.mate[i] = 0;
    }
    taken = used;
    plan.nchunk = static_cast<uint32_t>(run);
    return mfk_copy2d(&plan, static_cast<uint32_t>(gridCap == 0 || run < gridCap ? run : gridCap), stream);
}

}  // namespace

MF_EXPORT void mf_copy2d_describe(uint64_t width, uint32_t *rowsPerChunk, uint32_t *magic)
{
    *rowsPerChunk = RectRowsPerChunk(width);
    *magic = RectMagic(static_cast<uint32_t>(width / 16));
}

MF_EXPORT uint32_t mf_copy2d_rowcol_mismatches(uint32_t widthUnits, uint32_t rowsPerChunk, uint32_t magic, uint32_t unitsInChunk)
{
    uint32_t bad = 0;
    for (uint32_t u = 0; u < unitsInChunk; ++u) {
        uint32_t row = 0;
        uint32_t col = 0;
        RectRowCol(u, widthUnits, rowsPerChunk, magic, row, col);
        bad += (row != u / widthUnits || col != u % widthUnits) ? 1u : 0u;
    }
    return bad;
}

MF_EXPORT int32_t mf_xcopy_2d_batch(const mf_copy2d_desc *descs, uint32_t n, int32_t route, void *stream)
{
    if ((n != 0 && descs == nullptr) || route < 0 || route > MF_ROUTE_FROM_HOST) {
        MF_FAIL(BM_INVALID_PARAM, "mf_xcopy_2d_batch: null descriptors or unknown route");
    }
    XcopyEngine &engine = XcopyEngine::Instance();
    if (!engine.Started()) {
        MF_FAIL(BM_NOT_INITIALIZED, "GPU data plane is not running; call hybm_init first");
    }
    if (mfrt_bind_thread() != 0) {
        MF_FAIL(BM_ERROR, "cannot make the GPU current on this thread");
    }
    if (stream == nullptr) {
        stream = engine.ThreadStream();
    }
    engine.NoteQueued(stream, ~0ull);   // a wait behind these kernels sleeps on the stream
    for (uint32_t i = 0; i < n; ++i) {
        if (descs[i].width > descs[i].spitch && descs[i].height > 1) {
            MF_FAIL(BM_INVALID_PARAM, "rectangle " << i << ": width exceeds the source pitch");
        }
        if (descs[i].width > descs[i].dpitch && descs[i].height > 1) {
            MF_FAIL(BM_INVALID_PARAM, "rectangle " << i << ": width exceeds the destination pitch");
        }
    }
    std::vector<mf_copy2d_desc> rects;
    std::vector<uint64_t> rs;
    std::vector<uint64_t> rd;
    std::vector<uint64_t> rl;
    rects.reserve(n);
    uint64_t total = 0;
    for (uint32_t i = 0; i < n; ++i) {
        const mf_copy2d_desc &d = descs[i];
        if (d.width == 0 || d.height == 0) {
            continue;
        }
        if (Aligned16(d)) {
            rects.push_back(d);
            total += d.width * d.height;
            continue;
        }
        for (uint64_t r = 0; r < d.height; ++r) {
            rs.push_back(d.src + r * d.spitch);
            rd.push_back(d.dst + r * d.dpitch);
            rl.push_back(d.width);
        }
    }
    const uint32_t cu = mfrt_cu_count() == 0 ? 256 : mfrt_cu_count();
    const uint32_t gridCap = cu * engine.Tuning().wgPerCu;   // 0: one workgroup per row group
    // A windowed launch loses its schedule the likelier the longer it runs, so long lists go in even parts.
    const uint64_t parts = (total + kRectLaunchBytes / 2) / kRectLaunchBytes;
    const uint64_t target = parts < 2 ? ~0ull : (total + parts - 1) / parts;
    RectChunkPlan plan{};
    for (size_t at = 0; at < rects.size();) {
        int err = 0;
        uint32_t taken = 0;
        const RectRun run = route == MFRT_ROUTE_HBM && gridCap == 0 && total >= kRectChunksMinBytes
                                ? FillRectChunks(&rects[at], rects.size() - at, target, plan)
                                : RectRun{};
        const bool windowed = RectsHold(run) && engine.WindowsApply(run.bytes, route, kRectChunksMinBytes);
        if (run.bytes >= (windowed ? kRectChunksMinBytes : kRectPlainChunksMinBytes) &&
            CountRectChunks(run, windowed ? kRectWindowUnits : 64 * kRectChunkDepth, plan)) {
            taken = run.rects;
            err = mfk_copy2d_chunks(&plan, windowed ? RectRate(run, engine.Tuning()) : 0, stream);
        } else {
            err = LaunchRectRows(&rects[at], rects.size() - at, gridCap, stream, taken);
        }
        if (err != 0) {
            MF_FAIL(BM_ERROR, "2-D copy launch failed: " << mfrt_error_string(err));
        }
        at += taken;
    }
    if (!rs.empty()) {
        return engine.Submit(rs.data(), rd.data(), rl.data(), static_cast<uint32_t>(rs.size()), route, stream, nullptr, 0);
    }
    return BM_OK;
}
