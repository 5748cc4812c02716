// Host planner and submission engine of the xcopy kernels (plain C++, no HIP
// types).  It turns a caller's segment list into one fused kernel launch on a
// stream: the job HostDataOpSDMA::BatchCopyG2G / BatchCopyExtend do with one
// SDMA descriptor per segment or a 32-block plugin launch
// (src/hybm/csrc/data_operation/host/hybm_data_op_sdma.cpp:504-595).
#ifndef MF_XCOPY_ENGINE_H
#define MF_XCOPY_ENGINE_H

#include <stdint.h>

#include <atomic>
#include <vector>

#include "../kernels/xcopy_plan.h"

namespace mf {

// Segment list after normalisation: empty segments dropped, neighbours that
// continue each other on both sides merged (the reference merges the same
// way before building descriptors, hybm_data_op_sdma.cpp:571-574).
struct SegList {
    std::vector<uint64_t> src;
    std::vector<uint64_t> dst;
    std::vector<uint64_t> len;
    uint64_t totalBytes = 0;
    void Clear()
    {
        src.clear();
        dst.clear();
        len.clear();
        totalBytes = 0;
    }
    uint32_t Size() const
    {
        return static_cast<uint32_t>(src.size());
    }
};

// pieceLimit: segments longer than this are cut into pieces of at most that
// many bytes (the inline plan stores 32-bit lengths); 0 = never cut.
void NormalizeSegments(const uint64_t *src, const uint64_t *dst, const uint64_t *len, uint32_t n, uint64_t pieceLimit,
                       SegList &out);

constexpr int32_t kHoldPinnedDeepExtraNanos = kHoldLookupDeepExtraNanos - kHoldLookupExtraNanos;
// What the shape of a launch of pieces is chosen by, from one pass over a batch.
struct BatchStats {
    uint64_t total = 0;
    uint64_t longest = 0;
    uint64_t addressBits = 0;       // low bits that any address has set
    uint64_t lengthBits = 0;        // and any length
    uint64_t deepPieces = 0;        // of 16 KiB, at the most
};
BatchStats StatsOf(const uint64_t *src, const uint64_t *dst, const uint64_t *len, uint32_t n);
// Whether most of the first segments of a batch lie one behind the other, in source or destination, with at most `gap` bytes in between.
bool InOrder(const uint64_t *at, const uint64_t *len, uint32_t n, uint64_t gap = 0);

// A batch of this much and more is cut into pieces of 8 and 16 KiB.  Shorter ones keep 4 KiB, which more CUs share: 150 pages of 8 KiB
// 2.8 us, 4.0 in waves of 16 KiB; 200 pages of 32 KiB 4.4 / 4.6.  From there on the longer pieces are as fast and a quarter of the
// descriptors for the host to write, which had bounded those batches: a call of 500 pages of 32 KiB took 10.6 us, the launch 6.6 on
// 4 KiB and 7.0 on 16; uneven segments gain on the GPU too (1000 of 5000 bytes 5.9 / 5.2, 500 of 40 000 9.5 / 8.9).
constexpr uint64_t kPieceLongMinBytes = 4ull << 20;
// Pieces in windows: below, too few periods pay for the halves of the first and the last one in which the chip only reads or only
// writes (72 MB of K and V blocks 28.7 us without windows and 28.3 with them, 82 MB of pages 29.6 / 29.0, 90 MB of blocks 35.7 / 32.8).
constexpr uint64_t kPieceWindowMinBytes = 80ull << 20;
constexpr uint64_t kDonePiecesBytes = 4ull << 20; // blocking batches up to here report their own end,
constexpr uint32_t kDonePiecesSegments = 2048;    // and up to so many segments: every piece counts itself done
constexpr uint64_t kReportBytes = 12000000;       // launches on callers' streams up to here,
constexpr uint64_t kReportSegmentBytes = 16000;    // and this much more per segment, report that their list has been read
constexpr uint64_t kSliceMinNanos = 6000;         // planning that a blocking batch is not sliced for
constexpr uint64_t kPieceListMin = 1ull << 18;     // pieces that any batch may be cut into, 4 MiB of descriptors

struct XcopyTuning {
    uint32_t unitsOverride = 0;  // 16-byte units per chunk, 0 = choose from batch size
    uint32_t wgPerCu = 0;        // HBM routes: grid cap in workgroups per CU, 0 = one workgroup per chunk
    uint32_t wgPerCuLink = 0;    // routes bound by the host link: workgroups per CU; 0: kLinkGroups for the whole chip
    uint32_t minUnits = kXcopyThreads;   // 4 KiB: the chunk of HBM routes
    int32_t holdNanos = -1;      // stores held back in inline launches: -1 = HoldNanosFor's rule (+ holdDeltaNanos), 0 = never, else that long
    int32_t holdDeltaNanos = 0;  // added to the rule's wait: what the calibration at start found best on this GPU
    bool holdCalibratedOff = false;   // the calibration found no gain in holding stores on this GPU
    uint32_t unorderedStreams = 0;   // unordered batches are launched by this many submit threads of the library's, a stream each (0, 1: by the caller on its own stream)
    bool holdOnSideStreams = false;  // launches of the submit threads overlap on purpose: their stores are not held
    bool deepHold = true;        // batches of 24 to 64 MiB hold the stores of 16 KiB per wave
    int32_t holdPinnedExtraNanos = kHoldLookupExtraNanos;   // added to the rule for launches of more than kInlineSegs segments
    bool stageUnordered = true;  // the upload of a ragged table's descriptors is launched without a barrier
    uint32_t deviceTableWgPerCu = 0;   // grid of a device-resident table in workgroups per CU, 0 = four per segment between 16 and 1024 per CU, or 192 (SubmitDeviceTable)
    uint32_t windowMBps = 6800000;   // long HBM copies alternate between read and write windows cut for this rate; 0 = never
    // The same for launches whose sources and destinations agree modulo 16, which hold more; 0 = the rate above.  300 MB, us, at 6.8 / 7.3
    // TB/s: with the source 64 bytes off a cache line 91.8 / 86.0, the destination 91.8 / 86.2; 100 segments of 3 MB, 48 bytes off 92.6 / 86.8,
    // 92.6 / 86.9.
    uint32_t windowAlignedMBps = 7300000;
    // And for those of them that all start at multiples of kWindowAlignBytes in source and destination and are kWindowLongSegmentBytes and
    // longer on average, which hold more still; 0 = the rate above.  The highest that copies kept to in each of ten processes; us, the
    // mean back to back at 7.3 / 7.375 / 7.45 TB/s: one segment of 512 MiB 151.9 / 151.9 / 151.2, of 1 GiB 302 / 300 / 301, in one process of
    // four 303 / 300 / 307; waited for one by one, 512 MiB 165 / 165 / 163 to 176, 1 GiB 317 / 314 / 312.  At 7.5 one in some twenty-five saw
    // none of six keep to it.
    uint32_t windowLongMBps = 7375000;
};

// (A batch of up to 128 segments between HBM addresses is copied in windows from where held stores end, 64 MiB, 112 for one segment.  Back to back, 32
// segments on lines, windows of 4096 waves against none: 66 MiB 6.37 against 5.71 TB/s, 80 MiB 6.57 against 5.76, 130 MiB 6.94 against 6.14, 256 MiB 7.14
// against 6.37, 600 MiB 7.20 against 6.31.)
// Rectangles in chunks of their payload: in windows, and without (several threads, rows between cache lines), where whole rows are as
// fast up to 40 MB (Copy2dChunkKernel has the figures).
constexpr uint64_t kRectChunksMinBytes = 32ull << 20;
constexpr uint64_t kRectPlainChunksMinBytes = 48ull << 20;
constexpr uint64_t kRectShortBytes = 64ull << 20;             // launches below keep their schedule where longer ones of such rows lose it
constexpr uint64_t kRectLaunchBytes = 640ull << 20;
constexpr uint64_t kWindowPieceBytes = 512ull << 20;          // launches into which long segments are cut
constexpr uint64_t kWindowLongSegmentBytes = 64ull << 20;     // launches whose segments average this much go out in pieces of kWindowPieceBytes and more
constexpr uint64_t kWindowAlignBytes = 128;                   // a cache line: segments that start on one are read and written in whole lines by every wave
constexpr uint64_t kWindowSliceMinSegmentBytes = 4ull << 20;   // tables of segments this long on average are cut into windowed launches
constexpr uint64_t kWindowSliceMinAlignedSegmentBytes = 1ull << 20;   // the same for segments on cache lines: kInlineSegs of them are 128 MiB

// What Start() measured on the GPU it runs on and chose from it (XcopyEngine::Calibrate).
struct XcopyCalibration {
    bool ran = false;               // false: skipped (MF_HIP_CALIBRATE=0), failed, or not run yet: the fitted defaults apply
    bool holdEnabled = true;        // the held stores beat the launch that stores at once by kCalibrateMinGain
    int32_t holdDeltaNanos = 0;     // added to every wait HoldNanosFor gives
    uint32_t windowMBps = 0;        // rate the read and write windows are cut for; 0: the form lost against the plain kernel
    uint32_t windowAlignedMBps = 0;    // rate for launches of segments on cache-line boundaries
    uint32_t windowLongMBps = 0;       // rate for launches of long segments on cache-line boundaries; both the higher ones where a long copy held the highest, else the rate above
    float batchMicros[4] = {};      // 2196-chunk batch: not held, rule - step, rule, rule + step
    float copyMicros[4] = {};       // 512 MiB copy: no windows, default rate, reduced rate, the rate of long segments on cache lines
};
constexpr int32_t kCalibrateHoldStepNanos = 200;
constexpr float kCalibrateMinGain = 0.03f;          // held stores that do not gain this much over the plain launch are switched off
constexpr float kCalibrateMinWindowGain = 0.005f;   // windows stay unless they lose: on the 512 MiB that is measured they gain least (2 to 5 %, 8 % on 1 GiB)
constexpr uint32_t kCalibrateSlowerWindowPercent = 94;   // the second window rate tried, in percent of the default
// The choice, from the measured times alone (microseconds; a time of 0 means "not measured" and leaves the default).
void ChooseCalibration(const float *batchMicros, const float *copyMicros, uint32_t defaultWindowMBps, uint32_t defaultAlignedMBps, uint32_t defaultLongMBps,
                       XcopyCalibration &out);

uint32_t ChooseUnits(uint64_t totalBytes, uint32_t cuCount, int route, const XcopyTuning &tuning);

// Returns false when the list does not fit the inline form.
bool BuildInlinePlan(const SegList &segs, uint32_t units, InlinePlan &plan);

// The same result as NormalizeSegments + BuildInlinePlan in one pass over the caller's arrays;
// false when the batch does not fit the inline form (more than kInlineSegs merged segments, or
// one of 4 GiB and more, which the general path cuts into pieces).
bool BuildInlineDirect(const uint64_t *src, const uint64_t *dst, const uint64_t *len, uint32_t n, uint32_t units,
                       InlinePlan &plan);

// triples: 3 * segs.Size() words, first: segs.Size() + 1 words.  Returns total chunks.
uint64_t BuildTablePlan(const SegList &segs, uint32_t units, uint64_t *triples, uint32_t *first);

// The same result as NormalizeSegments (no piece limit) + BuildTablePlan in one pass over the
// caller's arrays.  triples: room for 3 * n words, first: room for n + 1; count = segments written.
// pattern (optional) receives the shortest period (up to kMaxPeriod) with which the chunk counts
// of the segments repeat, period 0 when there is none.
uint64_t BuildTableDirect(const uint64_t *src, const uint64_t *dst, const uint64_t *len, uint32_t n, uint32_t units,
                          uint64_t *triples, uint32_t *first, uint32_t &count, ChunkPattern *pattern = nullptr);

class XcopyEngine {
public:
    static XcopyEngine &Instance();

    int Start(int device);          // BM_* code
    void Stop();
    bool Started() const;

    XcopyTuning &Tuning()
    {
        return tuning_;
    }
    const XcopyCalibration &Calibration() const
    {
        return calibration_;
    }
    // Measures, on the calling thread's stream, the 2196-chunk batch with its stores not held and held for the rule's wait
    // and kCalibrateHoldStepNanos either side of it, and a 512 MiB copy without windows and at two window rates; keeps
    // the best wait (or none) and the best rate (or none) for the process.  About 15 ms and 1 GiB of HBM for its duration.
    // Start() runs it unless the environment says MF_HIP_CALIBRATE=0.
    int Calibrate();

    // Whether an ordered launch that moves `bytes` on `route` takes the form with read and write windows.
    bool WindowsApply(uint64_t bytes, int route, uint64_t minBytes) const;
    // Hardware queue (numbered in order of appearance) of each of the streams made at Start(), in the order they are handed out; returns their number.
    uint32_t StreamQueues(uint32_t *queues, uint32_t capacity) const;
    // No second thread holds a stream of the library: kernels that pace themselves for the whole chip may be used.
    bool SingleSubmitter() const;

    // The calling thread's own stream (created on first use).  Unordered batches that were handed to the submit
    // threads are joined first: work queued on the returned stream afterwards waits for them.
    void *ThreadStream();
    static constexpr uint32_t kFanStreams = 8;   // most submit threads for unordered batches (9 MB batches: 2 / 3 / 4 / 6 / 8 threads 4.3 / 3.8 / 3.6 / 3.8 / 3.6-4.0 us per batch)
    static constexpr uint32_t kDeckStreams = 8;   // streams made at Start() and dealt out so that consecutive takers sit on different hardware queues
    static constexpr uint64_t kFanMaxBytes = 64ull << 20;   // larger batches gain nothing from a second queue
    // Pinned, device-mapped staging memory of the calling thread, at least `bytes` long; it lives
    // until Stop().  NULL when it cannot be allocated.  *fresh: whether this call has allocated it.
    void *ThreadBounce(uint64_t bytes, bool *fresh = nullptr);
    // Wait for everything this thread enqueued on its own stream.
    int DrainThread();
    // Wait for everything queued on `stream` so far: what a blocking copy does after its launch.
    // Work of known size (`bytes` moved, 0 = unknown) is awaited by polling a word in pinned memory that a one-lane
    // launch behind the copy stores, for at most kSpinMicros more than the route needs for it; anything else,
    // and a poll that runs out of time, waits on the stream.
    static constexpr uint64_t kSpinBytes = 256ull << 20;
    static constexpr uint32_t kSpinMicros = 200;
    int WaitStream(void *stream, uint64_t bytes, int route = 0 /* MFRT_ROUTE_HBM */);
    // Submit() and WaitStream() of a blocking copy.
    int SubmitAndWait(const uint64_t *src, const uint64_t *dst, const uint64_t *len, uint32_t n, int route, void *stream);
    // The two halves for a thread that has several copies on their way on one stream: `ticket` says what WaitTicket() waits
    // for, everything queued on `stream` up to that copy.
    int SubmitTicket(const uint64_t *src, const uint64_t *dst, const uint64_t *len, uint32_t n, int route, void *stream, uint32_t &ticket);
    int WaitTicket(uint32_t ticket, void *stream);
    // Work that another part of the library has queued on `stream`: if it is the calling thread's own stream, the next
    // DrainThread() takes `bytes` into account when it chooses between polling and sleeping (~0: sleep).
    void NoteQueued(void *stream, uint64_t bytes);
    // The same for launches that move data and have been waited for, with everything queued on `stream` before them.
    void NoteDone(void *stream, uint32_t launches);

    // Enqueue one batch.  Addresses must be device-accessible.  stream may be
    // NULL (thread stream).  mask/maskValue: plugin completion word or NULL.
    // Returns 0 or a negative BM_* code; never waits for the copy itself.
    // unordered: the caller vouches that the batch is independent of everything still in flight on
    // `stream`; a batch that fits the kernel-argument form is then launched without a barrier.
    int Submit(const uint64_t *src, const uint64_t *dst, const uint64_t *len, uint32_t n, int route, void *stream,
               void *mask, uint32_t maskValue, bool unordered = false);

    // Same for a triple table that lives in device memory the host cannot read.
    int SubmitDeviceTable(const void *triples, uint32_t n, int route, void *stream, void *mask, uint32_t maskValue);

    // The same, with the list of long segments in the statically allocated device scratch: allocates nothing
    // (no stream either: `stream` is used as given, NULL being the null stream), at most
    // MFK_STATIC_TABLE_SEGMENTS segments, calls on one GPU must not overlap.
    int SubmitDeviceTableStatic(const void *triples, uint32_t n, int route, void *stream);

    // Returns once every batch handed to the submit threads so far has been launched (a device wait then covers it).
    void QuiesceSubmitters();

    uint64_t LaunchCount() const;

private:
    XcopyEngine() = default;

    uint32_t HoldFor(const InlinePlan &plan, uint32_t grid, int route, bool unordered) const;
    uint32_t HoldForPieces(const BatchStats &stats, uint32_t n, uint32_t count, uint32_t units, bool unordered) const;
    uint32_t HeldLaunches(const BatchStats &stats, const uint64_t *src, const uint64_t *dst, const uint64_t *len, uint32_t n, bool unordered) const;
    int SubmitHeld(const uint64_t *src, const uint64_t *dst, const uint64_t *len, uint32_t n, const BatchStats &stats, uint32_t parts, void *stream,
                   void *mask, uint32_t maskValue);
    uint32_t PieceUnits(const BatchStats &stats, uint32_t n, bool unordered) const;
    // Rate of the windows a list of `count` pieces of `units` units is copied in, 0: in none.  reading: 64ths of a period that are its read
    // part, unchanged for half of it.
    uint32_t PieceWindowRate(const BatchStats &stats, const uint64_t *src, const uint64_t *dst, const uint64_t *len, uint32_t n, uint32_t count,
                             uint32_t units, bool unordered, uint32_t &reading) const;
    // How a launch of a device table paces itself: the waits of its waves and the rate of its windows.
    void TablePaceFor(uint32_t &holdNanos, uint32_t &holdMoreNanos, uint32_t &windowMBps) const;
    // Whether a batch of `bytes` in n segments is planned in chunks of kDeepUnits units, to hold the stores of 16 KiB per wave.
    bool DeepHoldApplies(uint64_t bytes, uint32_t n, int route, bool unordered) const;
    // A launch that stores the thread's word itself, where that is the faster form: kNotLaunched where it is not.
    static constexpr int kNotLaunched = 1;
    int LaunchDone(const uint64_t *src, const uint64_t *dst, const uint64_t *len, uint32_t n, uint64_t bytes, int route, void *stream,
                   uint32_t &ticket);
    int LaunchPiecesDone(const uint64_t *src, const uint64_t *dst, const uint64_t *len, uint32_t n, uint64_t bytes, int route, void *stream,
                         uint32_t &ticket);
    int SubmitPieces(const uint64_t *src, const uint64_t *dst, const uint64_t *len, uint32_t n, const BatchStats &stats, uint32_t units,
                     void *stream, void *mask, uint32_t maskValue, bool unordered);
    int SubmitInSlices(const uint64_t *src, const uint64_t *dst, const uint64_t *len, uint32_t n, uint64_t bytes, int route, void *stream);
    int SubmitRecorded(const uint64_t *src, const uint64_t *dst, const uint64_t *len, uint32_t n, int route, void *stream, void *mask,
                       uint32_t maskValue);
    int SubmitInPieces(const uint64_t *src, const uint64_t *dst, const uint64_t *len, uint32_t n, uint64_t total, int route,
                       void *stream, void *mask, uint32_t maskValue);
    int SubmitOne(const uint64_t *src, const uint64_t *dst, const uint64_t *len, uint32_t n, int route, void *stream,
                  void *mask, uint32_t maskValue, bool unordered, bool maySlice);

    XcopyTuning tuning_;
    XcopyCalibration calibration_;
    bool windowRateCalibrated_ = false;  // tuning_.windowMBps holds what Calibrate() chose, not a caller's setting
    bool windowsAvailable_ = false;      // set by Start(): the device's constant-rate clock is known
    std::atomic<bool> started_{false};   // read by every calling thread, flipped by Start / Stop
};

}  // namespace mf

#endif  // MF_XCOPY_ENGINE_H
