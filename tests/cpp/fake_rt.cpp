// TEST INFRASTRUCTURE ONLY.  A CPU stand-in for the thin runtime layer (csrc/rt/mf_rt.h) so that the
// host stack above it - planner, staging ring, operator fallback, entity and C API - can be
// exercised without a GPU, the way the reference's unit tests run against stub vendor libraries
// (test/ut/mock/acl_stub.cpp of the reference).  "Device" memory is host memory, a launch executes
// its plan at once with the SAME chunk geometry the kernels use (csrc/kernels/xcopy_plan.h), streams
// and events are tokens.  Never linked into the product libraries.
#include <atomic>
#include <cstdint>
#include <cstdio>
#include <cstdlib>
#include <vector>
#include <cstring>
#include <chrono>
#include <map>
#include <mutex>
#include <thread>

#include <sys/mman.h>

#include "../../memfabric_hybrid_amd/csrc/kernels/copy2d_plan.h"
#include "../../memfabric_hybrid_amd/csrc/kernels/staging.h"
#include "../../memfabric_hybrid_amd/csrc/kernels/xcopy_plan.h"
#include "../../memfabric_hybrid_amd/csrc/rt/mf_rt.h"

namespace {
std::mutex g_lock;
std::map<uint64_t, std::pair<uint64_t, int>> g_allocs;  // base -> (size, kind)
int g_device = -1;
std::atomic<uint64_t> g_launches{0};   // launches may come from the engine's submit threads
std::atomic<uint32_t> g_lastHold{0};   // holdNanos of the latest inline launch
uint32_t g_lastReading = 0;  // read part of the latest windowed list
uint32_t g_lastWindow = 0;   // rate of the latest windowed launch, cleared by fake_rt_last_window()
uint32_t g_lastTableWindow = 0;   // rate handed to the latest launch of a long device table, and its grid
uint32_t g_lastTableGrid = 0;
std::atomic<uint64_t> g_chunksRun{0};
bool g_skipCopies = false;       // launches count and check their plans but move nothing (tables of segments no test can back with memory)
uint32_t g_lastTableShift = 0;   // group shift of the latest table launch that used a group map, 0 under a pattern
uint64_t g_groupMapErrors = 0;
uint32_t g_lastPieceWait = 0;    // what the waves of the latest launch of pieces wait
uint32_t g_mostPieces = 0;       // the most pieces of one launch, and the least its waves wait, since fake_rt_piece_launches()
uint32_t g_leastPieceWait = ~0u;
uint32_t g_lastTableHold = 0;    // holdNanos of the latest table launch
std::atomic<uint64_t> g_streamsMade{0};   // streams made since mfrt_init

// The stream that records a graph, and what a graph cannot hold or replay that was done while it did: allocations, events recorded
// on it, launches whose descriptors lie in memory of the host's.
void *g_capturing = nullptr;
uint64_t g_captureErrors = 0;
void NoteRecorded(const void *stream)
{
    g_captureErrors += g_capturing != nullptr && stream == g_capturing ? 1 : 0;
}
const void *g_lastRestList = nullptr;

bool g_failAllocations = false;

// Streamed copies run on a thread of their own; off unless a test asks for them, so that the others see copies in rounds.
uint32_t g_streamChunks = 0;              // chunks after which the launches of a copy leave; 0: it cannot be launched
std::atomic<uint32_t> g_streamsRunning{0};
std::atomic<uint64_t> g_chunksStreamed{0};
uint32_t g_streamLaunchMillis = 0;        // what the call that launches one takes
uint32_t g_streamBusyMillis = 0;          // of other work that is in front of it on its stream
uint32_t g_mostChunksLaunched = 0;        // of one launch
uint32_t g_streamLaunches = ~0u;          // after which they fail
uint64_t g_streamBase = 0;                // what the copy's first launch counts from
std::vector<std::thread> g_streamThreads;
void JoinStreamed()
{
    for (std::thread &thread : g_streamThreads) {
        thread.join();
    }
    g_streamThreads.clear();
}

void *Track(uint64_t bytes, int kind)
{
    NoteRecorded(g_capturing);
    if (g_failAllocations) {
        return nullptr;
    }
    void *p = nullptr;
    if (posix_memalign(&p, 4096, bytes == 0 ? 4096 : bytes) != 0) {
        return nullptr;
    }
    std::lock_guard<std::mutex> guard(g_lock);
    g_allocs[reinterpret_cast<uint64_t>(p)] = {bytes, kind};
    return p;
}

int Untrack(void *p)
{
    std::lock_guard<std::mutex> guard(g_lock);
    auto it = g_allocs.find(reinterpret_cast<uint64_t>(p));
    if (it == g_allocs.end()) {
        return 1;
    }
    g_allocs.erase(it);
    free(p);
    return 0;
}

void RunChunk(uint64_t src, uint64_t dst, uint64_t len, uint64_t k, uint32_t units)
{
    const mf::SegGeom g = mf::SegmentGeometry(dst, len);
    const uint64_t u0 = k * units;
    const uint64_t left = g.body > u0 ? g.body - u0 : 0;
    const uint64_t n = left < units ? left : units;
    std::memmove(reinterpret_cast<void *>(dst + g.head + u0 * 16), reinterpret_cast<void *>(src + g.head + u0 * 16), n * 16);
    if (k == 0) {
        std::memmove(reinterpret_cast<void *>(dst), reinterpret_cast<void *>(src), g.head);
    }
    if (u0 + units >= g.body) {
        const uint64_t off = g.head + g.body * 16;
        std::memmove(reinterpret_cast<void *>(dst + off), reinterpret_cast<void *>(src + off), g.tail);
    }
    ++g_chunksRun;
}
// Descriptor tables stay "in flight" until something the host has waited for covers their launch:
// an event recorded later, or a stream / device wait.  A table that changed in the meantime was
// rewritten while a kernel could still read it.
struct InFlight {
    uint64_t seq;
    const void *table;
    std::vector<uint8_t> snapshot;
};
std::mutex g_flightLock;
std::vector<InFlight> g_inFlight;
uint64_t g_flightSeq = 0;
uint64_t g_violations = 0;

void TrackTable(const void *table, size_t bytes)
{
    std::lock_guard<std::mutex> guard(g_flightLock);
    InFlight f{++g_flightSeq, table, {}};
    f.snapshot.assign(static_cast<const uint8_t *>(table), static_cast<const uint8_t *>(table) + bytes);
    g_inFlight.push_back(std::move(f));
}

void Retire(uint64_t upTo)
{
    std::lock_guard<std::mutex> guard(g_flightLock);
    size_t keep = 0;
    for (size_t i = 0; i < g_inFlight.size(); ++i) {
        InFlight &f = g_inFlight[i];
        if (f.seq <= upTo) {
            if (std::memcmp(f.table, f.snapshot.data(), f.snapshot.size()) != 0) {
                ++g_violations;
            }
        } else {
            if (keep != i) {
                g_inFlight[keep] = std::move(f);
            }
            ++keep;
        }
    }
    g_inFlight.resize(keep);
}

}  // namespace

extern "C" {
// After this call any allocation, free, mapping or launch aborts: the test binary arms it at the
// end of main() to prove that nothing touches the GPU runtime from static destructors.
static bool g_sealed = false;
void fake_rt_seal(void) { g_sealed = true; }
static void Guard(const char *what)
{
    if (g_sealed) {
        std::fprintf(stderr, "runtime call after main(): %s\n", what);
        std::abort();
    }
}
void fake_rt_capture(void *stream) { g_capturing = stream; }
uint64_t fake_rt_capture_errors(void) { return g_captureErrors; }
const void *fake_rt_last_rest_list(void) { return g_lastRestList; }
// Launches that say when they have read their list do so from now on only at fake_rt_release_reports().
static std::mutex g_reportLock;
static bool g_withholdReports = false;
static std::vector<std::pair<uint64_t *, uint64_t>> g_withheldReports;
void fake_rt_withhold_reports(void) { g_withholdReports = true; }
void fake_rt_release_reports(void)
{
    std::lock_guard<std::mutex> guard(g_reportLock);
    g_withholdReports = false;
    Retire(~0ull);
    for (const auto &report : g_withheldReports) {
        __atomic_store_n(report.first, report.second, __ATOMIC_RELEASE);
    }
    g_withheldReports.clear();
}
static std::atomic<int> g_streamState{1};
void fake_rt_stream_state(int state) { g_streamState = state; }
void fake_rt_fail_allocations(int on) { g_failAllocations = on != 0; }
uint64_t fake_rt_launches(void) { return g_launches; }
uint32_t fake_rt_last_hold(void) { return g_lastHold; }
uint32_t fake_rt_last_table_grid(void) { return g_lastTableGrid; }
uint32_t fake_rt_last_table_window(void) { return g_lastTableWindow; }
uint32_t fake_rt_last_reading(void) { return g_lastReading; }
uint32_t fake_rt_last_window(void) { const uint32_t w = g_lastWindow; g_lastWindow = 0; return w; }
// The next n xcopy launches fail with a runtime error code instead of running.
static int g_failLaunches = 0;
void fake_rt_fail_launches(int n) { g_failLaunches = n; }
uint64_t fake_rt_chunks(void) { return g_chunksRun; }
void fake_rt_skip_copies(int on) { g_skipCopies = on != 0; }
uint32_t fake_rt_last_table_shift(void) { return g_lastTableShift; }
uint64_t fake_rt_group_map_errors(void) { return g_groupMapErrors; }
uint32_t fake_rt_last_piece_wait(void) { return g_lastPieceWait; }
void fake_rt_piece_launches(uint32_t *mostPieces, uint32_t *leastWait)
{
    *mostPieces = g_mostPieces;
    *leastWait = g_leastPieceWait;
    g_mostPieces = 0;
    g_leastPieceWait = ~0u;
}
uint32_t fake_rt_last_table_hold(void) { return g_lastTableHold; }

int mfrt_init(int device)
{
    if (device != 0) {
        return 101;
    }
    g_device = 0;
    g_streamsMade = 0;
    return 0;
}
int mfrt_current_device(void) { return 0; }
int mfrt_bind_thread(void) { return g_device >= 0 ? 0 : 3; }
void mfrt_shutdown(void) { g_device = -1; }
int mfrt_is_initialised(void) { return g_device >= 0; }
int mfrt_device_id(void) { return g_device; }
uint32_t mfrt_cu_count(void) { return 256; }
const char *mfrt_error_string(int) { return "fake runtime error"; }
void *mfrt_alloc_device(uint64_t bytes) { return Track(bytes, MFRT_PTR_DEVICE); }
int mfrt_free_device(void *p) { Guard("mfrt_free_device"); Retire(~0ull); return Untrack(p); }   // hipFree waits for the device
void *mfrt_alloc_host(uint64_t bytes) { return Track(bytes, MFRT_PTR_PINNED_HOST); }
int mfrt_free_host(void *p) { Guard("mfrt_free_host"); Retire(~0ull); return Untrack(p); }
// Address windows: reserved as inaccessible pages, so a touch of an unmapped part ends the test
// with a fault just as it would fault the GPU; mapping makes the pages usable.
uint64_t mfrt_window_granularity(void) { return 2u << 20; }
void *mfrt_window_reserve(uint64_t bytes)
{
    void *p = mmap(nullptr, bytes, PROT_NONE, MAP_PRIVATE | MAP_ANONYMOUS | MAP_NORESERVE, -1, 0);
    return p == MAP_FAILED ? nullptr : p;
}
int mfrt_window_last_error(void) { return 0; }
int mfrt_window_release(void *base, uint64_t bytes) { Guard("mfrt_window_release"); return munmap(base, bytes) == 0 ? 0 : 1; }
void *mfrt_window_map(void *addr, uint64_t bytes, void *accessBase, uint64_t accessBytes)
{
    if (static_cast<char *>(accessBase) + accessBytes != static_cast<char *>(addr) + bytes) {
        return nullptr;   // the access run must end with the new piece
    }
    if (mprotect(addr, bytes, PROT_READ | PROT_WRITE) != 0) {
        return nullptr;
    }
    std::lock_guard<std::mutex> guard(g_lock);
    g_allocs[reinterpret_cast<uint64_t>(addr)] = {bytes, MFRT_PTR_DEVICE};
    return addr;
}
int mfrt_window_unmap(void *addr, uint64_t bytes, void *handle)
{ Guard("mfrt_window_unmap");
    if (handle != addr) {
        return 1;
    }
    std::lock_guard<std::mutex> guard(g_lock);
    g_allocs.erase(reinterpret_cast<uint64_t>(addr));
    (void)madvise(addr, bytes, MADV_DONTNEED);
    return mprotect(addr, bytes, PROT_NONE) == 0 ? 0 : 1;
}
int mfrt_pointer_kind(const void *p)
{
    std::lock_guard<std::mutex> guard(g_lock);
    const uint64_t a = reinterpret_cast<uint64_t>(p);
    auto it = g_allocs.upper_bound(a);
    if (it == g_allocs.begin()) {
        return MFRT_PTR_PAGEABLE;
    }
    --it;
    return a < it->first + it->second.first ? it->second.second : MFRT_PTR_PAGEABLE;
}
// A stream remembers the how-manieth stream since mfrt_init it is: the stand-in for "which hardware queue the runtime
// put it on" follows the pattern measured on the GPU (queues A B C C B A D C, then round robin).
static int g_queueAnswers = 0;      // 0: by the pattern, 1: not known
void fake_rt_queue_answers(int mode) { g_queueAnswers = mode; }
void *mfrt_stream_create(void)
{
    uint64_t *token = static_cast<uint64_t *>(malloc(8));
    *token = g_streamsMade.fetch_add(1);
    return token;
}
static uint32_t FakeQueueOf(const void *stream)
{
    static const uint32_t first[8] = {0, 1, 2, 2, 1, 0, 3, 2};
    const uint64_t index = *static_cast<const uint64_t *>(stream);
    return index < 8 ? first[index] : static_cast<uint32_t>(index % 4);
}
int mfrt_streams_share_queue(void *a, void *b)
{
    if (g_queueAnswers == 1) {
        return -1;
    }
    return FakeQueueOf(a) == FakeQueueOf(b) ? 1 : 0;
}
int mfrt_stream_destroy(void *s) { Guard("mfrt_stream_destroy"); free(s); return 0; }
uint64_t fake_rt_violations(void) { return g_violations; }
uint64_t fake_rt_in_flight(void)
{
    std::lock_guard<std::mutex> guard(g_flightLock);
    return g_inFlight.size();
}

extern "C" void fake_rt_count_stream_sync(void);
int mfrt_stream_sync(void *) { Guard("mfrt_stream_sync"); JoinStreamed(); Retire(~0ull); fake_rt_count_stream_sync(); return 0; }
int mfrt_stream_capturing(void *stream) { return g_capturing != nullptr && stream == g_capturing ? 1 : 0; }
int mfrt_stream_done(void *) { return g_streamsRunning.load() != 0 ? 0 : g_streamState.load(); }
int mfrt_device_sync(void) { Guard("mfrt_device_sync"); Retire(~0ull); return 0; }
void *mfrt_event_create(void) { return calloc(1, 8); }
int mfrt_event_destroy(void *e) { Guard("mfrt_event_destroy"); free(e); return 0; }
int mfrt_event_record(void *e, void *stream)
{
    NoteRecorded(stream);
    std::lock_guard<std::mutex> guard(g_flightLock);
    *static_cast<uint64_t *>(e) = g_flightSeq;
    return 0;
}
int mfrt_event_sync(void *e) { Retire(*static_cast<uint64_t *>(e)); return 0; }
static uint64_t g_streamWaits = 0;
extern "C" uint64_t fake_rt_stream_waits(void) { return g_streamWaits; }
int mfrt_stream_wait_event(void *, void *) { ++g_streamWaits; return 0; }
int mfrt_event_done(void *) { return g_streamsRunning.load() != 0 ? 0 : 1; }
float mfrt_event_elapsed_ms(void *, void *) { return 0.0f; }
int mfrt_memcpy(void *dst, const void *src, uint64_t bytes) { std::memmove(dst, src, bytes); return 0; }
int mfrt_memcpy_async(void *dst, const void *src, uint64_t bytes, void *) { std::memmove(dst, src, bytes); return 0; }
int mfrt_memset(void *dst, int value, uint64_t bytes) { std::memset(dst, value, bytes); return 0; }

int mfk_xcopy_inline(const void *inlinePlan, int, uint32_t, void *mask, uint32_t maskValue, void *, int, uint32_t holdNanos)
{
    const mf::InlinePlan &p = *static_cast<const mf::InlinePlan *>(inlinePlan);
    g_lastHold = holdNanos;
    if (g_failLaunches > 0) {
        --g_failLaunches;
        return 719;
    }
    ++g_launches;
    static const bool skip = std::getenv("FAKE_RT_SKIP_COPY") != nullptr;   // host-path timing: the launch is free
    if (skip || g_skipCopies) {
        if (mask != nullptr && g_skipCopies) {
            *static_cast<uint64_t *>(mask) = maskValue;
        }
        return 0;
    }
    for (uint32_t c = 0; c < p.nchunk; ++c) {
        uint32_t below = 0;
        for (uint32_t i = 0; i < mf::kInlineSegs; ++i) {
            below += p.first[i] <= c ? 1u : 0u;
        }
        const uint32_t s = below - 1;
        RunChunk(p.src[s], p.dst[s], p.len[s], c - p.first[s], p.units);
    }
    if (mask != nullptr) {
        *static_cast<uint64_t *>(mask) = maskValue;
    }
    return 0;
}

int mfk_xcopy_done(const void *inlinePlan, int route, uint32_t, void *word, uint32_t value, void *counter, void *stream)
{
    return counter == nullptr ? -1 : mfk_xcopy_inline(inlinePlan, route, 0, word, value, stream, 0, 0);
}
int mfk_xcopy_windows_available(void) { return 1; }
int mfk_xcopy_prelaunch(void *) { return 0; }
// The calibration "measures" what the test has put here (all zero: nothing measured, the defaults stay).
static float g_calibration[8] = {};
static uint32_t g_calibrationHolds[3] = {};
static uint32_t g_calibrationRates[3] = {};
extern "C" void fake_rt_set_calibration(const float *us) { std::memcpy(g_calibration, us, sizeof(g_calibration)); }
extern "C" const uint32_t *fake_rt_calibration_holds(void) { return g_calibrationHolds; }
extern "C" const uint32_t *fake_rt_calibration_rates(void) { return g_calibrationRates; }
int mfk_xcopy_calibrate(void *, const uint32_t *holdNanos, const uint32_t *windowMBps, float *out)
{
    std::memcpy(g_calibrationHolds, holdNanos, sizeof(g_calibrationHolds));
    std::memcpy(g_calibrationRates, windowMBps, sizeof(g_calibrationRates));
    std::memcpy(out, g_calibration, sizeof(g_calibration));
    return 0;
}
uint32_t mfk_xcopy_window_units(void) { return 1024; }
int mfk_xcopy_windowed(const void *inlinePlan, uint32_t windowMBps, void *mask, uint32_t maskValue, void *stream)
{
    const mf::InlinePlan &p = *static_cast<const mf::InlinePlan *>(inlinePlan);
    if (p.units != 1024 || p.nchunk == 0 || windowMBps == 0) {
        return -1;
    }
    g_lastWindow = windowMBps;
    return mfk_xcopy_inline(inlinePlan, 0, p.nchunk, mask, maskValue, stream, 0, 0);
}

// As the kernel: the owner of a chunk by division under a pattern, else from the two group-map entries around it and the prefix between
// them.  A map whose entries do not bracket the owner fails the launch.
int mfk_xcopy_table(const void *tablePlan, int, uint32_t grid, void *mask, uint32_t maskValue, void *stream)
{
    NoteRecorded(stream);
    const mf::TablePlan &plan = *static_cast<const mf::TablePlan *>(tablePlan);
    const uint64_t *t = plan.triples;
    const uint32_t *f = plan.first;
    const uint32_t total = plan.nchunk;
    const uint32_t shift = plan.groupShift;
    const mf::ChunkPattern pat = plan.pattern;
    if (plan.nseg == 0 || grid == 0 || t == nullptr) {
        return -1;
    }
    if (pat.period != 0 && (pat.period > mf::kMaxPeriod || mf::PatternChunks(pat, plan.nseg) != total)) {
        return -1;
    }
    if (pat.period == 0 && (f == nullptr || plan.group == nullptr || shift < mf::kGroupShiftMin || shift > 31)) {
        return -1;
    }
    if (g_failLaunches > 0) {
        --g_failLaunches;
        return 719;
    }
    ++g_launches;
    g_lastTableShift = pat.period != 0 ? 0 : shift;
    TrackTable(t, 24ull * plan.nseg);
    if (g_skipCopies) {
        if (mask != nullptr) {
            *static_cast<uint64_t *>(mask) = maskValue;
        }
        return 0;
    }
    for (uint32_t c = 0; pat.period != 0 && c < total; ++c) {
        uint32_t seg = 0;
        uint32_t k = 0;
        mf::PatternOwner(pat, c, seg, k);
        RunChunk(t[3 * seg], t[3 * seg + 1], t[3 * seg + 2], k, plan.units);
    }
    for (uint32_t c = 0; pat.period == 0 && c < total; ++c) {
        const uint32_t lo = plan.group[c >> shift];
        const uint32_t hiEx = plan.group[(c >> shift) + 1] + 1;
        if (lo >= hiEx || hiEx > plan.nseg || f[lo] > c || f[hiEx] <= c) {
            ++g_groupMapErrors;
            return 720;
        }
        uint32_t s = lo;
        while (s + 1 < hiEx && f[s + 1] <= c) {
            ++s;
        }
        RunChunk(t[3 * s], t[3 * s + 1], t[3 * s + 2], c - f[s], plan.units);
    }
    if (mask != nullptr) {
        *static_cast<uint64_t *>(mask) = maskValue;
    }
    return 0;
}

void fake_rt_stream_chunks(uint32_t most) { g_streamChunks = most; }
void fake_rt_stream_launch_takes(uint32_t millis) { g_streamLaunchMillis = millis; }
uint64_t fake_rt_chunks_streamed(void) { return g_chunksStreamed.exchange(0); }

void fake_rt_stream_launches(uint32_t most) { g_streamLaunches = most; }
void fake_rt_stream_busy(uint32_t millis) { g_streamBusyMillis = millis; }
uint32_t g_streamPrelaunches = 0;
uint32_t fake_rt_stream_prelaunches(void) { return g_streamPrelaunches; }
int mfk_stream_prelaunch(void *) { ++g_streamPrelaunches; return 0; }

uint32_t fake_rt_most_chunks_launched(void)
{
    const uint32_t most = g_mostChunksLaunched;
    g_mostChunksLaunched = 0;
    return most;
}

// Chunk after chunk, with the words of both sides as the kernel reads and writes them.
static int RunChunks(bool beside, int toHost, void *ring, const void *chunks, void *hostWords, void *gpuWords, uint64_t base, uint32_t count, uint32_t slots,
                     uint32_t limitMillis)
{
    if (g_streamChunks == 0 || count == 0 || (toHost != 0 && count > slots) || g_streamLaunches == 0) {
        return -1;
    }
    --g_streamLaunches;
    if (!beside) {
        JoinStreamed();
        g_streamBase = base;
    }
    std::this_thread::sleep_for(std::chrono::milliseconds(g_streamLaunchMillis));
    ++g_launches;
    ++g_streamsRunning;
    g_mostChunksLaunched = count > g_mostChunksLaunched ? count : g_mostChunksLaunched;
    const uint64_t most = g_streamBase + g_streamChunks;
    const uint32_t busy = beside ? 0 : g_streamBusyMillis;
    g_streamThreads.emplace_back([=] {
        std::this_thread::sleep_for(std::chrono::milliseconds(busy));
        auto word = [](void *words, uint32_t slot) {
            return reinterpret_cast<uint64_t *>(static_cast<uint8_t *>(words) + static_cast<uint64_t>(slot) * mf::kStreamWordBytes);
        };
        for (uint32_t c = 0; c < count && base + c < most; ++c) {
            const mf::StreamChunk &chunk = static_cast<const mf::StreamChunk *>(chunks)[c];
            const uint32_t slot = c % slots;
            if (toHost == 0) {
                const auto start = std::chrono::steady_clock::now();
                while (__atomic_load_n(word(hostWords, slot), __ATOMIC_ACQUIRE) != base + c + 1) {
                    if (std::chrono::steady_clock::now() - start > std::chrono::milliseconds(limitMillis)) {
                        --g_streamsRunning;
                        return;
                    }
                    std::this_thread::yield();
                }
            }
            const uint64_t skip = chunk.at & (mf::kStreamLine - 1);
            uint8_t *there = static_cast<uint8_t *>(ring) + static_cast<uint64_t>(slot) * mf::kStreamChunkBytes + skip;
            if (chunk.len == 0 || skip + chunk.len > mf::kStreamChunkBytes) {
                break;
            }
            uint8_t *at = reinterpret_cast<uint8_t *>(chunk.at);
            std::memcpy(toHost != 0 ? there : at, toHost != 0 ? at : there, chunk.len);
            ++g_chunksStreamed;
            __atomic_store_n(word(gpuWords, slot), base + c + 1, __ATOMIC_RELEASE);
        }
        --g_streamsRunning;
    });
    return 0;
}
int mfk_stream_chunks(int toHost, void *ring, const void *chunks, void *hostWords, void *gpuWords, uint64_t base, uint32_t count, uint32_t slots,
                      uint32_t limitMillis, void *)
{
    return RunChunks(false, toHost, ring, chunks, hostWords, gpuWords, base, count, slots, limitMillis);
}
int mfk_stream_chunks_beside(int toHost, void *ring, const void *chunks, void *hostWords, void *gpuWords, uint64_t base, uint32_t count,
                             uint32_t slots, uint32_t limitMillis, void *)
{
    return RunChunks(true, toHost, ring, chunks, hostWords, gpuWords, base, count, slots, limitMillis);
}

// The pieces in the order of the kernel's workgroups.  One that is longer than its workgroup or reaches past the end of the list
// fails the launch.
int mfk_xcopy_pieces(const void *pieces, uint32_t count, uint64_t bytes, uint32_t units, void *mask, uint32_t maskValue,
                     void *stream, uint32_t holdNanos, void *event)
{
    NoteRecorded(stream);
    g_lastTableHold = holdNanos;
    g_lastPieceWait = mf::PieceHoldNanos(holdNanos, count, bytes, units);
    g_mostPieces = count > g_mostPieces ? count : g_mostPieces;
    g_leastPieceWait = g_lastPieceWait < g_leastPieceWait ? g_lastPieceWait : g_leastPieceWait;
    if (pieces == nullptr || count == 0 || (units != 256 && units != 512 && units != 1024)) {
        return -1;
    }
    if (g_failLaunches > 0) {
        --g_failLaunches;
        return 719;
    }
    ++g_launches;
    const mf::Piece *p = static_cast<const mf::Piece *>(pieces);
    TrackTable(p, sizeof(mf::Piece) * count);
    uint64_t moved = 0;
    for (uint32_t w = 0; w < (count + 63) / 64 * 64; ++w) {
        const uint32_t at = mf::PieceOf(w);
        if (at >= count) {
            continue;
        }
        const uint64_t src = p[at].src & mf::kPieceAddress;
        const uint64_t dst = p[at].dst & mf::kPieceAddress;
        const uint32_t len = mf::PieceLength(p[at].src, p[at].dst);
        if (len == 0 || mf::SegmentGeometry(dst, len).body > units) {
            return 720;
        }
        moved += len;
        if (!g_skipCopies) {
            RunChunk(src, dst, len, 0, units);
        }
    }
    if (moved != bytes) {
        return 721;
    }
    if (event != nullptr) {
        (void)mfrt_event_record(event, stream);
    }
    if (mask != nullptr) {
        *static_cast<uint64_t *>(mask) = maskValue;
    }
    return 0;
}

// The same with a word for the end of the copy.
int mfk_xcopy_pieces_done(const void *pieces, uint32_t count, void *word, uint32_t value, void *counter, void *stream)
{
    return counter == nullptr || word == nullptr ? -1 : mfk_xcopy_pieces(pieces, count, 0, 256, word, value, stream, 0, nullptr);
}
// The same in windows, whatever the addresses: the rate is noted.
int mfk_xcopy_pieces_windowed(const void *pieces, uint32_t count, uint64_t bytes, uint32_t windowMBps, uint32_t reading, void *mask,
                              uint32_t maskValue, void *stream, void *event)
{
    g_lastWindow = windowMBps;
    g_lastReading = reading;
    return windowMBps == 0 ? -1 : mfk_xcopy_pieces(pieces, count, bytes, 1024, mask, maskValue, stream, 0, event);
}

// When this launch starts, those before it have ended; with a counter its own list has been read when it says so.
int mfk_xcopy_pieces_reported(const void *pieces, uint32_t count, uint64_t bytes, uint32_t units, uint32_t holdNanos, uint32_t windowMBps,
                              uint32_t reading, void *word, uint32_t value, void *counter, void *stream)
{
    if (counter == nullptr) {
        Retire(g_flightSeq);
    }
    const int err = windowMBps != 0 ? mfk_xcopy_pieces_windowed(pieces, count, bytes, windowMBps, reading, nullptr, 0, stream, nullptr)
                                    : mfk_xcopy_pieces(pieces, count, bytes, units, nullptr, 0, stream, holdNanos, nullptr);
    if (err == 0 && counter != nullptr && g_withholdReports) {
        std::lock_guard<std::mutex> guard(g_reportLock);
        g_withheldReports.emplace_back(static_cast<uint64_t *>(word), value);
        return 0;
    }
    if (err == 0) {
        if (counter != nullptr) {
            std::lock_guard<std::mutex> guard(g_flightLock);
            g_inFlight.pop_back();
        }
        __atomic_store_n(static_cast<uint64_t *>(word), static_cast<uint64_t>(value), __ATOMIC_RELEASE);
    }
    return err;
}

// The direct copy of a device-resident table restated: the parts of every segment, and the pieces of what long ones have left out
// of a list.
int mfk_xcopy_direct(const void *triples, uint32_t nseg, uint32_t units, int, uint32_t grid, uint32_t restGrid, void *rest,
                     uint32_t capacity, uint32_t windowMBps, void *mask, uint32_t maskValue, void *stream, void *event)
{
    if (event != nullptr) {
        (void)mfrt_event_record(event, stream);
    }
    g_lastRestList = rest;
    g_lastTableWindow = windowMBps;
    g_lastTableGrid = grid;
    mf::RestList *list = static_cast<mf::RestList *>(rest);
    if (nseg == 0 || nseg > capacity || grid == 0 || restGrid == 0 || list == nullptr || list->taken != 0 || list->done[0].count != 0) {
        return -1;
    }
    ++g_launches;
    const uint64_t *t = static_cast<const uint64_t *>(triples);
    uint64_t parts = 1;
    for (uint32_t i = 0; i < mf::kDirectSample && i < nseg; ++i) {
        const uint64_t chunks = mf::SegmentChunks(t[3 * i + 1], t[3 * i + 2], units);
        parts = chunks > parts ? (chunks < mf::kDirectMaxParts ? chunks : mf::kDirectMaxParts) : parts;
    }
    const uint64_t own = parts * mf::kDirectRounds;
    for (uint64_t item = 0; item < nseg * parts; ++item) {
        const uint64_t seg = item / parts;
        const uint64_t part = item % parts;
        const uint64_t src = t[3 * seg];
        const uint64_t dst = t[3 * seg + 1];
        const uint64_t len = t[3 * seg + 2];
        const uint64_t chunks = mf::SegmentChunks(dst, len, units);
        for (uint64_t c = part; c < chunks && c < own; c += parts) {
            RunChunk(src, dst, len, c, units);
        }
        if (part != 0 || chunks <= own) {
            continue;
        }
        const uint64_t at = mf::SegmentGeometry(dst, len).head + own * units * mf::kUnitBytes;
        const uint64_t before = list->taken;
        list->taken += mf::kRestEntry + mf::RestPieces(len - at);
        list->entry[before / mf::kRestEntry] = mf::RestSegment{before % mf::kRestEntry, src + at, dst + at, len - at};
    }
    ++g_launches;
    const uint64_t pieces = list->taken % mf::kRestEntry;
    uint32_t e = 0;
    for (uint64_t p = 0; p < pieces; ++p) {
        while (e + 1 < list->taken / mf::kRestEntry && list->entry[e + 1].first <= p) {
            ++e;
        }
        const mf::RestSegment &r = list->entry[e];
        const uint64_t from = (p - r.first) * mf::kRestPieceBytes;
        const uint64_t len = r.len - from < mf::kRestPieceBytes ? r.len - from : mf::kRestPieceBytes;
        for (uint64_t c = 0; c < mf::SegmentChunks(r.dst + from, len, units); ++c) {
            RunChunk(r.src + from, r.dst + from, len, c, units);
        }
    }
    list->taken = 0;
    if (mask != nullptr) {
        *static_cast<uint64_t *>(mask) = maskValue;
    }
    return 0;
}

// One launch without a list: as far as the users of lists go, one that no other call has.
int mfk_xcopy_planned(const void *triples, uint32_t nseg, uint32_t, uint32_t, uint32_t, void *mask, uint32_t maskValue, void *)
{
    static uint8_t none[4096];
    static uint32_t turn = 0;
    g_lastRestList = &none[++turn % 4096];
    if (triples == nullptr || nseg == 0 || nseg > mf::kPlannedSegments) {
        return -1;
    }
    ++g_launches;
    const uint64_t *t = static_cast<const uint64_t *>(triples);
    for (uint32_t i = 0; i < nseg; ++i) {
        for (uint64_t c = 0; c < mf::SegmentChunks(t[3 * i + 1], t[3 * i + 2], 1024); ++c) {
            RunChunk(t[3 * i], t[3 * i + 1], t[3 * i + 2], c, 1024);
        }
    }
    if (mask != nullptr) {
        *static_cast<uint64_t *>(mask) = maskValue;
    }
    return 0;
}

static uint64_t g_signals = 0;
static uint64_t g_streamSyncs = 0;
extern "C" uint64_t fake_rt_signals() { return g_signals; }
extern "C" uint64_t fake_rt_stream_syncs() { return g_streamSyncs; }
extern "C" void fake_rt_count_stream_sync(void) { ++g_streamSyncs; }
int mfk_xcopy_signal(void *word, uint32_t value, void *)
{
    // not counted: fake_rt_launches() counts the launches that move data
    ++g_signals;
    __atomic_store_n(static_cast<uint64_t *>(word), static_cast<uint64_t>(value), __ATOMIC_RELEASE);
    return 0;
}
int mfk_xcopy_clear_lists(void *lists, uint32_t count, uint64_t stride, void *)
{
    for (uint32_t i = 0; i < count; ++i) {
        std::memset(static_cast<uint8_t *>(lists) + i * stride, 0, mf::kRestHeadBytes);
    }
    return 0;
}
int mfk_xcopy_static_setup(void) { return 0; }
int mfk_xcopy_table_static(const void *triples, uint32_t nseg, uint32_t units, int route, uint32_t grid, uint32_t restGrid, void *stream)
{
    static std::vector<uint64_t> list(mf::RestListBytes(MFK_STATIC_TABLE_SEGMENTS) / 8, 0);
    if (nseg == 0 || nseg > MFK_STATIC_TABLE_SEGMENTS) {
        return -1;
    }
    return mfk_xcopy_direct(triples, nseg, units, route, grid, restGrid, list.data(), MFK_STATIC_TABLE_SEGMENTS, 0, nullptr, 0, stream, nullptr);
}

static uint32_t g_lastRectMates = 0;
extern "C" uint32_t fake_rt_last_rect_mates() { return g_lastRectMates; }

// Walks the chunks as the kernel's workgroups do, so a wrong chunk-to-rectangle rule leaves rows uncopied.
int mfk_copy2d(const void *rectPlan, uint32_t, void *)
{
    const mf::RectPlan &p = *static_cast<const mf::RectPlan *>(rectPlan);
    ++g_launches;
    g_lastRectMates = 0;
    for (uint32_t r = 0; r < mf::kRectInline; ++r) {
        g_lastRectMates += p.mate[r] != 0 ? 1u : 0u;
    }
    for (uint32_t c = 0; c < p.nchunk; ++c) {
        uint32_t r = 0;
        uint32_t k = 0;
        mf::RectOfChunk(p, c, r, k);
        const uint32_t row0 = k * p.rowsPerChunk[r];
        for (uint32_t row = row0; row < row0 + p.rowsPerChunk[r] && row < p.height[r]; ++row) {
            std::memmove(reinterpret_cast<void *>(p.dst[r] + 16ull * p.dpitchUnits[r] * row),
                         reinterpret_cast<void *>(p.src[r] + 16ull * p.spitchUnits[r] * row), 16ull * p.widthUnits[r]);
        }
    }
    return 0;
}

// Chunks of the payload taken row-major, unit by unit as the kernel's lanes do; pairs of rectangles as rows of two halves.
static uint32_t g_rectWindowed = 0;
static uint32_t g_rectChunked = 0;
extern "C" uint32_t fake_rt_rect_windowed_launches() { return g_rectWindowed; }
extern "C" uint32_t fake_rt_rect_chunked_launches() { return g_rectChunked; }
int mfk_copy2d_chunks(const void *rectChunkPlan, uint32_t windowMBps, void *)
{
    const mf::RectChunkPlan &p = *static_cast<const mf::RectChunkPlan *>(rectChunkPlan);
    const uint32_t units = windowMBps != 0 ? mf::kRectWindowUnits : 64 * mf::kRectChunkDepth;
    ++g_launches;
    ++g_rectChunked;
    g_rectWindowed += windowMBps != 0 ? 1 : 0;
    g_lastWindow = windowMBps;
    for (uint32_t c = 0; c < p.nchunk && !g_skipCopies; ++c) {
        uint32_t r = 0;
        while (r + 1 < mf::kRectInline && p.first[r + 1] <= c) {
            ++r;
        }
        const uint32_t ru = p.rowUnits[r];
        const uint32_t base = (c - p.first[r]) * units;
        const uint32_t total = p.height[r] * ru;
        const uint32_t row0 = base / ru;
        for (uint32_t u = 0; u < units && base + u < total; ++u) {
            uint32_t row = 0;
            uint32_t col = 0;
            mf::RectWindowRowCol(base - row0 * ru + u, ru, p.magic[r], row, col);
            const uint64_t from = col < p.halfUnits[r] ? p.src[r] : p.other[r] - 16ull * p.halfUnits[r];
            std::memmove(reinterpret_cast<void *>(p.dst[r] + 16ull * (static_cast<uint64_t>(p.dpitchUnits[r]) * (row0 + row) + col)),
                         reinterpret_cast<void *>(from + 16ull * (static_cast<uint64_t>(p.spitchUnits[r]) * (row0 + row) + col)), 16);
        }
    }
    return 0;
}
int mfk_copy2d_prelaunch(void *) { return 0; }

uint64_t mfk_moe_workspace_bytes(uint32_t, uint32_t, uint32_t) { return 0; }
int mfk_moe_dispatch(const void *, const void *, uint32_t, uint32_t, uint32_t, uint32_t, void *, void *, void *, void *, void *,
                     void *, void *) { return -1; }
static int g_lastCombinePaced = -1;
extern "C" int fake_rt_last_combine_paced() { return g_lastCombinePaced; }
int mfk_moe_combine(const void *, const void *, const void *, uint32_t, uint32_t, uint32_t, void *, void *, int paced)
{
    g_lastCombinePaced = paced;
    return 0;
}
void mfk_moe_combine_windows(uint32_t, uint32_t) {}
int mfk_moe_dispatch_counts(uint32_t, uint32_t, uint32_t, uint32_t) { return 0; }
int mfk_moe_combine_stays(uint32_t, uint32_t, uint32_t) { return 0; }
int mfk_moe_setup(void) { return 0; }
int mfk_moe_xcd_streams(void) { return 0; }
}
