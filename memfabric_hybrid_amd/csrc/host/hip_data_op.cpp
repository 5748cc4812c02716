#include "hip_data_op.h"
#include "host_copy.h"

#include <algorithm>
#include <atomic>
#include <chrono>
#include <cstring>
#include <thread>
#include <vector>

#include "../../../include/mf_hip_dataplane.h"
#include "../kernels/staging.h"
#include "../rt/mf_rt.h"
#include "copy_direction.h"
#include "mf_log.h"
#include "xcopy_engine.h"

namespace mf {
namespace {

// The staging ring.  A round is a launch, which has a start and an end in which the link is not full (8 MiB move at 55.4 GB/s, 2 MiB at
// 51.9), so rounds are as long as the ring allows; the first of a copy to the GPU and the last of one from it are short, because
// the other side waits for them.
constexpr uint32_t kSlots = 4;
constexpr uint64_t kRoundBytes = 8ull << 20;           // bytes per slot, the most one round moves
// A little more than HostCopyHelper shares among cores, so that a round stays shared when its pieces are padded: at 512 KiB 1 MB in
// seven parts took 44 us to the GPU, in one part 37.
constexpr uint64_t kRoundMinBytes = 576ull << 10;
static_assert(kRoundMinBytes > HostCopyHelper::kSplitMin, "a round of the least size is copied by several cores");
constexpr uint64_t kBounceBytes = kSlots * kRoundBytes;
constexpr uint32_t kAhead = 2;                         // launches queued beyond the slot being emptied (device to pageable memory)

// Caller memory the GPU cannot address (ordinary pageable host memory) goes through a pinned
// staging area.  The reference allocates and frees a device buffer per segment for these
// directions (src/hybm/csrc/data_operation/host/hybm_data_op_sdma.cpp:171-221); here one pinned
// area per thread, owned by the engine, is filled by the CPU and scattered by one launch.

inline void CpuRelax()
{
#if defined(__x86_64__) || defined(__i386__)
    __builtin_ia32_pause();
#else
    std::this_thread::yield();
#endif
}

bool AnyPageable(void *const *ptrs, uint32_t n)
{
    for (uint32_t i = 0; i < n; ++i) {
        if (mfrt_pointer_kind(ptrs[i]) == MFRT_PTR_PAGEABLE) {
            return true;
        }
    }
    return false;
}

// Walks the bytes of a batch in rounds.
class RoundCursor {
public:
    RoundCursor(void *const *src, void *const *dst, const uint64_t *len, uint32_t n) : src_(src), dst_(dst), len_(len), n_(n)
    {
        for (uint32_t i = 0; i < n; ++i) {
            left_ += len[i];
        }
        Skip();
    }
    uint64_t Left() const
    {
        return left_;
    }
    // The next pieces, at most `bytes` with every piece on a 64-byte boundary of the slot; place(src, dst, len, offset in the slot).
    template <class Place>
    void Next(uint64_t bytes, Place place)
    {
        uint64_t used = 0;
        while (i_ < n_ && used < bytes) {
            const uint64_t rest = len_[i_] - at_;
            const uint64_t take = rest < bytes - used ? rest : bytes - used;
            if (take < rest && take < kSliver && used != 0) {
                break;   // too little of a segment to be worth a piece of its own
            }
            place(reinterpret_cast<uint64_t>(src_[i_]) + at_, reinterpret_cast<uint64_t>(dst_[i_]) + at_, take, used);
            used += (take + 63) & ~63ull;
            at_ += take;
            left_ -= take;
            Skip();
        }
    }

private:
    static constexpr uint64_t kSliver = 4096;
    void Skip()   // finished and empty segments
    {
        while (i_ < n_ && at_ == len_[i_]) {
            ++i_;
            at_ = 0;
        }
    }
    void *const *src_;
    void *const *dst_;
    const uint64_t *len_;
    uint32_t n_;
    uint32_t i_ = 0;
    uint64_t at_ = 0;
    uint64_t left_ = 0;
};

// The launches of one staged copy.  Whatever way it ends, nothing of it is in flight afterwards: its slots are free.
class StagedLaunches {
public:
    explicit StagedLaunches(void *stream) : stream_(stream) {}
    ~StagedLaunches()
    {
        (void)Finish();
    }
    int Launch(const std::vector<uint64_t> &src, const std::vector<uint64_t> &dst, const std::vector<uint64_t> &len, int route)
    {
        const int ret = XcopyEngine::Instance().SubmitTicket(src.data(), dst.data(), len.data(), static_cast<uint32_t>(len.size()), route,
                                                             stream_, tickets_[count_ % kSlots]);
        count_ += ret == BM_OK ? 1 : 0;
        return ret;
    }
    // Waits for launch `index`, one of the last kSlots.
    int Wait(uint32_t index)
    {
        waited_ = index + 1 > waited_ ? index + 1 : waited_;
        return XcopyEngine::Instance().WaitTicket(tickets_[index % kSlots], stream_);
    }
    int Finish()
    {
        return waited_ < count_ ? Wait(count_ - 1) : BM_OK;
    }
    uint32_t Count() const
    {
        return count_;
    }

private:
    void *stream_;
    uint32_t count_ = 0;
    uint32_t waited_ = 0;
    uint32_t tickets_[kSlots] = {};
};

// Bytes of the next round, of `left`.  What is left may be half as much again: a round of its own would cost it more than it overlaps.
uint64_t RoundBytes(uint64_t wanted, uint64_t left)
{
    const uint64_t bytes = wanted < kRoundMinBytes ? kRoundMinBytes : wanted > kRoundBytes ? kRoundBytes : wanted & ~63ull;
    return left <= bytes + bytes / 2 && bytes + bytes / 2 <= kRoundBytes ? kRoundBytes : bytes;
}

// The same area as a ring of short slots, for copies whose launches run while the CPU fills or empties it (kernels/staging.hip): the
// link has work from the first 64 KiB on, and no round waits for a launch or for its completion word.  What follows the ring stays from
// copy to copy: the words of both sides, what they count from, and the launches' list.
constexpr uint32_t kStreamSlots = 512;
constexpr uint32_t kStreamListChunks = 1u << 13;       // 512 MiB: a longer copy is several
// Chunks of one launch, 4 MiB.  A launch that waits for the CPU holds its hardware queue, and with it the launches of other streams that the
// runtime has put there: a small kernel and its wait beside loads of 64 MiB, median and 99 % in us, one launch for the whole copy 1201 and 1243, of 8
// MiB 157 / 173, of 4 MiB 81 / 98, of 2 MiB 43 / 79 (in rounds 95 to 146 / 470); the load 1252, 1253, 1257 and 1274 (1330 to 1350).  Beside loads of 4 MiB
// 92 / 102, of 2 MiB 50 / 80 (41 to 54 / 91).
constexpr uint32_t kStreamLaunchChunks = 64;
constexpr uint32_t kStreamLead = 24;                    // chunks in front of its end at which the next one goes out: the link takes 28 us for them
static_assert(kStreamSlots % kStreamLaunchChunks == 0, "a launch's slots lie side by side");
struct StreamArea {
    uint8_t ring[kStreamSlots][kStreamChunkBytes];
    struct Word {
        uint64_t value;
        uint64_t reserved[7];
    };
    static_assert(sizeof(Word) == kStreamWordBytes, "");
    Word host[kStreamSlots];
    Word gpu[kStreamSlots];
    Word base;
    StreamChunk list[kStreamListChunks];
};
static_assert(sizeof(StreamArea::ring) == kBounceBytes, "the rounds use it too, and nothing behind it");
// What is one round stays one: 512 KiB to the host 21.9 us, streamed 24.5, and below kSplitMin a copy of its own would wake the helpers for it (260 KB to the GPU 2 ms
// behind the last 24 us, streamed 33).  Before / streamed, us, to the GPU and back: 1 MiB 37.7 / 32.4, 40.8 /
// 36.5, 2 MiB 65.6 / 54.4, 63.4 / 56.0; 2 ms behind the last 53.2 / 45.2, 54.5 / 50.0, 74.4 / 67.7, 73.1 / 68.0.
constexpr uint64_t kStreamMinBytes = kRoundMinBytes / 2 * 3 + 1;
// A chunk costs a launch 0.33 us beyond its bytes, so a list that makes many more of them than full ones would be goes in rounds, which gather: at most 16 more, and one for 128 KiB, up
// to 64.  us, rounds / streamed, one behind the other and 2 ms apart, to the GPU and back:
//     segments              more chunks, of     to the GPU                        back
//     32 of 32 768             16      24       37 / 34          58 / 49          42 / 35          60 / 49
//     20 of 4096 and 61 440    20      26       41 / 44          68 / 60          41 / 43          57 / 57
//     36 of 28 672             20      24       37 / 36          58 / 52          42 / 36          58 / 51
//     42 of 24 576             26      24       37 / 39          60 / 56          42 / 37          60 / 51
//     52 of 20 000             36      24       37 / 42          60 / 58          42 / 39          60 / 54
//     64 of 16 384             48      24       38 / 46          60 / 62          43 / 41          60 / 56
//     60 of 1024, 1 MiB        60      24       39 / 66          59 / 75          46 / 52          59 / 67
//     64 of 32 768             32      32       62 / 63          76 / 75          63 / 57          77 / 72
//     128 of 32 768            64      48      106 / 112        122 / 123        107 / 101        115 / 116
//     119 of 70 000           111      64      190 / 198        204 / 210        186 / 178        192 / 193
//     204 of 40 960            77      64      186 / 192        204 / 205        180 / 180        189 / 193
//     512 of 16 384           384      64      195 / 301            -            187 / 252            -
//     292 of 57 344            36      64      339 / 339            -
//     341 of 49 152            85      64      341 / 348        357 / 356
//     4096 of 16 384         3072      64     1267 / 2294           -
constexpr uint64_t kStreamShortLeast = 16;
constexpr uint64_t kStreamShortBytes = 128ull << 10;
constexpr uint64_t kStreamShortMost = 64;
// A segment whose last chunk would be this short is cut into equal ones: full chunks and short ones in turn leave most of the work to a part of the launch's
// workgroups, which take every eighth or sixteenth.  us, a launch a round / full chunks and a tail / equal ones: 22 segments of 68 181 bytes in 47.8 / 51.6 /
// 46.9, out 46.4 / 47.6 / 46.1; 32 of 72 022 in 71.0 / 74.3 / 69.8; out 32 of 203 125 145.4 / 147.6 / 139.7, of 100 000 80.6 / 78.5 / 75.1; but 4 of 375 000, a tail of
// 47 320, 46.0 / 43.9 / 45.8, and 32 of 250 000, one of 53 392, 179.0 / 168.5 / 170.9.
constexpr uint64_t kStreamShortTail = kStreamChunkBytes / 8 * 5;
// To the host rounds are the better from here on: a core empties its share of one, 2 MiB, in one piece, sooner than as many chunks (10 MiB 216 to 229 us, streamed 214 in
// some processes and 245 in others; 8 MiB in 20 parts 188 / 175).
constexpr uint64_t kStreamMostBytesOut = kRoundBytes;
static_assert(2 * (kStreamMostBytesOut / kStreamChunkBytes + kStreamShortMost) <= kStreamSlots, "to the host no slot is used twice, and a segment off a line may make one chunk more");
// Copies of so many bytes go past the CPU's caches, which they would sweep, ring and all.  us, rounds by memcpy / rounds past the caches / streamed: to the host 4 MiB 103 / 108 / 96, 8 MiB in 20
// parts 188 / 191 / 172, 12 MiB 265 / 255 / 253, 16 MiB 376 / 338 / 334, 64 MiB 1273 / 1242 / 1352; to the GPU 4 MiB 109 / 114 / 101, 16 MiB 370 / 350 / 340, 64 MiB 1339 / 1286 /
// 1262, 128 MiB 2559 / 2503 / 2490.  What reads the caller's array next is no slower for it, as the caches that memcpy leaves it in are mostly other cores': a save and a sum over
// the array on one core, by memcpy / past the caches, medians on three machines, 12 MiB 629 / 582, 16 MiB 816 / 724, 64 MiB 2834 / 2739; and a copy of it 705 / 706 (on one of them 632 / 721),
// 918 / 876, 3403 / 3362.
// Saves of short segments do so from 48 MiB on only.  us, rounds by memcpy / past the caches, two processes each: 16 MiB in segments of 16 KiB 359 / 385, 64 KiB 334 / 348, 512 KiB 329 / 338, 1 MiB, which memcpy
// itself writes another way, 367 / 337; 24 MiB 516 / 536, 484 / 498, 483 / 487, 508 / 486; 32 MiB of 16 and 512 KiB 676 / 691, 630 / 634; 40 MiB 852 / 848, 782 / 783; 48 MiB 1032 / 1002, 948 / 931; 64 MiB 1354 /
// 1315, 1267 / 1232.  Loads of short segments gain as the others do: 1024 of 16 KiB 383 / 361.
constexpr uint64_t kPastCachesBytes = 12ull << 20;
constexpr uint64_t kPastCachesLongSegment = 1ull << 20;
constexpr uint64_t kPastCachesShortBytes = 48ull << 20;
constexpr uint32_t kStreamLimitMillis = 1000;
constexpr uint32_t kStreamLookMillis = 50;              // without a word from the GPU: then whether it has left
constexpr uint32_t kStreamIdleMicros = 100;             // a launch on an idle stream says its first word after some 20
constexpr uint32_t kStreamPollMicros = 1000;
constexpr uint32_t kStreamSleepMicros = 100;            // what the ring holds keeps the GPU busy for as long and longer

StreamArea *AreaOf(XcopyEngine &engine)
{
    bool fresh = false;
    auto *area = static_cast<StreamArea *>(engine.ThreadBounce(sizeof(StreamArea), &fresh));
    if (area != nullptr && fresh) {
        std::memset(area->host, 0, sizeof area->host);
        std::memset(area->gpu, 0, sizeof area->gpu);
        area->base.value = 0;
    }
    return area;
}

// A copy of up to kStreamListChunks.  The caller and the helpers take chunk after chunk, each only when the GPU is done with its slot, so that whoever
// finds nothing to do can leave at any time.  The helpers do so after kStreamIdleMicros: a stream that has other work in front of the
// launch is waited for by the caller alone, which polls as long as it does for a round, and then sleeps.  CPU time of a call behind 30 ms
// of matrix products, with all of them polling for it / so: 1 MiB to the host 115 ms / 31 (the runtime polls too), 64 MiB to the GPU 127 / 6.
struct Streaming {
    StreamArea *area;
    bool toHost;
    bool pastCaches;
    uint64_t base;
    uint32_t count;
    void *stream;
    const uint8_t *const *memory;       // the caller's, by chunk
    std::atomic<uint32_t> next{0};
    uint32_t launched = 0;              // chunks; the caller launches
    uint32_t launches = 0;
    int error = 0;                      // of a launch
    bool stopped = false;               // the launches have ended, or never began, with chunks left

    // The next launch goes out when the one before is nearly done, and beside it, so that the link is not left idle in between.
    bool LaunchMore()
    {
        if (launched >= count || error != 0 || (launched != 0 && !Done(launched - kStreamLead))) {
            return false;
        }
        const uint32_t slot = launched % kStreamSlots;
        const uint32_t some = std::min(count - launched, kStreamLaunchChunks);
        const auto launch = launched == 0 ? mfk_stream_chunks : mfk_stream_chunks_beside;
        error = launch(toHost ? 1 : 0, area->ring[slot], area->list + launched, area->host + slot, area->gpu + slot, base + launched, some,
                       kStreamSlots - slot, kStreamLimitMillis, stream);
        if (error != 0) {
            return false;
        }
        launched += some;
        ++launches;
        return true;
    }
    bool Done(uint32_t c) const         // the GPU with chunk c in its slot
    {
        return __atomic_load_n(&area->gpu[c % kStreamSlots].value, __ATOMIC_ACQUIRE) == base + c + 1;
    }
    bool MayTake(uint32_t c) const
    {
        return toHost ? Done(c) : c < kStreamSlots || Done(c - kStreamSlots);
    }
    void Copy(void *to, const void *from, uint32_t len) const
    {
        if (pastCaches) {
            HostCopyHelper::StreamCopy(to, from, len);
        } else {
            std::memcpy(to, from, len);
        }
    }
    void Move(uint32_t c)
    {
        const uint32_t slot = c % kStreamSlots;
        const StreamChunk &chunk = area->list[c];
        uint8_t *there = area->ring[slot] + (chunk.at & (kStreamLine - 1));
        if (toHost) {
            Copy(const_cast<uint8_t *>(memory[c]), there, chunk.len);
        } else {
            Copy(there, memory[c], chunk.len);
        }
        __atomic_store_n(&area->host[slot].value, base + c + 1, __ATOMIC_RELEASE);
    }
    // Until all chunks are taken, or none can be for a while.
    void Work(bool helps)
    {
        std::chrono::steady_clock::time_point since{};
        for (uint32_t idle = 0;;) {
            if (!helps) {
                (void)LaunchMore();
            }
            uint32_t c = next.load(std::memory_order_relaxed);
            if (c >= count) {
                return;
            }
            if (MayTake(c)) {
                if (next.compare_exchange_weak(c, c + 1, std::memory_order_relaxed)) {
                    Move(c);
                    idle = 0;
                }
                continue;
            }
            CpuRelax();
            if (++idle % 64 != 0) {
                continue;
            }
            const auto now = std::chrono::steady_clock::now();
            if (idle == 64) {
                since = now;
            } else if (now - since > std::chrono::microseconds(kStreamIdleMicros)) {
                return;
            }
        }
    }
    static void Part(void *context)
    {
        static_cast<Streaming *>(context)->Work(true);
    }
    // The caller's wait for the GPU, with the helpers given back.  What ends it is that done() says so, or that the launches have.
    template <class F>
    bool Await(F done)
    {
        // Behind the launches: others may put work on the stream for as long as this lasts, so that it need not become idle.
        struct Marker {
            void *event = nullptr;
            bool recorded = false;
            ~Marker()
            {
                if (event != nullptr) {
                    (void)mfrt_event_destroy(event);
                }
            }
        } marker;
        auto start = std::chrono::steady_clock::now();
        auto looked = start;
        for (uint32_t polls = 1; !done(); ++polls) {
            if (LaunchMore()) {
                start = looked = std::chrono::steady_clock::now();
                marker.recorded = false;
            }
            if (error != 0) {
                return false;
            }
            if (polls % 64 != 0) {
                CpuRelax();
                continue;
            }
            const auto now = std::chrono::steady_clock::now();
            if (now - start < std::chrono::microseconds(kStreamPollMicros)) {
                continue;
            }
            polls = 63;
            if (launched >= count && (toHost || next.load(std::memory_order_relaxed) >= count)) {    // they need nothing more of the CPU
                stopped = mfrt_stream_sync(stream) != 0 || !done();
                return !stopped;
            }
            std::this_thread::sleep_for(std::chrono::microseconds(kStreamSleepMicros));
            if (now - looked > std::chrono::milliseconds(kStreamLookMillis)) {
                looked = now;
                if (!marker.recorded) {
                    marker.event = marker.event != nullptr ? marker.event : mfrt_event_create();
                    marker.recorded = marker.event != nullptr && mfrt_event_record(marker.event, stream) == 0;
                }
                // the words of a launch that is over have all arrived
                const int over = marker.recorded ? mfrt_event_done(marker.event) : mfrt_stream_done(stream);
                if (over != 0 && !done()) {
                    if (LaunchMore()) {
                        marker.recorded = false;
                        continue;
                    }
                    stopped = true;
                    return false;
                }
            }
        }
        return true;
    }
    void Run(HostCopyHelper &helper)
    {
        bool begun = helper.Begin(&Streaming::Part, this);
        for (;;) {
            Work(false);
            helper.End(begun);
            if (next.load(std::memory_order_relaxed) >= count) {
                break;
            }
            if (!Await([&] { return MayTake(next.load(std::memory_order_relaxed)); })) {
                return;
            }
            begun = helper.Begin(&Streaming::Part, this);
        }
        uint32_t seen = count <= kStreamSlots ? 0 : count - kStreamSlots;
        (void)(toHost || Await([&] {
            while (seen < count && Done(seen)) {
                ++seen;
            }
            return seen == count;
        }));
    }
};

bool Streams(const uint64_t *len, uint32_t n, bool toHost, void *stream)
{
    uint64_t total = 0;
    uint64_t chunks = 0;
    for (uint32_t i = 0; i < n; ++i) {
        total += len[i];
        chunks += len[i] / kStreamChunkBytes + (len[i] % kStreamChunkBytes != 0 ? 1 : 0);
    }
    return total >= kStreamMinBytes && !(toHost && total > kStreamMostBytesOut) &&
           chunks <= total / kStreamChunkBytes + std::min(kStreamShortLeast + total / kStreamShortBytes, kStreamShortMost) && mfrt_stream_capturing(stream) == 0;
}

constexpr int kNotStreamed = 1;

// kNotStreamed where the copy has to be made in rounds, all of it: it cannot be launched, or the GPU has left it.
int StreamAll(void *const *src, void *const *dst, const uint64_t *len, uint32_t n, bool toHost, void *stream)
{
    StreamArea *area = AreaOf(XcopyEngine::Instance());
    if (area == nullptr || mfrt_bind_thread() != 0) {
        return kNotStreamed;
    }
    uint64_t total = 0;
    for (uint32_t i = 0; i < n; ++i) {
        total += len[i];
    }
    std::vector<const uint8_t *> memory;
    memory.reserve(std::min<uint64_t>(kStreamListChunks, total / kStreamChunkBytes + 2ull * n));
    HostCopyHelper &helper = HostCopyHelper::Instance();
    uint32_t i = 0;
    uint64_t at = 0;
    while (i < n) {
        memory.clear();
        uint32_t count = 0;
        while (i < n && count < kStreamListChunks) {
            const uint64_t left = len[i] - at;
            if (left == 0) {
                ++i;
                at = 0;
                continue;
            }
            const uint8_t *gpu = static_cast<const uint8_t *>(toHost ? src[i] : dst[i]) + at;
            const uint64_t skip = reinterpret_cast<uint64_t>(gpu) & (kStreamLine - 1);
            uint64_t end = kStreamChunkBytes;       // the next begins on a line
            if ((skip + left) % kStreamChunkBytes <= kStreamShortTail) {
                const uint64_t chunks = (skip + left + kStreamChunkBytes - 1) / kStreamChunkBytes;
                end = ((skip + left + chunks - 1) / chunks + kStreamLine - 1) / kStreamLine * kStreamLine;
            }
            const uint64_t take = std::min<uint64_t>(left, end - skip);
            area->list[count++] = StreamChunk{reinterpret_cast<uint64_t>(gpu), static_cast<uint32_t>(take), 0};
            memory.push_back(static_cast<const uint8_t *>(toHost ? dst[i] : src[i]) + at);
            at += take;
        }
        if (count == 0) {
            break;
        }
        Streaming job{area, toHost, total >= kPastCachesBytes, area->base.value, count, stream, memory.data()};
        area->base.value += count;
        job.Run(helper);
        XcopyEngine::Instance().NoteDone(stream, job.launches);     // waited for here or below
        if (job.error != 0 || job.stopped) {
            const int sync = job.launched == 0 ? 0 : mfrt_stream_sync(stream);
            if (sync != 0) {
                MF_FAIL(BM_ERROR, "copy failed on the GPU: " << mfrt_error_string(sync));
            }
            return kNotStreamed;
        }
    }
    return BM_OK;
}

// Pageable memory to the GPU: the CPU fills a slot while the launches of the slots before it run.  Rounds grow from
// kRoundMinBytes, so that the link does not wait for the first slot longer than it has to.
int StageIn(void *const *src, void *const *dst, const uint64_t *len, uint32_t n, void *stream)
{
    XcopyEngine &engine = XcopyEngine::Instance();
    const auto bounce = reinterpret_cast<uint64_t>(AreaOf(engine));
    if (bounce == 0) {
        MF_FAIL(BM_MALLOC_FAILED, "pinned staging allocation failed");
    }
    RoundCursor cursor(src, dst, len, n);
    const bool pastCaches = cursor.Left() >= kPastCachesBytes;
    StagedLaunches launches(stream);
    std::vector<uint64_t> a, b, l;
    std::vector<HostCopyHelper::Task> tasks;   // the CPU copies of one round
    uint64_t last = 0;   // bytes of the round before; the cores together fill a slot in half the time the link takes to empty it
    while (cursor.Left() != 0) {
        const uint32_t round = launches.Count();
        if (round >= kSlots) {
            const int ret = launches.Wait(round - kSlots);   // the slot's last reader
            if (ret != BM_OK) {
                return ret;
            }
        }
        a.clear();
        b.clear();
        l.clear();
        tasks.clear();
        const uint64_t slot = bounce + round % kSlots * kRoundBytes;
        const uint64_t before = cursor.Left();
        cursor.Next(RoundBytes(2 * last, before), [&](uint64_t from, uint64_t to, uint64_t bytes, uint64_t at) {
            tasks.push_back(HostCopyHelper::Task{reinterpret_cast<void *>(slot + at), reinterpret_cast<const void *>(from), bytes});
            a.push_back(slot + at);
            b.push_back(to);
            l.push_back(bytes);
        });
        last = before - cursor.Left();
        HostCopyHelper::Instance().CopySet(tasks.data(), tasks.size(), pastCaches);
        if (round == 0 && cursor.Left() == 0) {
            return engine.SubmitAndWait(a.data(), b.data(), l.data(), static_cast<uint32_t>(l.size()), MFRT_ROUTE_FROM_HOST, stream);
        }
        const int ret = launches.Launch(a, b, l, MFRT_ROUTE_FROM_HOST);
        if (ret != BM_OK) {
            return ret;
        }
    }
    return launches.Finish();   // the caller's memory has been consumed before; the copy itself is done as well
}

// The GPU to pageable memory: the CPU empties a slot while the launches that fill the next ones run.  Rounds shrink to
// kRoundMinBytes at the end, so that the CPU is not left with a whole slot when the link is done.
int StageOut(void *const *src, void *const *dst, const uint64_t *len, uint32_t n, void *stream)
{
    XcopyEngine &engine = XcopyEngine::Instance();
    const auto bounce = reinterpret_cast<uint64_t>(AreaOf(engine));
    if (bounce == 0) {
        MF_FAIL(BM_MALLOC_FAILED, "pinned staging allocation failed");
    }
    RoundCursor cursor(src, dst, len, n);
    const bool pastCaches = cursor.Left() >= (cursor.Left() / n >= kPastCachesLongSegment ? kPastCachesBytes : kPastCachesShortBytes);
    StagedLaunches launches(stream);
    std::vector<uint64_t> a, b, l;
    std::vector<HostCopyHelper::Task> tasks[kSlots];   // the CPU copies of the rounds in flight
    uint32_t emptied = 0;
    auto empty = [&]() -> int {
        const int ret = launches.Wait(emptied);
        if (ret == BM_OK) {
            HostCopyHelper::Instance().CopySet(tasks[emptied % kSlots].data(), tasks[emptied % kSlots].size(), pastCaches);
            ++emptied;
        }
        return ret;
    };
    while (cursor.Left() != 0) {
        const uint32_t round = launches.Count();
        a.clear();
        b.clear();
        l.clear();
        tasks[round % kSlots].clear();
        const uint64_t slot = bounce + round % kSlots * kRoundBytes;
        cursor.Next(RoundBytes(cursor.Left() / 2, cursor.Left()), [&](uint64_t from, uint64_t to, uint64_t bytes, uint64_t at) {
            tasks[round % kSlots].push_back(
                HostCopyHelper::Task{reinterpret_cast<void *>(to), reinterpret_cast<const void *>(slot + at), bytes});
            a.push_back(from);
            b.push_back(slot + at);
            l.push_back(bytes);
        });
        if (round == 0 && cursor.Left() == 0) {
            const int ret = engine.SubmitAndWait(a.data(), b.data(), l.data(), static_cast<uint32_t>(l.size()), MFRT_ROUTE_TO_HOST, stream);
            if (ret == BM_OK) {
                HostCopyHelper::Instance().CopySet(tasks[0].data(), tasks[0].size());
            }
            return ret;
        }
        int ret = launches.Launch(a, b, l, MFRT_ROUTE_TO_HOST);
        if (ret == BM_OK && round - emptied >= kAhead) {
            ret = empty();
        }
        if (ret != BM_OK) {
            return ret;
        }
    }
    while (emptied < launches.Count()) {
        const int ret = empty();
        if (ret != BM_OK) {
            return ret;
        }
    }
    return BM_OK;
}

int RouteOf(bool srcOnHost, bool dstOnHost)
{
    if (dstOnHost) {
        return MFRT_ROUTE_TO_HOST;
    }
    return srcOnHost ? MFRT_ROUTE_FROM_HOST : MFRT_ROUTE_HBM;
}

}  // namespace

HipDataOp::Result HipDataOp::Initialize() noexcept
{
    if (inited_) {
        return BM_OK;
    }
    if (!XcopyEngine::Instance().Started()) {
        MF_FAIL(BM_NOT_INITIALIZED, "GPU copy engine is not running; call hybm_init first");
    }
    inited_ = true;
    return BM_OK;
}

void HipDataOp::UnInitialize() noexcept
{
    inited_ = false;
}

HipDataOp::Result HipDataOp::Wait(int32_t) noexcept
{
    if (!inited_) {
        return BM_NOT_INITIALIZED;
    }
    return XcopyEngine::Instance().DrainThread();
}

void HipDataOp::CleanUp() noexcept
{
    (void)XcopyEngine::Instance().DrainThread();
    XcopyEngine::Instance().QuiesceSubmitters();   // batches of other threads that a submit thread has not launched yet
}

HipDataOp::Result HipDataOp::DataCopy(hybm_copy_params &params, hybm_data_copy_direction direction,
                                      const ExtOptions &options) noexcept
{
    void *src = params.src;
    void *dst = params.dest;
    uint64_t len = params.dataSize;
    return Run(&src, &dst, &len, 1, direction, options, (options.flags & ASYNC_COPY_FLAG) != 0);
}

HipDataOp::Result HipDataOp::DataCopyAsync(hybm_copy_params &params, hybm_data_copy_direction direction,
                                           const ExtOptions &options) noexcept
{
    void *src = params.src;
    void *dst = params.dest;
    uint64_t len = params.dataSize;
    return Run(&src, &dst, &len, 1, direction, options, true);
}

HipDataOp::Result HipDataOp::BatchDataCopy(hybm_batch_copy_params &params, hybm_data_copy_direction direction,
                                           const ExtOptions &options) noexcept
{
    return Run(params.sources, params.destinations, params.dataSizes, params.batchSize, direction, options,
               (options.flags & ASYNC_COPY_FLAG) != 0);
}

HipDataOp::Result HipDataOp::Run(void *const *src, void *const *dst, const uint64_t *len, uint32_t n,
                                 hybm_data_copy_direction direction, const ExtOptions &options, bool async) noexcept
{
    if (!inited_) {
        return BM_NOT_INITIALIZED;
    }
    if (!DirectionValid(direction)) {
        MF_FAIL(BM_INVALID_PARAM, "copy direction " << direction << " is not executable");
    }
    XcopyEngine &engine = XcopyEngine::Instance();
    const Endpoint se = SourceOf(direction);
    const Endpoint de = DestinationOf(direction);
    const bool srcOnHost = !se.device;
    const bool dstOnHost = !de.device;
    // Only caller-private host memory can be invisible to the GPU; pool memory is pinned by construction.
    const bool srcPageable = !se.pool && srcOnHost && AnyPageable(src, n);
    const bool dstPageable = !de.pool && dstOnHost && AnyPageable(dst, n);
    const bool unordered = async && (options.flags & MF_COPY_UNORDERED_FLAG) != 0;
    void *stream = options.stream;
    if (stream == nullptr && !(unordered && !srcPageable && !dstPageable)) {
        // (an unordered copy without a stream of the caller's leaves the choice to the engine, which may deal it to a side stream)
        stream = engine.ThreadStream();
        if (stream == nullptr) {
            MF_FAIL(BM_ERROR, "no stream available for the copy");
        }
    }

    if (!srcPageable && !dstPageable) {
        static_assert(sizeof(void *) == sizeof(uint64_t), "64-bit addresses expected");
        const auto *from = reinterpret_cast<const uint64_t *>(src);
        const auto *to = reinterpret_cast<const uint64_t *>(dst);
        const int route = RouteOf(srcOnHost, dstOnHost);
        return async ? engine.Submit(from, to, len, n, route, stream, nullptr, 0, unordered)
                     : engine.SubmitAndWait(from, to, len, n, route, stream);
    }

    // Host DRAM to host DRAM with a pageable side: both buffers are only a CPU
    // store away from each other, no accelerator is involved.
    if (srcOnHost && dstOnHost) {
        int err = mfrt_stream_sync(stream);  // keep order with copies queued earlier
        if (err != 0) {
            MF_FAIL(BM_ERROR, "stream wait failed: " << mfrt_error_string(err));
        }
        // Elements whose own source and destination overlap are moved in place; the rest is shared
        // with the helper thread, one element at a time (elements may depend on one another only
        // if the caller broke the rule that destinations overlap nothing else in the batch).
        for (uint32_t i = 0; i < n; ++i) {
            const uint64_t s = reinterpret_cast<uint64_t>(src[i]);
            const uint64_t d = reinterpret_cast<uint64_t>(dst[i]);
            if (s < d + len[i] && d < s + len[i]) {
                std::memmove(dst[i], src[i], len[i]);
            } else {
                HostCopyHelper::Instance().Copy(dst[i], src[i], len[i]);
            }
        }
        return BM_OK;
    }

    if (Streams(len, n, dstPageable, stream)) {
        const int ret = StreamAll(src, dst, len, n, dstPageable, stream);
        if (ret != kNotStreamed) {
            return ret;
        }
    }
    return srcPageable ? StageIn(src, dst, len, n, stream) : StageOut(src, dst, len, n, stream);
}

}  // namespace mf
