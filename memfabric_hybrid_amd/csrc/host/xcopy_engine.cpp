#include "xcopy_engine.h"

#include <algorithm>
#include <atomic>
#include <chrono>
#include <condition_variable>
#include <cstdlib>
#include <cstring>
#include <memory>
#include <mutex>
#include <thread>

#include "../../../include/mf_xcopy_types.h"
#include "../rt/mf_rt.h"
#include "mf_log.h"

namespace mf {
namespace {

constexpr uint32_t kSlots = 8;                // table staging slots per thread
constexpr uint32_t kGuardEvery = 4;           // one event is recorded per this many table launches
constexpr uint64_t kInlinePiece = 1ull << 30; // cut for segments the 32-bit inline length cannot hold

std::atomic<uint64_t> g_launches{0};

// One descriptor table in flight: the host fills `host`; the table kernel reads it there, or a copy
// kernel moves it to `dev` first.  The slot may be rewritten once an event recorded behind its
// kernels has fired.  Recording an event costs the stream about 3 us, as much as the launch gap
// it sits in, so one event guards kGuardEvery consecutive launches: a slot is Queued until that
// event is recorded and Guarded (by the slot that owns the event) afterwards.  A launch of pieces on the thread's
// own stream needs none: the next one there says in a pinned word, when it starts, that this one has ended, and until then
// its slot is Followed (batches of 129 to 1000 segments 0.8 to 1.1 us a launch less than with an event per four, which the stream
// executes too: 168 K and V blocks 6.5 -> 5.5 us, 200 pages of 8 KiB 5.3 -> 4.7).  On a caller's stream, which may be gone before
// there is a next one, the launch itself says in a word of the slot when every wave has read its piece (Reported), for an event of
// its own costs 2.7 us of the host (129 / 500 / 1000 ragged segments of up to 40 000 bytes 7.4 / 11.0 / 15.7 us, so 6.2 / 9.6 / 14.4).
struct StagingSlot {
    enum State : uint8_t { kFree, kQueued, kGuarded, kFollowed, kReported };
    void *host = nullptr;
    void *dev = nullptr;
    void *rest = nullptr;       // RestList of device-resident tables, in device memory
    uint64_t capacity = 0;      // of host
    uint64_t devCapacity = 0;
    void *event = nullptr;
    State state = kFree;
    StagingSlot *guard = nullptr;
    uint32_t startSeq = 0;      // of its launch, where it is Followed
    uint32_t readSeq = 0;       // of its latest launch that reports
};

// GPU resources of one calling thread: its stream, its staging slots, its bounce area.  They are
// owned by the engine, not by the thread: a thread holds a lease, and when the thread ends the
// lease goes back to the idle list without any GPU call (thread-exit destructors run when the
// runtime, or a tool hooked into it, may already have torn down its own per-thread state).  The
// next new thread takes an idle lease over; Stop() releases all of them.
struct ThreadLease {
    uint32_t ordinal = 0;           // position in creation order
    void *stream = nullptr;
    StagingSlot slots[kSlots];
    uint32_t cursor = 0;
    uint32_t queued = 0;            // slots in state kQueued; their kernels all run on queuedStream
    void *queuedStream = nullptr;
    StagingSlot *lastQueued = nullptr;
    bool adopted = false;           // taken over from a thread that ended: its queued kernels ran on streams unknown here
    uint64_t *doneWord = nullptr;   // pinned; a one-lane launch stores doneSeq there behind a blocking copy
    uint32_t doneSeq = 0;
    uint32_t startSeq = 0;          // of the latest launch of pieces on `stream` that stores it in StartedWord() when it starts
    void *doneCounter = nullptr;    // device memory, for launches that store the word themselves
    uint64_t *readWords = nullptr;  // pinned, a line for every slot,
    void *readCounters = nullptr;   // and counters in device memory, for launches that report that they have read it
    void *graphRests = nullptr;     // kSlots RestLists for the device-table calls that become nodes of a graph: not those plain calls use
    uint32_t graphCursor = 0;
    uint64_t pendingBytes = 0;      // bytes of the copies queued on `stream` since the thread last waited for it
    void *bounce = nullptr;
    uint64_t bounceBytes = 0;
    // unordered batches handed to the submit threads: fanDirty bit w = submitter w holds batches of this thread that the
    // thread's stream has not been made to wait for, the last of them under ticket fanTicket[w]
    void *fanEvent[XcopyEngine::kFanStreams] = {};
    uint64_t fanTicket[XcopyEngine::kFanStreams] = {};
    uint32_t fanDirty = 0;
    uint32_t fanCursor = 0;

    void Destroy()   // GPU calls: only from Stop(), on a thread that is alive and bound
    {
        bool busy = false;
        for (auto &slot : slots) {
            busy = busy || slot.state != StagingSlot::kFree;
        }
        if (busy) {
            (void)mfrt_device_sync();   // kernels that read the slots may run on streams of the callers
        }
        queued = 0;
        queuedStream = nullptr;
        lastQueued = nullptr;
        for (auto &slot : slots) {
            if (slot.event != nullptr) {
                (void)mfrt_event_destroy(slot.event);
            }

            if (slot.host != nullptr) {
                (void)mfrt_free_host(slot.host);
            }
            if (slot.dev != nullptr) {
                (void)mfrt_free_device(slot.dev);
            }
            if (slot.rest != nullptr) {
                (void)mfrt_free_device(slot.rest);
            }
            slot = StagingSlot{};
        }
        if (stream != nullptr) {
            (void)mfrt_stream_sync(stream);
            (void)mfrt_stream_destroy(stream);
            stream = nullptr;
        }

        if (bounce != nullptr) {
            (void)mfrt_free_host(bounce);
            bounce = nullptr;
            bounceBytes = 0;
        }
        if (doneWord != nullptr) {
            (void)mfrt_free_host(doneWord);
            doneWord = nullptr;
        }
        if (doneCounter != nullptr) {
            (void)mfrt_free_device(doneCounter);
            doneCounter = nullptr;
        }
        if (readWords != nullptr) {
            (void)mfrt_free_host(readWords);
            readWords = nullptr;
        }
        if (readCounters != nullptr) {
            (void)mfrt_free_device(readCounters);
            readCounters = nullptr;
        }
        if (graphRests != nullptr) {
            (void)mfrt_free_device(graphRests);
            graphRests = nullptr;
        }
        for (uint32_t i = 0; i < XcopyEngine::kFanStreams; ++i) {
            if (fanEvent[i] != nullptr) {
                (void)mfrt_event_destroy(fanEvent[i]);
                fanEvent[i] = nullptr;
            }
        }
        fanDirty = 0;
    }
};

// The streams of the engine, made at Start() and dealt out in an order in which consecutive takers sit on different
// hardware queues.  The runtime spreads the streams of a process over a few hardware queues (four here), not
// evenly (of the first eight streams after the thread's own, the second and third shared a queue in every process
// measured), and launches on streams that share a queue run one after the other: four submit threads whose streams
// sat on two queues measured 4.3 us per 9 MB batch, on four queues 3.6 us.  So the deck asks
// (mfrt_streams_share_queue, 50 us per pair, all streams idle) which of its streams share, and deals one stream of
// every queue before the second of any.  Streams beyond the deck are made on demand and not classified.
struct StreamDeck {
    std::mutex lock;
    std::vector<void *> order;          // untaken streams, the next one last
    std::vector<uint32_t> classes;      // hardware queue of the deck's streams in the order they are dealt, for reports

    void Build(uint32_t count)
    {
        std::lock_guard<std::mutex> guard(lock);
        DestroyLocked();
        std::vector<void *> made;
        std::vector<uint32_t> queueOf;
        std::vector<void *> firstOfQueue;
        bool known = true;
        for (uint32_t i = 0; i < count; ++i) {
            void *stream = mfrt_stream_create();
            if (stream == nullptr) {
                break;
            }
            uint32_t q = static_cast<uint32_t>(firstOfQueue.size());   // a queue of its own unless it shares one
            for (uint32_t c = 0; known && c < firstOfQueue.size(); ++c) {
                const int shared = mfrt_streams_share_queue(firstOfQueue[c], stream);
                if (shared < 0) {
                    known = false;      // no answer: from here on the streams keep the order they were made in
                    q = static_cast<uint32_t>(firstOfQueue.size());
                } else if (shared == 1) {
                    q = c;
                    break;
                }
            }
            if (q == firstOfQueue.size()) {
                firstOfQueue.push_back(stream);
            }
            made.push_back(stream);
            queueOf.push_back(q);
        }
        // round by round: the first untaken stream of every queue, queues in the order they appeared
        std::vector<bool> dealt(made.size(), false);
        std::vector<void *> sequence;
        const uint32_t queues = static_cast<uint32_t>(firstOfQueue.size());
        while (sequence.size() < made.size()) {
            for (uint32_t q = 0; q < queues; ++q) {
                for (size_t i = 0; i < made.size(); ++i) {
                    if (!dealt[i] && queueOf[i] == q) {
                        dealt[i] = true;
                        sequence.push_back(made[i]);
                        classes.push_back(q);
                        break;
                    }
                }
            }
        }
        order.assign(sequence.rbegin(), sequence.rend());
    }

    void *Take()
    {
        {
            std::lock_guard<std::mutex> guard(lock);
            if (!order.empty()) {
                void *stream = order.back();
                order.pop_back();
                return stream;
            }
        }
        return mfrt_stream_create();
    }

    void DestroyLocked()
    {
        for (void *stream : order) {
            (void)mfrt_stream_destroy(stream);
        }
        order.clear();
        classes.clear();
    }

    void Destroy()
    {
        std::lock_guard<std::mutex> guard(lock);
        DestroyLocked();
    }
};

StreamDeck &Deck()
{
    static StreamDeck *deck = new StreamDeck();   // never destroyed, as the lease pool
    return *deck;
}

std::atomic<uint32_t> g_leasesOut{0};   // leases held by live threads: more than one means launches of several streams may overlap

struct LeasePool {
    std::mutex lock;
    std::vector<std::unique_ptr<ThreadLease>> all;
    std::vector<ThreadLease *> idle;
    uint64_t epoch = 1;   // bumped by Stop(): leases handed out before are gone

    ThreadLease *Take(uint64_t &epochOut)
    {
        std::lock_guard<std::mutex> guard(lock);
        epochOut = epoch;
        if (!idle.empty()) {
            // The oldest idle lease, not the one handed back last: the runtime spreads streams over its
            // few hardware queues in creation order, and two streams on one hardware queue do not overlap
            // (two submitting threads whose streams share a queue measured 4.9 us per 9 MB batch, the same
            // as one thread; on different queues 4.1 us).  N threads alive at a time then hold the N
            // oldest streams, which sit on different queues as far as there are queues.
            size_t best = 0;
            for (size_t i = 1; i < idle.size(); ++i) {
                if (idle[i]->ordinal < idle[best]->ordinal) {
                    best = i;
                }
            }
            ThreadLease *lease = idle[best];
            idle.erase(idle.begin() + static_cast<std::ptrdiff_t>(best));
            lease->adopted = true;
            g_leasesOut.store(static_cast<uint32_t>(all.size() - idle.size()), std::memory_order_relaxed);
            return lease;
        }
        all.emplace_back(new ThreadLease());
        all.back()->ordinal = static_cast<uint32_t>(all.size() - 1);
        g_leasesOut.store(static_cast<uint32_t>(all.size() - idle.size()), std::memory_order_relaxed);
        return all.back().get();
    }
    void GiveBack(ThreadLease *lease, uint64_t leaseEpoch)
    {
        std::lock_guard<std::mutex> guard(lock);
        if (leaseEpoch == epoch) {
            idle.push_back(lease);
            g_leasesOut.store(static_cast<uint32_t>(all.size() - idle.size()), std::memory_order_relaxed);
        }
    }
    void DestroyAll()
    {
        std::lock_guard<std::mutex> guard(lock);
        for (auto &lease : all) {
            lease->Destroy();
        }
        all.clear();
        idle.clear();
        g_leasesOut.store(0, std::memory_order_relaxed);
        ++epoch;
    }
    uint64_t Epoch()
    {
        std::lock_guard<std::mutex> guard(lock);
        return epoch;
    }
};

LeasePool &Leases()
{
    static LeasePool *pool = new LeasePool();   // never destroyed: threads may end after static destructors ran
    return *pool;
}

std::atomic<uint64_t> g_leaseEpoch{1};   // copy of the pool's epoch that can be read without the lock

struct ThreadCtx {
    ThreadLease *lease = nullptr;
    uint64_t epoch = 0;
    SegList segs;
    ~ThreadCtx()
    {
        if (lease != nullptr) {
            Leases().GiveBack(lease, epoch);
            lease = nullptr;
        }
    }
    ThreadLease &Lease()
    {
        if (lease == nullptr || epoch != g_leaseEpoch.load(std::memory_order_acquire)) {
            lease = Leases().Take(epoch);
        }
        return *lease;
    }
    bool HasLiveLease() const
    {
        return lease != nullptr && epoch == g_leaseEpoch.load(std::memory_order_acquire);
    }
};

thread_local ThreadCtx t_ctx;

// Copies queued on the calling thread's own stream are added up, so that its next wait knows whether polling pays.
void NotePending(void *stream, uint64_t bytes)
{
    if (t_ctx.HasLiveLease() && stream == t_ctx.lease->stream) {
        uint64_t &pending = t_ctx.lease->pendingBytes;
        pending = pending + bytes < pending ? ~0ull : pending + bytes;
    }
}

// Submit threads.  One thread that launches on several streams in turn gains nothing (the launches cost it more
// than they cost on one stream: 4.6 to 5.1 us per 9 MB batch on two to four streams against 4.5 us), while several
// threads with a stream each do overlap on the GPU (eight threads: 3.9 us).  So a caller that declares its batches
// unordered can have them launched by up to kFanStreams threads of the library's, each with a stream of its own
// (six of them: 3.87 us per batch with the caller's thread spending 1.2 us on each): the caller plans the batch and puts the
// plan into a submitter's queue (a bounded queue of sequence-numbered cells, any number of producers, one consumer),
// the submitter launches it.  A ticket per queue tells the caller how far the submitter has got.
struct FanJob {
    InlinePlan plan;
    int route;
    uint32_t grid;
    uint32_t hold;
};

struct Submitter {
    static constexpr uint32_t kCells = 64;
    struct Cell {
        std::atomic<uint64_t> seq;
        FanJob job;
    };
    Cell cells[kCells];
    std::atomic<uint64_t> head{0};          // tickets handed to producers
    std::atomic<uint64_t> launched{0};      // jobs the thread has launched (in ticket order)
    std::atomic<int> error{0};              // first launch error, sticky until a caller has seen it
    std::atomic<bool> stop{false};
    std::atomic<bool> asleep{false};
    std::atomic<bool> ready{false};         // Run() has made its stream (or failed to)
    std::mutex lock;
    std::condition_variable wake;
    void *stream = nullptr;
    std::thread thread;

    Submitter()
    {
        for (uint32_t i = 0; i < kCells; ++i) {
            cells[i].seq.store(i, std::memory_order_relaxed);
        }
    }

    // Producer: returns the job's ticket.  Waits while the queue is full.
    uint64_t Push(const InlinePlan &plan, int route, uint32_t grid, uint32_t hold)
    {
        const uint64_t ticket = head.fetch_add(1, std::memory_order_relaxed);
        Cell &cell = cells[ticket % kCells];
        while (cell.seq.load(std::memory_order_acquire) != ticket) {
            std::this_thread::yield();      // kCells jobs ahead: the submitter is behind, or asleep and about to be woken
            Wake();
        }
        cell.job.plan = plan;
        cell.job.route = route;
        cell.job.grid = grid;
        cell.job.hold = hold;
        cell.seq.store(ticket + 1, std::memory_order_seq_cst);   // before the look at `asleep`: the submitter does both in the other order
        Wake();
        return ticket;
    }

    void Wake()
    {
        if (asleep.load(std::memory_order_seq_cst)) {
            std::lock_guard<std::mutex> guard(lock);
            wake.notify_one();
        }
    }

    void Run()
    {
        if (mfrt_bind_thread() != 0) {
            error.store(-1, std::memory_order_relaxed);
        }
        stream = Deck().Take();
        ready.store(true, std::memory_order_release);
        if (stream == nullptr) {
            return;
        }
        uint64_t next = 0;
        uint32_t idle = 0;
        while (!stop.load(std::memory_order_acquire)) {
            Cell &cell = cells[next % kCells];
            if (cell.seq.load(std::memory_order_acquire) == next + 1) {
                // a copy of its own first: the cell's lines come from the producer's core, and fetching them inside the launch
                // call would keep whatever the runtime holds locked there for as long
                const FanJob job = cell.job;
                const int err = mfk_xcopy_inline(&job.plan, job.route, job.grid, nullptr, 0, stream, 0, job.hold);
                if (err != 0) {
                    int none = 0;
                    (void)error.compare_exchange_strong(none, err, std::memory_order_relaxed);
                }
                cell.seq.store(next + kCells, std::memory_order_release);
                ++next;
                launched.store(next, std::memory_order_release);
                idle = 0;
                continue;
            }
            if (++idle < 20000) {           // some tens of microseconds of polling before the thread gives up its core
                continue;
            }
            std::unique_lock<std::mutex> guard(lock);
            asleep.store(true, std::memory_order_seq_cst);
            if (cell.seq.load(std::memory_order_seq_cst) != next + 1 && !stop.load(std::memory_order_acquire)) {
                // the bound is a net under the handshake, not part of it (by the system clock: the wait on the steady
                // clock is a call the thread sanitizer of this toolchain does not know, and it then misreads the mutex)
                wake.wait_until(guard, std::chrono::system_clock::now() + std::chrono::milliseconds(50));
            }
            asleep.store(false, std::memory_order_release);
            idle = 0;
        }
    }
};

struct SubmitPool {
    std::mutex lock;
    Submitter *submitters[XcopyEngine::kFanStreams] = {};
    std::atomic<uint32_t> alive{0};

    // Submitter w, started on first use; NULL when its stream or thread cannot be had.
    Submitter *Get(uint32_t w)
    {
        if (w < alive.load(std::memory_order_acquire)) {
            return submitters[w];
        }
        std::lock_guard<std::mutex> guard(lock);
        while (alive.load(std::memory_order_relaxed) <= w) {
            const uint32_t at = alive.load(std::memory_order_relaxed);
            Submitter *raw = new Submitter();
            raw->thread = std::thread([raw] { raw->Run(); });
            while (!raw->ready.load(std::memory_order_acquire)) {
                std::this_thread::yield();
            }
            if (raw->stream == nullptr) {
                raw->thread.join();
                delete raw;
                return nullptr;
            }
            submitters[at] = raw;
            alive.store(at + 1, std::memory_order_release);
        }
        return submitters[w];
    }

    // Submitter w if it runs.
    Submitter *Peek(uint32_t w)
    {
        return w < alive.load(std::memory_order_acquire) ? submitters[w] : nullptr;
    }

    // From Stop(): the threads end, their streams are drained and destroyed.
    void Shutdown()
    {
        std::lock_guard<std::mutex> guard(lock);
        const uint32_t count = alive.load(std::memory_order_relaxed);
        for (uint32_t w = 0; w < count; ++w) {
            Submitter *sub = submitters[w];
            sub->stop.store(true, std::memory_order_release);
            {
                std::lock_guard<std::mutex> inner(sub->lock);
                sub->wake.notify_one();
            }
            sub->thread.join();
            (void)mfrt_stream_sync(sub->stream);
            (void)mfrt_stream_destroy(sub->stream);
            delete sub;
            submitters[w] = nullptr;
        }
        alive.store(0, std::memory_order_release);
    }
};

SubmitPool &Submitters()
{
    static SubmitPool *pool = new SubmitPool();   // never destroyed: see Leases()
    return *pool;
}

// Makes `stream` (the lease's own) wait for the unordered batches the lease has handed to the submit threads: first until
// each has been launched, then, by an event on the submitter's stream, until it has run.
int JoinFan(ThreadLease &lease, void *stream)
{
    int failed = 0;
    for (uint32_t w = 0; lease.fanDirty != 0 && w < XcopyEngine::kFanStreams; ++w) {
        if ((lease.fanDirty & (1u << w)) == 0) {
            continue;
        }
        lease.fanDirty &= ~(1u << w);
        Submitter *sub = Submitters().Peek(w);
        if (sub == nullptr) {
            continue;   // stopped in the meantime: Stop() has drained it
        }
        while (sub->launched.load(std::memory_order_acquire) <= lease.fanTicket[w]) {
            sub->Wake();
            std::this_thread::yield();
        }
        const int err = sub->error.exchange(0, std::memory_order_relaxed);
        failed = failed != 0 ? failed : err;
        if (lease.fanEvent[w] == nullptr) {
            lease.fanEvent[w] = mfrt_event_create();
        }
        const bool joined = lease.fanEvent[w] != nullptr && mfrt_event_record(lease.fanEvent[w], sub->stream) == 0 &&
                            mfrt_stream_wait_event(stream, lease.fanEvent[w]) == 0;
        if (!joined) {
            const int syncErr = mfrt_stream_sync(sub->stream);
            if (syncErr != 0) {
                MF_FAIL(BM_ERROR, "unordered copies could not be awaited: " << mfrt_error_string(syncErr));
            }
        }
    }
    if (failed != 0) {
        MF_FAIL(BM_ERROR, "an unordered copy failed to launch: " << mfrt_error_string(failed));
    }
    return BM_OK;
}

uint64_t RoundUp(uint64_t v, uint64_t to)
{
    return (v + to - 1) / to * to;
}

// Records the event that guards every queued slot.  If the record fails the stream is drained instead.
int SealQueued(ThreadLease &ctx)
{
    if (ctx.queued == 0) {
        return BM_OK;
    }
    StagingSlot *owner = ctx.lastQueued;
    const bool recorded = owner != nullptr && owner->event != nullptr && mfrt_event_record(owner->event, ctx.queuedStream) == 0;
    if (!recorded && mfrt_stream_sync(ctx.queuedStream) != 0) {
        const int err = mfrt_device_sync();
        if (err != 0) {
            MF_FAIL(BM_ERROR, "staging slots could not be released: " << mfrt_error_string(err));
        }
    }
    for (auto &slot : ctx.slots) {
        if (slot.state == StagingSlot::kQueued) {
            slot.state = recorded ? StagingSlot::kGuarded : StagingSlot::kFree;
            slot.guard = recorded ? owner : nullptr;
        }
    }
    ctx.queued = 0;
    ctx.lastQueued = nullptr;
    return BM_OK;
}

// The event a launch on `stream` should complete for its slot: launches on a caller's stream are guarded one by one, since nothing
// says how long the stream lives; those on the thread's own stream several at a time, by an event recorded behind them.
void *EventOfLaunch(const ThreadLease &ctx, const StagingSlot &slot, const void *stream)
{
    return stream != ctx.stream ? slot.event : nullptr;
}

// The kernels just launched on `stream` read `slot`.  Only launches on the lease's own stream wait
// for a shared event: a caller's stream may be gone by the time the next launch comes.
int MarkQueued(ThreadLease &ctx, StagingSlot *slot, void *stream, bool sealNow, bool attached = false)
{
    if (attached) {   // its launch completes the slot's event
        slot->state = StagingSlot::kGuarded;
        slot->guard = slot;
        return BM_OK;
    }
    sealNow = sealNow || stream != ctx.stream;
    slot->state = StagingSlot::kQueued;
    slot->guard = nullptr;
    ctx.queuedStream = stream;
    ctx.lastQueued = slot;
    ++ctx.queued;
    return sealNow || ctx.queued >= kGuardEvery ? SealQueued(ctx) : BM_OK;
}

// Behind the word of the blocking copies, which the GPU stores too.
uint64_t *StartedWord(ThreadLease &lease)
{
    return lease.doneWord + 4;
}

constexpr uint32_t kReadWordStride = 8;     // 64-bit words

bool HasReadMarks(ThreadLease &lease)
{
    if (lease.readWords == nullptr) {
        lease.readWords = static_cast<uint64_t *>(mfrt_alloc_host(kSlots * kReadWordStride * sizeof(uint64_t)));
        if (lease.readWords == nullptr) {
            return false;
        }
        std::fill_n(lease.readWords, kSlots * kReadWordStride, 0);
    }
    if (lease.readCounters == nullptr) {
        lease.readCounters = mfrt_alloc_device(kSlots * kDoneCounterBytes);
        if (lease.readCounters != nullptr && mfrt_memset(lease.readCounters, 0, kSlots * kDoneCounterBytes) != 0) {
            (void)mfrt_free_device(lease.readCounters);
            lease.readCounters = nullptr;
        }
    }
    return lease.readCounters != nullptr;
}

uint64_t *ReadWord(ThreadLease &lease, const StagingSlot &slot)
{
    return lease.readWords + (&slot - lease.slots) * kReadWordStride;
}

void *ReadCounter(ThreadLease &lease, const StagingSlot &slot)
{
    return static_cast<uint8_t *>(lease.readCounters) + (&slot - lease.slots) * kDoneCounterBytes;
}

// Polls a word until it has come to `value`, for `most` at the longest; after a while the thread sleeps between looks.
bool AwaitWord(const uint64_t *word, uint32_t value, std::chrono::milliseconds most)
{
    constexpr auto kSpin = std::chrono::microseconds(100);
    constexpr auto kSleep = std::chrono::microseconds(20);
    const auto from = std::chrono::steady_clock::now();
    for (uint32_t polls = 1;; ++polls) {
        if (static_cast<int32_t>(static_cast<uint32_t>(__atomic_load_n(word, __ATOMIC_ACQUIRE)) - value) >= 0) {
            return true;
        }
        if ((polls & 63u) == 0) {
            const auto waited = std::chrono::steady_clock::now() - from;
            if (waited > most) {
                return false;
            }
            if (waited > kSpin) {
                std::this_thread::sleep_for(kSleep);
                polls |= 62u;           // two looks, then the next sleep
            }
        }
    }
}

constexpr auto kWordPatience = std::chrono::milliseconds(200);

// Waits until the kernel that reads a Followed slot has ended: until a later launch has started or, if there is none or none that
// starts, by an event.
int AwaitFollower(ThreadLease &ctx, StagingSlot &slot)
{
    if (ctx.startSeq != slot.startSeq && AwaitWord(StartedWord(ctx), slot.startSeq + 1, kWordPatience)) {
        return 0;
    }
    const int err = mfrt_event_record(slot.event, ctx.stream);
    return err != 0 ? err : mfrt_event_sync(slot.event);
}

// Waits until the kernel that reads a Reported slot says that it has read it, however much work is queued in front of it.  A GPU that
// has failed never gets there: it shows on `stream`, which the next launch goes to (the kernel's own may be gone).
int AwaitReport(ThreadLease &ctx, const StagingSlot &slot, void *stream)
{
    while (!AwaitWord(ReadWord(ctx, slot), slot.readSeq, kWordPatience)) {
        const int state = mfrt_stream_done(stream);
        if (state < 0) {
            return -state;
        }
    }
    return 0;
}

// The next slot of the ring, free to be rewritten, with at least `bytes` of pinned host memory.  Not for launches that become nodes
// of a graph: a replay would read what a later call has left in the slot, memory may not be allocated while a stream records, and
// an event recorded there is none that anybody could wait for.
int AcquireSlot(ThreadLease &ctx, uint64_t bytes, void *stream, StagingSlot *&out)
{
    if (ctx.adopted) {
        // The thread that filled these slots is gone, and with it the knowledge which streams its
        // last launches went to: wait for the whole device once.
        bool busy = false;
        for (auto &slot : ctx.slots) {
            busy = busy || slot.state != StagingSlot::kFree;
        }
        if (busy) {
            const int err = mfrt_device_sync();
            if (err != 0) {
                MF_FAIL(BM_ERROR, "device wait failed: " << mfrt_error_string(err));
            }
            for (auto &slot : ctx.slots) {
                slot.state = StagingSlot::kFree;
                slot.guard = nullptr;
            }
        }
        ctx.queued = 0;
        ctx.lastQueued = nullptr;
        ctx.adopted = false;
    }
    StagingSlot &slot = ctx.slots[ctx.cursor];
    ctx.cursor = (ctx.cursor + 1) % kSlots;
    if (ctx.queued != 0 && (slot.state == StagingSlot::kQueued || ctx.queuedStream != stream)) {
        // one event guards launches of one stream only; and a slot about to be reused needs its guard now
        const int ret = SealQueued(ctx);
        if (ret != BM_OK) {
            return ret;
        }
    }
    if (slot.state == StagingSlot::kFollowed) {
        const int err = AwaitFollower(ctx, slot);
        if (err != 0) {
            MF_FAIL(BM_ERROR, "staging slot wait failed: " << mfrt_error_string(err));
        }
        slot.state = StagingSlot::kFree;
    }
    if (slot.state == StagingSlot::kReported) {
        const int err = AwaitReport(ctx, slot, stream);
        if (err != 0) {
            MF_FAIL(BM_ERROR, "staging slot wait failed: " << mfrt_error_string(err));
        }
        slot.state = StagingSlot::kFree;
    }
    if (slot.state == StagingSlot::kGuarded) {
        StagingSlot *guard = slot.guard;
        const int err = mfrt_event_sync(guard->event);
        if (err != 0) {
            MF_FAIL(BM_ERROR, "staging slot wait failed: " << mfrt_error_string(err));
        }
        for (auto &other : ctx.slots) {   // everything that event guarded is free now
            if (other.state == StagingSlot::kGuarded && other.guard == guard) {
                other.state = StagingSlot::kFree;
                other.guard = nullptr;
            }
        }
    }
    if (slot.capacity < bytes) {
        if (slot.host != nullptr) {
            (void)mfrt_free_host(slot.host);
            slot.host = nullptr;
        }
        const uint64_t cap = RoundUp(bytes < 65536 ? 65536 : bytes, 65536);
        slot.host = mfrt_alloc_host(cap);
        if (slot.host == nullptr) {
            slot.capacity = 0;
            MF_FAIL(BM_MALLOC_FAILED, "descriptor staging allocation of " << cap << " bytes failed");
        }
        slot.capacity = cap;
    }
    if (slot.event == nullptr) {
        slot.event = mfrt_event_create();
        if (slot.event == nullptr) {
            MF_FAIL(BM_ERROR, "event creation failed");
        }
    }
    out = &slot;
    return BM_OK;
}

// Device half of a slot, for the forms that need the table or the prefix in HBM.
int EnsureDevice(StagingSlot &slot, uint64_t bytes)
{
    if (slot.devCapacity >= bytes) {
        return BM_OK;
    }
    if (slot.dev != nullptr) {
        (void)mfrt_free_device(slot.dev);
        slot.dev = nullptr;
        slot.devCapacity = 0;
    }
    const uint64_t cap = RoundUp(bytes < 65536 ? 65536 : bytes, 65536);
    slot.dev = mfrt_alloc_device(cap);
    if (slot.dev == nullptr) {
        MF_FAIL(BM_MALLOC_FAILED, "descriptor staging allocation of " << cap << " bytes in HBM failed");
    }
    slot.devCapacity = cap;
    return BM_OK;
}

uint64_t RestListStride(uint32_t capacity)
{
    return RoundUp(RestListBytes(capacity), 256);
}

int EnsureRestLists(void *&lists, uint32_t count, uint32_t capacity)
{
    if (lists != nullptr) {
        return BM_OK;
    }
    lists = mfrt_alloc_device(count * RestListStride(capacity));
    if (lists == nullptr) {
        MF_FAIL(BM_MALLOC_FAILED, "lists of " << capacity << " segments could not be allocated in HBM");
    }
    // cleared once, on a stream of the engine: the caller's may be recording
    void *own = XcopyEngine::Instance().ThreadStream();
    const int err = own == nullptr ? -1 : mfk_xcopy_clear_lists(lists, count, RestListStride(capacity), own);
    if (err != 0 || mfrt_stream_sync(own) != 0) {
        (void)mfrt_free_device(lists);
        lists = nullptr;
        MF_FAIL(BM_ERROR, "lists of segments could not be cleared: " << mfrt_error_string(err));
    }
    return BM_OK;
}

constexpr uint32_t kLinkGroups = 64;

uint32_t GridFor(uint64_t nchunk, uint32_t cuCount, int route, const XcopyTuning &tuning)
{
    // HBM routes: one workgroup per chunk unless a cap is set.  Measured on 128 MiB ... 4 GiB copies:
    // letting the hardware dispatcher hand out the chunks one by one sustains 6.0-6.2 TB/s, a
    // grid capped at 16 workgroups per CU that strides over the chunks 5.3-5.7 TB/s (its static
    // assignment leaves a tail).  Link routes: kLinkGroups for the whole chip.  They keep 256 KiB in flight, more than the link's
    // rate times its round trip, from the host; what is in flight beyond that queues in front of the link and lowers its rate.
    // Back to back, from the host 256 workgroups on 8 KiB / 64 on 4 KiB: 1 / 2 / 4 / 8 / 64 MiB 23.8 / 44.6 / 81.2 / 154.6 / 1178 us
    // against 22.6 / 41.3 / 77.9 / 151.0 / 1173; to the host, both on 4 KiB: 22.1 / 41.1 / 77.8 / 151.2 / 1179 against 20.9 / 39.7 /
    // 76.5 / 149.9 / 1178.
    const bool link = route == MFRT_ROUTE_TO_HOST || route == MFRT_ROUTE_FROM_HOST;
    const uint32_t perCu = link ? tuning.wgPerCuLink : tuning.wgPerCu;
    const uint64_t limit = (1ull << 24) - 1;   // grid size in lanes must stay below 2^32 with up to 256 lanes per workgroup
    uint64_t cap = perCu != 0 ? static_cast<uint64_t>(cuCount == 0 ? 256 : cuCount) * perCu : link ? kLinkGroups : limit;
    if (cap > limit) {
        cap = limit;
    }
    uint64_t grid = nchunk < cap ? nchunk : cap;
    return grid == 0 ? 1u : static_cast<uint32_t>(grid);
}

// Grid of the launch that copies a table only the GPU can read.  Workgroups walk the items of the table with the grid as their
// stride, surplus workgroups leave at once, at 0.4 ns each.  Four per segment between 16 and 1024 per CU: 16 080 pages of 8 KiB
// (two chunks) take 53 / 58 / 71 us with two / four / eight per segment, 4096 pages of 32 KiB (eight chunks) 49.8 / 47.1 / 48.5.
uint32_t DeviceTableGrid(uint32_t nseg, uint32_t cuCount, int route, const XcopyTuning &tuning)
{
    const uint64_t cus = cuCount == 0 ? 256 : cuCount;
    uint64_t want = 4ull * nseg;
    want = want < 16 * cus ? 16 * cus : want > 1024 * cus ? 1024 * cus : want;
    return GridFor(tuning.deviceTableWgPerCu != 0 ? cus * tuning.deviceTableWgPerCu : want, cuCount, route, tuning);
}

// Grid of the launch behind it, which usually finds nothing to do (the kernel has the figures).
uint32_t DeviceTableRestGrid(uint32_t cuCount, int route, const XcopyTuning &tuning)
{
    return GridFor(2ull * (cuCount == 0 ? 256 : cuCount), cuCount, route, tuning);
}

}  // namespace

void NormalizeSegments(const uint64_t *src, const uint64_t *dst, const uint64_t *len, uint32_t n, uint64_t pieceLimit,
                       SegList &out)
{
    out.Clear();
    uint64_t curSrc = 0;
    uint64_t curDst = 0;
    uint64_t curLen = 0;
    auto flush = [&]() {
        while (curLen > 0) {
            uint64_t piece = (pieceLimit != 0 && curLen > pieceLimit) ? pieceLimit : curLen;
            out.src.push_back(curSrc);
            out.dst.push_back(curDst);
            out.len.push_back(piece);
            out.totalBytes += piece;
            curSrc += piece;
            curDst += piece;
            curLen -= piece;
        }
    };
    for (uint32_t i = 0; i < n; ++i) {
        if (len[i] == 0) {
            continue;
        }
        if (curLen > 0 && curSrc + curLen == src[i] && curDst + curLen == dst[i]) {
            curLen += len[i];
            continue;
        }
        flush();
        curSrc = src[i];
        curDst = dst[i];
        curLen = len[i];
    }
    flush();
}

uint32_t ChooseUnits(uint64_t totalBytes, uint32_t cuCount, int route, const XcopyTuning &tuning)
{
    (void)cuCount;
    if (tuning.unitsOverride != 0) {
        return static_cast<uint32_t>(RoundUp(tuning.unitsOverride, 64));
    }
    // Measured on MI355X (256 CUs).  HBM routes: 4 KiB chunks, which the launcher gives to single-wave
    // workgroups, one workgroup per chunk: the fastest shape from a 1 MiB copy (3.4 us against 4.5 us
    // with four-wave workgroups on 16 KiB chunks) over the 9 MB KV batch (4.8 against 5.5 us) to a
    // 1 GiB copy (6.4 against 6.25 TB/s).  4 KiB also divides the usual power-of-two block sizes, so
    // no workgroup runs a ragged tile.
    if (route == MFRT_ROUTE_TO_HOST || route == MFRT_ROUTE_FROM_HOST) {
        // See GridFor for the workgroups.  From the host one access per lane for short copies (512 KiB 19.8 us, 20.6 with two), two
        // beyond (122 blocks, 9 MB: 162.9, 165.4 with one), four for the longest, which take any.
        if (totalBytes > (256ull << 20)) {
            return 4 * kXcopyThreads;
        }
        return route == MFRT_ROUTE_TO_HOST || totalBytes <= (2ull << 20) ? kXcopyThreads : 2 * kXcopyThreads;
    }
    (void)totalBytes;
    return tuning.minUnits;
}

bool BuildInlinePlan(const SegList &segs, uint32_t units, InlinePlan &plan)
{
    const uint32_t n = segs.Size();
    if (n > kInlineSegs) {
        return false;
    }
    uint64_t run = 0;
    for (uint32_t i = 0; i < n; ++i) {
        if (segs.len[i] > 0xFFFFFFFFull) {
            return false;
        }
        plan.src[i] = segs.src[i];
        plan.dst[i] = segs.dst[i];
        plan.len[i] = static_cast<uint32_t>(segs.len[i]);
        plan.first[i] = static_cast<uint32_t>(run);
        run += SegmentChunks(segs.dst[i], segs.len[i], units);
        if (run >= kNoChunk) {
            return false;
        }
    }
    for (uint32_t i = n; i < kInlineSegs; ++i) {
        plan.src[i] = 0;
        plan.dst[i] = 0;
        plan.len[i] = 0;
        plan.first[i] = kNoChunk;
    }
    plan.nchunk = static_cast<uint32_t>(run);
    plan.units = units;
    return true;
}

// Normalisation and inline planning in one pass over the caller's arrays, for the common case
// of a batch that ends up with at most kInlineSegs segments below 4 GiB each.  Returns false
// (plan contents undefined) when the batch needs the general path.
bool BuildInlineDirect(const uint64_t *src, const uint64_t *dst, const uint64_t *len, uint32_t n, uint32_t units,
                       InlinePlan &plan)
{
    const bool pow2 = (units & (units - 1)) == 0;
    const uint32_t shift = pow2 ? static_cast<uint32_t>(__builtin_ctz(units)) : 0;
    // The usual batch (blocks scattered over a pool) has nothing to merge, nothing empty and nothing of 4 GiB: one pass
    // without branches says so, and the plan is then filled by a straight-line loop (the general loop below merges as it
    // goes and tests every step).
    if (n != 0 && n <= kInlineSegs && pow2) {
        uint64_t special = (len[n - 1] == 0 ? 1u : 0u) | (len[n - 1] >> 32);
        for (uint32_t i = 0; i + 1 < n; ++i) {
            const uint64_t l = len[i];
            special |= (l == 0 ? 1u : 0u) | (l >> 32) |
                       ((src[i] + l == src[i + 1] ? 1u : 0u) & (dst[i] + l == dst[i + 1] ? 1u : 0u));
        }
        if (special == 0) {
            uint32_t run32 = 0;
            for (uint32_t i = 0; i < n; ++i) {
                const uint64_t l = len[i];
                uint64_t head = (0 - dst[i]) & (kUnitBytes - 1);
                head = head > l ? l : head;
                const uint64_t chunks = ((l - head) / kUnitBytes + units - 1) >> shift;
                plan.src[i] = src[i];
                plan.dst[i] = dst[i];
                plan.len[i] = static_cast<uint32_t>(l);
                plan.first[i] = run32;
                run32 += static_cast<uint32_t>(chunks == 0 ? 1 : chunks);      // n * 2^32 / 4096 chunks at most: no overflow
            }
            for (uint32_t i = n; i < kInlineSegs; ++i) {
                plan.src[i] = 0;
                plan.dst[i] = 0;
                plan.len[i] = 0;
                plan.first[i] = kNoChunk;
            }
            plan.nchunk = run32;
            plan.units = units;
            return run32 < kNoChunk;
        }
    }
    uint32_t used = 0;
    uint64_t run = 0;
    uint64_t curSrc = 0;
    uint64_t curDst = 0;
    uint64_t curLen = 0;
    auto flush = [&]() -> bool {
        if (curLen == 0) {
            return true;
        }
        if (used == kInlineSegs || curLen > 0xFFFFFFFFull) {
            return false;
        }
        uint64_t head = (0 - curDst) & (kUnitBytes - 1);
        if (head > curLen) {
            head = curLen;
        }
        const uint64_t body = (curLen - head) / kUnitBytes;
        uint64_t chunks = pow2 ? (body + units - 1) >> shift : (body + units - 1) / units;
        if (chunks == 0) {
            chunks = 1;
        }
        plan.src[used] = curSrc;
        plan.dst[used] = curDst;
        plan.len[used] = static_cast<uint32_t>(curLen);
        plan.first[used] = static_cast<uint32_t>(run);
        run += chunks;
        ++used;
        return true;
    };
    for (uint32_t i = 0; i < n; ++i) {
        const uint64_t l = len[i];
        if (l == 0) {
            continue;
        }
        if (curLen > 0 && curSrc + curLen == src[i] && curDst + curLen == dst[i]) {
            curLen += l;
            continue;
        }
        if (!flush()) {
            return false;
        }
        curSrc = src[i];
        curDst = dst[i];
        curLen = l;
    }
    if (!flush() || run >= kNoChunk) {
        return false;
    }
    for (uint32_t i = used; i < kInlineSegs; ++i) {
        plan.src[i] = 0;
        plan.dst[i] = 0;
        plan.len[i] = 0;
        plan.first[i] = kNoChunk;
    }
    plan.nchunk = static_cast<uint32_t>(run);
    plan.units = units;
    return true;
}

uint64_t BuildTablePlan(const SegList &segs, uint32_t units, uint64_t *triples, uint32_t *first)
{
    const uint32_t n = segs.Size();
    uint64_t run = 0;
    for (uint32_t i = 0; i < n; ++i) {
        triples[3 * i] = segs.src[i];
        triples[3 * i + 1] = segs.dst[i];
        triples[3 * i + 2] = segs.len[i];
        first[i] = static_cast<uint32_t>(run);
        run += SegmentChunks(segs.dst[i], segs.len[i], units);
    }
    first[n] = static_cast<uint32_t>(run);
    return run;
}

// Normalisation (empty segments dropped, neighbours that continue each other merged) and table
// planning in one pass over the caller's arrays, straight into the staging slot: a 4096-segment
// batch costs the host about as long as the GPU needs to copy it, so nothing is built twice.
// triples: room for 3 * n words, first: room for n + 1.  Returns the chunk count, count = segments.
uint64_t BuildTableDirect(const uint64_t *src, const uint64_t *dst, const uint64_t *len, uint32_t n, uint32_t units,
                          uint64_t *triples, uint32_t *first, uint32_t &count, ChunkPattern *pattern)
{
    const bool pow2 = (units & (units - 1)) == 0;
    const uint32_t shift = pow2 ? static_cast<uint32_t>(__builtin_ctz(units)) : 0;
    uint32_t used = 0;
    uint64_t run = 0;
    uint64_t recent[kMaxPeriod] = {};   // chunk counts of the last kMaxPeriod segments, by index modulo kMaxPeriod
    uint64_t leading[kMaxPeriod] = {};  // and of the first ones
    uint32_t alive = 0x1FEu;            // bit p: the counts so far repeat with period p (1 .. kMaxPeriod)
    uint64_t curSrc = 0;
    uint64_t curDst = 0;
    uint64_t curLen = 0;
    auto flush = [&]() {
        if (curLen == 0) {
            return;
        }
        uint64_t head = (0 - curDst) & (kUnitBytes - 1);
        if (head > curLen) {
            head = curLen;
        }
        const uint64_t body = (curLen - head) / kUnitBytes;
        uint64_t chunks = pow2 ? (body + units - 1) >> shift : (body + units - 1) / units;
        if (chunks == 0) {
            chunks = 1;
        }
        triples[3 * used] = curSrc;
        triples[3 * used + 1] = curDst;
        triples[3 * used + 2] = curLen;
        first[used] = static_cast<uint32_t>(run < kNoChunk ? run : kNoChunk);
        if (alive != 0) {
            for (uint32_t p = 1; p <= kMaxPeriod; ++p) {
                if (used >= p && recent[(used - p) % kMaxPeriod] != chunks) {
                    alive &= ~(1u << p);
                }
            }
            recent[used % kMaxPeriod] = chunks;
            if (used < kMaxPeriod) {
                leading[used] = chunks;
            }
        }
        run += chunks;
        ++used;
    };
    for (uint32_t i = 0; i < n; ++i) {
        const uint64_t l = len[i];
        if (l == 0) {
            continue;
        }
        if (curLen > 0 && curSrc + curLen == src[i] && curDst + curLen == dst[i]) {
            curLen += l;
            continue;
        }
        flush();
        curSrc = src[i];
        curDst = dst[i];
        curLen = l;
    }
    flush();
    first[used] = static_cast<uint32_t>(run < kNoChunk ? run : kNoChunk);
    count = used;
    if (pattern != nullptr) {
        *pattern = ChunkPattern{};
        if (used != 0 && alive != 0 && run < kNoChunk) {
            const uint32_t period = static_cast<uint32_t>(__builtin_ctz(alive));
            uint32_t sum = 0;
            for (uint32_t i = 0; i < period; ++i) {
                pattern->start[i] = sum;
                sum += static_cast<uint32_t>(leading[i]);   // the shortest period never exceeds the segment count
            }
            pattern->start[period] = sum;
            pattern->period = period;
            pattern->chunksPerPeriod = sum;
        }
    }
    return run;
}

// The pieces of a batch (xcopy_plan.h), empty segments dropped and neighbours that continue each other merged, straight into the
// staging slot.  `out` has room for PieceBound() of them; returns their number.
uint32_t BuildPieces(const uint64_t *src, const uint64_t *dst, const uint64_t *len, uint32_t n, uint32_t units, Piece *out)
{
    const uint64_t most = static_cast<uint64_t>(units) * kUnitBytes;
    const uint32_t shift = static_cast<uint32_t>(__builtin_ctzll(most));
    Piece *p = out;
    uint64_t lastSpan = 0;
    uint64_t each = 0;
    for (uint32_t i = 0; i < n;) {
        const uint64_t s = src[i];
        const uint64_t d = dst[i];
        uint64_t l = len[i];
        ++i;
        if (l == 0) {
            continue;
        }
        for (; i < n && (len[i] == 0 || (s + l == src[i] && d + l == dst[i])); ++i) {
            l += len[i];
        }
        // pieces of equal length between multiples of kPieceAlign, counted from the one at or below the first byte
        const uint64_t skip = d & (kPieceAlign - 1);
        const uint64_t span = skip + l;
        if (span <= most) {
            *p++ = MakePiece(s, d, static_cast<uint32_t>(l));
            continue;
        }
        if (span != lastSpan) {     // a division a segment of another size
            lastSpan = span;
            const uint64_t parts = (span + most - 1) >> shift;
            const uint64_t lines = (span + kPieceAlign - 1) / kPieceAlign;
            each = kPieceAlign * (lines >> 31 == 0 ? (static_cast<uint32_t>(lines) + static_cast<uint32_t>(parts) - 1) / static_cast<uint32_t>(parts)
                                                   : (lines + parts - 1) / parts);
        }
        *p++ = MakePiece(s, d, static_cast<uint32_t>(each - skip));
        const Piece length = MakePiece(0, 0, static_cast<uint32_t>(each));
        uint64_t left = l - (each - skip);
        uint64_t from = (s + (each - skip)) & kPieceAddress;
        uint64_t to = (d + (each - skip)) & kPieceAddress;
        for (; left > each; left -= each) {
            *p++ = Piece{from | length.src, to | length.dst};
            from += each;
            to += each;
        }
        *p++ = MakePiece(from, to, static_cast<uint32_t>(left));
    }
    return static_cast<uint32_t>(p - out);
}

uint64_t PieceBound(uint64_t bytes, uint32_t n, uint32_t units)
{
    return n + (bytes + static_cast<uint64_t>(n) * (kPieceAlign - 1)) / (static_cast<uint64_t>(units) * kUnitBytes);
}

void ChooseCalibration(const float *batchMicros, const float *copyMicros, uint32_t defaultWindowMBps, uint32_t defaultAlignedMBps,
                       uint32_t defaultLongMBps, XcopyCalibration &out)
{
    out = XcopyCalibration{};
    out.windowMBps = defaultWindowMBps;
    out.windowAlignedMBps = defaultAlignedMBps;
    out.windowLongMBps = defaultLongMBps;
    for (int i = 0; i < 4; ++i) {
        out.batchMicros[i] = batchMicros[i];
    }
    for (int i = 0; i < 4; ++i) {
        out.copyMicros[i] = copyMicros[i];
    }
    const bool batchMeasured = batchMicros[0] > 0 && batchMicros[1] > 0 && batchMicros[2] > 0 && batchMicros[3] > 0;
    if (batchMeasured) {
        // the rule's own wait unless a neighbour is clearly better (2 %: less is noise between rounds and between boxes)
        int best = 2;
        for (int v : {1, 3}) {
            if (batchMicros[v] < batchMicros[best] * 0.98f) {
                best = v;
            }
        }
        out.holdDeltaNanos = (best - 2) * kCalibrateHoldStepNanos;
        out.holdEnabled = batchMicros[best] <= batchMicros[0] * (1.0f - kCalibrateMinGain);
        out.ran = true;
    }
    const bool copyMeasured = copyMicros[0] > 0 && copyMicros[1] > 0 && copyMicros[2] > 0;
    if (copyMeasured) {
        const bool slowerWins = copyMicros[2] < copyMicros[1] * 0.99f;
        const float windowed = slowerWins ? copyMicros[2] : copyMicros[1];
        const uint32_t rate = slowerWins ? static_cast<uint32_t>(static_cast<uint64_t>(defaultWindowMBps) * kCalibrateSlowerWindowPercent / 100)
                                         : defaultWindowMBps;
        out.windowMBps = windowed <= copyMicros[0] * (1.0f - kCalibrateMinWindowGain) ? rate : 0u;
        // the higher rate of aligned segments only where an aligned copy held it here: 2 % better than the rate just chosen
        // (the rate between the two, for shorter segments on cache lines, goes with it: a GPU that holds the highest holds that one)
        const bool higherHolds = out.windowMBps != 0 && copyMicros[3] > 0 && copyMicros[3] < windowed * 0.98f;
        out.windowLongMBps = higherHolds ? defaultLongMBps : out.windowMBps;
        out.windowAlignedMBps = higherHolds ? defaultAlignedMBps : out.windowMBps;
        out.ran = true;
    }
}

int XcopyEngine::Calibrate()
{
    if (!Started()) {
        return BM_NOT_INITIALIZED;
    }
    void *stream = ThreadStream();
    if (stream == nullptr) {
        return BM_ERROR;
    }
    const uint32_t rule = HoldNanosFor(2196, 2196, kXcopyThreads, false);
    const uint32_t holds[3] = {rule - kCalibrateHoldStepNanos, rule, rule + kCalibrateHoldStepNanos};
    const uint32_t defaultRate = XcopyTuning{}.windowMBps;
    const uint32_t defaultLong = XcopyTuning{}.windowLongMBps;
    const uint32_t rates[3] = {defaultRate, static_cast<uint32_t>(static_cast<uint64_t>(defaultRate) * kCalibrateSlowerWindowPercent / 100), defaultLong};
    float us[8] = {};
    const int err = mfk_xcopy_calibrate(stream, holds, rates, us);
    if (err != 0) {
        calibration_ = XcopyCalibration{};
        MF_ERROR("calibration run failed (" << mfrt_error_string(err) << "): the fitted defaults stay");
        return BM_ERROR;
    }
    ChooseCalibration(us, us + 4, defaultRate, XcopyTuning{}.windowAlignedMBps, defaultLong, calibration_);
    if (calibration_.ran) {
        tuning_.holdDeltaNanos = calibration_.holdDeltaNanos;
        tuning_.holdCalibratedOff = !calibration_.holdEnabled;
        if (windowsAvailable_) {
            tuning_.windowMBps = calibration_.windowMBps;
            tuning_.windowAlignedMBps = calibration_.windowAlignedMBps;
            tuning_.windowLongMBps = calibration_.windowLongMBps;
            windowRateCalibrated_ = true;
        }
    }
    return BM_OK;
}

XcopyEngine &XcopyEngine::Instance()
{
    static XcopyEngine engine;
    return engine;
}

int XcopyEngine::Start(int device)
{
    int err = mfrt_init(device);
    if (err != 0) {
        MF_FAIL(BM_ERROR, "GPU runtime start on device " << device << " failed: " << mfrt_error_string(err));
    }
#ifndef MF_RT_HIDDEN
    err = mfk_xcopy_static_setup();   // the device is current on this thread: mfrt_init has just selected it
    if (err != 0) {
        // only the entry point that allocates nothing needs it, and that one reports the missing set-up itself
        MF_ERROR("address of the static descriptor scratch not available: " << mfrt_error_string(err));
    }
#endif
    windowsAvailable_ = mfk_xcopy_windows_available() != 0;
    Deck().Build(kDeckStreams);   // before the first stream is handed out: the calling thread's own is the deck's first
    tuning_.holdDeltaNanos = 0;
    tuning_.holdCalibratedOff = false;
    if (windowRateCalibrated_) {   // what an earlier start of this process chose does not outlive it
        tuning_.windowMBps = XcopyTuning{}.windowMBps;
        tuning_.windowAlignedMBps = XcopyTuning{}.windowAlignedMBps;
        tuning_.windowLongMBps = XcopyTuning{}.windowLongMBps;
        windowRateCalibrated_ = false;
    }
    calibration_ = XcopyCalibration{};
    started_.store(true, std::memory_order_release);
    {
        // every copy kernel once, then the timing rules checked against this GPU
        void *stream = ThreadStream();
        if (stream == nullptr || mfk_xcopy_prelaunch(stream) != 0) {
            MF_ERROR("the copy kernels could not be launched once at start");
        }
        const char *env = std::getenv("MF_HIP_CALIBRATE");
        if (stream != nullptr && !(env != nullptr && env[0] == '0')) {
            (void)Calibrate();
        }
        if (stream != nullptr) {
            (void)mfrt_stream_sync(stream);
        }
    }
    started_.store(true, std::memory_order_release);
    return BM_OK;
}

void XcopyEngine::Stop()
{
    if (!started_.load(std::memory_order_acquire)) {
        return;
    }
    (void)mfrt_bind_thread();
    Submitters().Shutdown();
    (void)mfrt_device_sync();
    Leases().DestroyAll();   // every thread's stream and staging memory, not only the caller's
    Deck().Destroy();
    g_leaseEpoch.store(Leases().Epoch(), std::memory_order_release);
    started_.store(false, std::memory_order_release);
    mfrt_shutdown();
}

uint32_t XcopyEngine::StreamQueues(uint32_t *queues, uint32_t capacity) const
{
    StreamDeck &deck = Deck();
    std::lock_guard<std::mutex> guard(deck.lock);
    const uint32_t count = static_cast<uint32_t>(deck.classes.size());
    for (uint32_t i = 0; i < count && i < capacity; ++i) {
        queues[i] = deck.classes[i];
    }
    return count;
}

bool XcopyEngine::Started() const
{
    return started_.load(std::memory_order_acquire);
}

void *XcopyEngine::ThreadStream()
{
    ThreadLease &lease = t_ctx.Lease();
    if (lease.stream == nullptr) {
        if (mfrt_bind_thread() != 0) {
            return nullptr;
        }
        lease.stream = Deck().Take();
    }
    if (lease.fanDirty != 0 && lease.stream != nullptr && JoinFan(lease, lease.stream) != BM_OK) {
        return nullptr;
    }
    return lease.stream;
}

void *XcopyEngine::ThreadBounce(uint64_t bytes, bool *fresh)
{
    ThreadLease &lease = t_ctx.Lease();
    if (lease.bounceBytes < bytes) {
        if (mfrt_bind_thread() != 0) {
            return nullptr;
        }
        if (lease.bounce != nullptr) {
            (void)mfrt_free_host(lease.bounce);
            lease.bounce = nullptr;
            lease.bounceBytes = 0;
        }
        lease.bounce = mfrt_alloc_host(bytes);
        lease.bounceBytes = lease.bounce != nullptr ? bytes : 0;
        if (fresh != nullptr) {
            *fresh = true;
        }
    }
    return lease.bounce;
}

int XcopyEngine::DrainThread()
{
    if (!Started()) {
        return BM_NOT_INITIALIZED;
    }
    if (!t_ctx.HasLiveLease() || t_ctx.lease->stream == nullptr) {
        return BM_OK;
    }
    // a short queue is awaited like a blocking call: by polling (20 KV batches and a wait: 3 us sooner than the stream wait)
    return WaitStream(t_ctx.lease->stream, t_ctx.lease->pendingBytes);
}

namespace {

bool HasDoneWord(ThreadLease &lease)
{
    if (lease.doneWord == nullptr) {
        lease.doneWord = static_cast<uint64_t *>(mfrt_alloc_host(64));
        if (lease.doneWord != nullptr) {
            *lease.doneWord = 0;
            lease.doneSeq = 0;
            *StartedWord(lease) = lease.startSeq;
        }
    }
    return lease.doneWord != nullptr;
}

bool HasDoneCounter(ThreadLease &lease)
{
    if (lease.doneCounter == nullptr) {
        lease.doneCounter = mfrt_alloc_device(kDoneCounterBytes);
        if (lease.doneCounter != nullptr && mfrt_memset(lease.doneCounter, 0, kDoneCounterBytes) != 0) {
            (void)mfrt_free_device(lease.doneCounter);
            lease.doneCounter = nullptr;
        }
    }
    return lease.doneCounter != nullptr;
}

uint32_t NextDoneSeq(ThreadLease &lease)
{
    return ++lease.doneSeq == 0 ? ++lease.doneSeq : lease.doneSeq;   // 0 is the initial contents
}

// What the route needs at the least for `bytes`: a link route 58 GB/s, HBM 7.4 TB/s of reads and writes.
uint64_t LeastMicros(uint64_t bytes, int route)
{
    return route == MFRT_ROUTE_HBM ? bytes / 3700000u : bytes / 58000u;
}

// Polls the lease's word until it has come to `seq`, for at most kSpinMicros more than `least`; false when that takes longer
// than expected (or the GPU is busy with other work).  A thread with a millisecond and more ahead of it sleeps for most of it.
bool PollDone(const ThreadLease &lease, uint32_t seq, uint64_t least)
{
    const auto start = std::chrono::steady_clock::now();
    if (least > 1000) {
        std::this_thread::sleep_for(std::chrono::microseconds(least * 9 / 10 - 100));   // a sleep may last 50 us longer
    }
    const auto most = std::chrono::microseconds(least + XcopyEngine::kSpinMicros);
    for (uint32_t polls = 1;; ++polls) {
        const auto seen = static_cast<uint32_t>(__atomic_load_n(lease.doneWord, __ATOMIC_ACQUIRE));
        if (static_cast<int32_t>(seen - seq) >= 0) {
            return true;
        }
        if ((polls & 63u) == 0 && std::chrono::steady_clock::now() - start > most) {
            return false;
        }
    }
}

}  // namespace

int XcopyEngine::LaunchDone(const uint64_t *src, const uint64_t *dst, const uint64_t *len, uint32_t n, uint64_t bytes, int route,
                            void *stream, uint32_t &ticket)
{
    // To the host a copy has few workgroups whatever its size, and each costs the launch one atomic at its end.  In HBM they are worth
    // it (a launch less for the host, a launch boundary less for the GPU) up to the bytes that held stores gain more with:
    // 2 / 4 / 8 MiB 11.4 / 11.5 / 11.9 us with a signal launch, 9.5 / 9.6 / 10.8 so, 16 MiB 13.9 / 14.6; K and V blocks of 1.8 / 3.7 MB 11.5 /
    // 12.0 and 10.3 / 10.8, of 8 MB 12.1 and 12.8.  From the host written-through stores cost more than the
    // launch they save beyond kDoneFromHostBytes (1 MiB 33.1 us, 30.2 with a signal launch; 256 KiB 14.2 either way).
    constexpr uint64_t kDoneSingleBytes = 8ull << 20;
    constexpr uint64_t kDoneFromHostBytes = 128ull << 10;
    const uint64_t most = route == MFRT_ROUTE_TO_HOST ? ~0ull
                          : route != MFRT_ROUTE_HBM   ? kDoneFromHostBytes
                          : n == 1                    ? kDoneSingleBytes
                                                      : kDonePiecesBytes;
    InlinePlan plan;
    if (n > kInlineSegs || bytes == 0 || bytes > most || tuning_.unitsOverride != 0 || !Started() || mfrt_bind_thread() != 0 ||
        !BuildInlineDirect(src, dst, len, n, kDeepUnits, plan)) {
        return kNotLaunched;
    }
    ThreadLease &lease = t_ctx.Lease();
    if (!HasDoneWord(lease) || !HasDoneCounter(lease)) {
        return kNotLaunched;
    }
    ticket = NextDoneSeq(lease);
    const uint32_t grid = GridFor(plan.nchunk, mfrt_cu_count(), route, tuning_);
    const int err = mfk_xcopy_done(&plan, route, grid, lease.doneWord, ticket, lease.doneCounter, stream);
    if (err != 0) {
        MF_FAIL(BM_ERROR, "xcopy launch failed: " << mfrt_error_string(err));
    }
    g_launches.fetch_add(1, std::memory_order_relaxed);
    NotePending(stream, bytes);
    return BM_OK;
}

// A batch of pieces that reports its own end.  Its slot is free again when it has, so no event guards it.
int XcopyEngine::LaunchPiecesDone(const uint64_t *src, const uint64_t *dst, const uint64_t *len, uint32_t n, uint64_t bytes, int route,
                                  void *stream, uint32_t &ticket)
{
    const uint64_t bound = PieceBound(bytes, n, kXcopyThreads);
    if (route != MFRT_ROUTE_HBM || bytes == 0 || bytes > kDonePiecesBytes || n > kDonePiecesSegments || tuning_.unitsOverride != 0 || !Started() ||
        mfrt_bind_thread() != 0 || mfrt_stream_capturing(stream) != 0) {
        return kNotLaunched;
    }
    ThreadLease &lease = t_ctx.Lease();
    StagingSlot *slot = nullptr;
    if (lease.fanDirty != 0 || !HasDoneWord(lease) || !HasDoneCounter(lease) || AcquireSlot(lease, bound * sizeof(Piece), stream, slot) != BM_OK) {
        return kNotLaunched;
    }
    const uint32_t count = BuildPieces(src, dst, len, n, kXcopyThreads, static_cast<Piece *>(slot->host));
    ticket = NextDoneSeq(lease);
    const int err = mfk_xcopy_pieces_done(slot->host, count, lease.doneWord, ticket, lease.doneCounter, stream);
    if (err != 0) {
        MF_FAIL(BM_ERROR, "xcopy launch failed: " << mfrt_error_string(err));
    }
    g_launches.fetch_add(1, std::memory_order_relaxed);
    NotePending(stream, bytes);
    return BM_OK;
}

int XcopyEngine::SubmitTicket(const uint64_t *src, const uint64_t *dst, const uint64_t *len, uint32_t n, int route, void *stream,
                              uint32_t &ticket)
{
    uint64_t bytes = 0;
    for (uint32_t i = 0; i < n; ++i) {
        bytes += len[i];
    }
    int ret = LaunchDone(src, dst, len, n, bytes, route, stream, ticket);
    if (ret != kNotLaunched) {
        return ret;
    }
    ret = Submit(src, dst, len, n, route, stream, nullptr, 0);
    if (ret != BM_OK) {
        return ret;
    }
    ThreadLease &lease = t_ctx.Lease();
    if (!HasDoneWord(lease)) {
        MF_FAIL(BM_MALLOC_FAILED, "the thread's pinned word could not be allocated");
    }
    ticket = NextDoneSeq(lease);
    const int err = mfk_xcopy_signal(lease.doneWord, ticket, stream);
    if (err != 0) {
        MF_FAIL(BM_ERROR, "signal launch failed: " << mfrt_error_string(err));
    }
    return BM_OK;
}

int XcopyEngine::WaitTicket(uint32_t ticket, void *stream)
{
    ThreadLease &lease = t_ctx.Lease();
    const uint64_t queued = stream == lease.stream ? lease.pendingBytes : 0;
    const int err = PollDone(lease, ticket, 4 * kSpinMicros) ? 0 : mfrt_stream_sync(stream);
    if (err != 0) {
        MF_FAIL(BM_ERROR, "copy failed on the GPU: " << mfrt_error_string(err));
    }
    if (ticket == lease.doneSeq && queued != 0) {
        lease.pendingBytes = 0;     // the thread's latest: nothing else is queued on its stream
    }
    return BM_OK;
}

int XcopyEngine::SubmitAndWait(const uint64_t *src, const uint64_t *dst, const uint64_t *len, uint32_t n, int route, void *stream)
{
    uint64_t bytes = 0;
    for (uint32_t i = 0; i < n; ++i) {
        bytes += len[i];
    }
    uint32_t ticket = 0;
    int ret = n <= kInlineSegs ? LaunchDone(src, dst, len, n, bytes, route, stream, ticket)
                               : LaunchPiecesDone(src, dst, len, n, bytes, route, stream, ticket);
    if (ret == kNotLaunched) {
        ret = SubmitInSlices(src, dst, len, n, bytes, route, stream);
        return ret != BM_OK ? ret : WaitStream(stream, bytes, route);
    }
    if (ret != BM_OK) {
        return ret;
    }
    ThreadLease &lease = t_ctx.Lease();
    if (stream == lease.stream) {
        lease.pendingBytes = 0;
    }
    const int err = PollDone(lease, ticket, LeastMicros(bytes, route)) ? 0 : mfrt_stream_sync(stream);
    if (err != 0) {
        MF_FAIL(BM_ERROR, "copy failed on the GPU: " << mfrt_error_string(err));
    }
    return BM_OK;
}

// The GPU of a caller that waits has nothing to do while the host plans, so a long batch whose planning takes a while goes in two or
// three launches, the first of them a quarter or an eighth of it: the GPU then needs longer for each than the host for the next.
// Not below kDeepMaxBytes: a launch more costs the host 3 us, and short launches leave the GPU idle at their ends (2000 ragged segments
// of up to 40 000 bytes, 40 MB, 48 us in one launch and 59 in four).
int XcopyEngine::SubmitInSlices(const uint64_t *src, const uint64_t *dst, const uint64_t *len, uint32_t n, uint64_t bytes, int route,
                                void *stream)
{
    const uint64_t planNanos = 3ull * n + bytes / 16384;        // segments, and pieces of 16 KiB
    const bool sliced = route == MFRT_ROUTE_HBM && n > 4 * kInlineSegs && planNanos >= kSliceMinNanos && bytes >= kDeepMaxBytes &&
                        tuning_.unitsOverride == 0 && bytes / n < kWindowSliceMinAlignedSegmentBytes;
    const bool three = bytes >= 3 * kDeepMaxBytes;
    const uint32_t ends[3] = {sliced ? (three ? n / 8 : n / 4) : 0, sliced && three ? n / 8 * 3 : 0, n};
    uint32_t at = 0;
    for (uint32_t end : ends) {
        if (end <= at && end != n) {
            continue;
        }
        const int ret = Submit(src + at, dst + at, len + at, end - at, route, stream, nullptr, 0, false);
        if (ret != BM_OK) {
            if (at != 0) {
                (void)mfrt_stream_sync(stream);     // what has gone out is not left running behind a call that failed
            }
            return ret;
        }
        at = end;
    }
    return BM_OK;
}

// A blocking call is a launch and a wait.  hipStreamSynchronize first has to put a marker with a
// completion signal behind the kernel and then takes 7 us to see it fire, whatever the wait policy
// of the device (measured: 16.1 us per blocking 9 MB batch with the default policy and with
// hipDeviceScheduleSpin alike; an event recorded behind the launch and polled or waited for:
// 15.5 us; hipStreamWriteValue64 polled: 13.1 us; the kernel launched with a stop event of its own
// and that event polled: 13.3 us).  A one-lane launch that stores a sequence number
// into pinned memory, polled by the caller, is the shortest way round: 11.8 us.  It starts after
// the copy kernel has ended, so it carries the same guarantee as the stream wait: the copy's
// end-of-kernel release has made its stores visible to the device, and stores to host memory were
// issued, in order, before the word's.
int XcopyEngine::WaitStream(void *stream, uint64_t bytes, int route)
{
    if (t_ctx.HasLiveLease() && stream == t_ctx.lease->stream) {
        const uint64_t queued = t_ctx.lease->pendingBytes;
        bytes = queued > bytes ? queued : bytes;     // what else the thread has queued there is waited for as well
        t_ctx.lease->pendingBytes = 0;
        if (t_ctx.lease->fanDirty != 0) {            // and the unordered batches on its side streams
            const int ret = JoinFan(*t_ctx.lease, stream);
            if (ret != BM_OK) {
                return ret;
            }
        }
    }
    if (bytes != 0 && bytes <= kSpinBytes) {
        ThreadLease &lease = t_ctx.Lease();
        if (HasDoneWord(lease)) {
            const uint32_t seq = NextDoneSeq(lease);
            // (the signal is not counted by LaunchCount(): it moves no data)
            if (mfk_xcopy_signal(lease.doneWord, seq, stream) == 0 && PollDone(lease, seq, LeastMicros(bytes, route))) {
                return BM_OK;
            }
        }
    }
    const int err = mfrt_stream_sync(stream);
    if (err != 0) {
        MF_FAIL(BM_ERROR, "copy failed on the GPU: " << mfrt_error_string(err));
    }
    return BM_OK;
}

void XcopyEngine::NoteQueued(void *stream, uint64_t bytes)
{
    NotePending(stream, bytes);
}

void XcopyEngine::NoteDone(void *stream, uint32_t launches)
{
    g_launches.fetch_add(launches, std::memory_order_relaxed);
    if (t_ctx.HasLiveLease() && stream == t_ctx.lease->stream) {
        t_ctx.lease->pendingBytes = 0;
    }
}

void XcopyEngine::QuiesceSubmitters()
{
    for (uint32_t w = 0; w < kFanStreams; ++w) {
        Submitter *sub = Submitters().Peek(w);
        if (sub == nullptr) {
            break;
        }
        const uint64_t handed = sub->head.load(std::memory_order_acquire);
        while (sub->launched.load(std::memory_order_acquire) < handed) {
            sub->Wake();
            std::this_thread::yield();
        }
    }
}

uint64_t XcopyEngine::LaunchCount() const
{
    return g_launches.load();
}

// How long the waves of a launch keep their data before they store (0: not at all): the tuning knob over
// HoldNanosFor's rule, for HBM routes and ordered launches only.
uint32_t XcopyEngine::HoldFor(const InlinePlan &plan, uint32_t grid, int route, bool unordered) const
{
    if (route != MFRT_ROUTE_HBM || unordered || tuning_.holdNanos == 0) {
        return 0;
    }
    // With launches of another thread's stream on the chip at the same time not every wave of a large launch is
    // resident at once, and the wait costs instead of gaining (two submitting threads, 24 MiB copies: 8.2 us per
    // copy without, 9.0 us with; 21 MB batches 7.9 / 8.2 us; 16 MB and below: the same or better with the wait).
    if ((plan.nchunk > kHoldSharedMaxChunks || plan.units == kDeepUnits) && g_leasesOut.load(std::memory_order_relaxed) > 1) {
        return 0;
    }
    const uint32_t rule = HoldNanosFor(plan.nchunk, grid, plan.units, plan.first[1] == kNoChunk);
    if (rule == 0 || tuning_.holdNanos > 0) {
        return rule != 0 ? static_cast<uint32_t>(tuning_.holdNanos) : 0;
    }
    if (tuning_.holdCalibratedOff) {
        return 0;
    }
    const int64_t with = static_cast<int64_t>(rule) + tuning_.holdDeltaNanos;
    return with > 0 ? static_cast<uint32_t>(with) : 0;
}

// Pieces of 16 KiB that a segment of a batch is cut into, at the most; `over` is DeepOver() of its addresses.
static uint64_t DeepOver(uint64_t addressBits)
{
    return static_cast<uint64_t>(kDeepUnits) * kUnitBytes - 1 + ((addressBits & (kPieceAlign - 1)) == 0 ? 0 : kPieceAlign - 1);
}
static uint64_t DeepPiecesOf(uint64_t bytes, uint64_t over)
{
    return (bytes + over) / (static_cast<uint64_t>(kDeepUnits) * kUnitBytes);
}

static bool OnLines(const BatchStats &stats)
{
    return (stats.addressBits & (kWindowAlignBytes - 1)) == 0;
}

// Mean length from which a list of unequal segments may go in several held launches.
constexpr uint64_t kHeldLaunchBytes = static_cast<uint64_t>(kDeepUnits) * kUnitBytes / 4 * 7;
// Mean length of segments at odd addresses from which neither several held launches nor windows were faster.
constexpr uint64_t kHeldOddBytes = static_cast<uint64_t>(kDeepUnits) * kUnitBytes * 24;

BatchStats StatsOf(const uint64_t *src, const uint64_t *dst, const uint64_t *len, uint32_t n)
{
    constexpr uint64_t kDeepBytes = static_cast<uint64_t>(kDeepUnits) * kUnitBytes;
    BatchStats st;
    for (uint32_t i = 0; i < n; ++i) {
        st.total += len[i];
        st.longest = len[i] > st.longest ? len[i] : st.longest;
        st.addressBits |= src[i] | dst[i];
        st.lengthBits |= len[i];
    }
    // A second pass costs the host 0.2 to 0.4 ns a segment (4096 pages of 8 KiB 14.5 us with it, 12.6; 12 441 segments of which half are up to 2000 bytes 42.2
    // and 39.8): only where the count decides, which is not where even the most pieces there can be are held, nor where there are
    // more segments than that, too short for several launches (HeldLaunches).
    const uint64_t over = DeepOver(st.addressBits);
    const uint64_t most = n + (st.total + n * (over - (kDeepBytes - 1))) / kDeepBytes;
    if (st.longest + kPieceAlign <= kDeepBytes) {
        st.deepPieces = n;
    } else if (st.total == st.longest * n) {
        st.deepPieces = n * DeepPiecesOf(st.longest, over);
    } else if (most <= kHeldMaxPieces || (n > kHeldMaxPieces && st.total < n * kHeldLaunchBytes)) {
        st.deepPieces = most;
    } else {
        for (uint32_t i = 0; i < n; ++i) {
            st.deepPieces += DeepPiecesOf(len[i], over);
        }
    }
    return st;
}

bool InOrder(const uint64_t *at, const uint64_t *len, uint32_t n, uint64_t gap)
{
    const uint32_t seen = n < 256 ? n : 256;
    uint32_t following = 0;
    for (uint32_t i = 1; i < seen; ++i) {
        following += at[i] - (at[i - 1] + len[i - 1]) <= gap ? 1 : 0;
    }
    return following >= seen / 2;
}

// Hold of a launch of pieces, as that of a table of as many chunks whose waves fetch their descriptors across the host link and
// issue their loads that much later than those of a launch whose descriptors are kernel arguments; of a batch of up to
// kDeepMinBytes, of its chunks of 4 KiB, whatever its pieces.  (The launcher takes off what pieces wait less, PieceLessNanos, so a
// wait set by hand, which is meant as it is, gets that on top.)
uint32_t XcopyEngine::HoldForPieces(const BatchStats &stats, uint32_t n, uint32_t count, uint32_t units, bool unordered) const
{
    if (unordered || tuning_.holdNanos == 0) {
        return 0;
    }
    if ((count > kHoldSharedMaxChunks || units != kXcopyThreads) && g_leasesOut.load(std::memory_order_relaxed) > 1) {
        return 0;
    }
    const bool byChunks = stats.total <= kDeepMinBytes && units != kXcopyThreads && count <= (units == kDeepUnits ? kHeldMaxPieces : kDeepMaxChunks);
    constexpr uint64_t kChunkBytes = static_cast<uint64_t>(kXcopyThreads) * kUnitBytes;
    const uint64_t allChunks = (stats.total + kChunkBytes - 1) / kChunkBytes + (stats.lengthBits % kChunkBytes != 0 ? n / 2 : 0);
    const uint32_t chunks = static_cast<uint32_t>(std::min<uint64_t>(allChunks, kHoldMaxChunks));
    // pieces of 8 KiB, two waves of four loads per lane, wait as those of 16 KiB for the same bytes
    const bool deep = units == kDeepUnits && !byChunks;
    const uint32_t rule = byChunks ? HoldNanosFor(chunks, chunks, kXcopyThreads, false)
                          : deep ? (count >= kHoldMinChunks / 4 && count <= kHeldMaxPieces ? DeepRuleNanos(count) : 0)
                          : units != kDeepUnits / 2 ? HoldNanosFor(count, count, units, false)
                          : count <= kDeepMaxChunks ? HoldNanosFor(count / 2, count / 2, kDeepUnits, false)
                                                    : 0;
    if (rule == 0) {
        return 0;
    }
    if (tuning_.holdNanos > 0) {
        return static_cast<uint32_t>(tuning_.holdNanos) + PieceLessNanos(count, stats.total, units);
    }
    if (tuning_.holdCalibratedOff) {
        return 0;
    }
    const int32_t whole = !deep ? 0 : static_cast<int32_t>(PieceWholeNanos(count, stats.total));
    const int32_t extra = tuning_.holdPinnedExtraNanos + (!byChunks && units != kXcopyThreads ? kHoldPinnedDeepExtraNanos : 0) +
                          (count <= n ? whole : (stats.addressBits & (kUnitBytes - 1)) != 0 ? whole / 2 : 0);
    const int64_t with = static_cast<int64_t>(rule) + extra + tuning_.holdDeltaNanos;
    return with > 0 ? static_cast<uint32_t>(with) : 0;
}

// Units of the pieces of a batch.  Waves that are resident together hold their stores, and from kPieceLongMinBytes on the longer
// pieces are the better shape for that (see there) as long as the chip holds the batch: kHeldMaxPieces waves of 16 KiB, or two of 4 KiB
// for each of up to 4096 segments of 6 to 8 KiB (4000 pages of 8 KiB 11.6 to 12.4 us, 13.8 to 15.4 without hold, 11.9
// to 12.5 in waves of 16 KiB; 4000 of 5120 bytes 10.0, 10.4 and 8.6; 5500 of 8 KiB 17.9 to 19.8 without hold, 15.5 to 17.5 so).  Beyond, what the
// usual segment fills: each workgroup twice the size halves the descriptors the host writes and the link carries, but lanes
// without a unit cost (16 080 pages of 8 KiB 45.2 / 46.1 / 47.0 us with one, two and four waves; 4096 of 32 KiB 45.8 / 46.8 / 46.4).
// Threads with streams of their own hold nothing but 4 KiB pieces (HoldFor).
uint32_t XcopyEngine::PieceUnits(const BatchStats &stats, uint32_t n, bool unordered) const
{
    const uint64_t mean = stats.total / n;
    const bool holds = !unordered && tuning_.holdNanos != 0 && tuning_.deepHold && g_leasesOut.load(std::memory_order_relaxed) <= 1;
    if (holds && stats.total > kPieceLongMinBytes && stats.longest > kXcopyThreads * kUnitBytes && stats.deepPieces <= kHeldMaxPieces) {
        const bool twoWaves = mean > 6144 && stats.longest <= kDeepUnits / 2 * kUnitBytes && stats.deepPieces <= kDeepMaxChunks;
        return twoWaves ? kDeepUnits / 2 : kDeepUnits;
    }
    if (stats.total <= kDeepMinBytes) {
        return kXcopyThreads;
    }
    return mean <= 6144 ? kXcopyThreads : mean <= 12288 ? kDeepUnits / 2 : kDeepUnits;
}

// Rates of lists in windows of 6144 waves, in 68ths of the general rate, which is 6.8 TB/s: what holds by where the segments lie and how full their pieces
// of 16 KiB are.  A rate is one or two steps below the one at which the list falls apart, so that a process whose memory lies badly keeps it too; one that does
// not hold costs 8 to 12 %, a step 1.7 %.  us back to back, the mean of four to seven processes on two machines:
//
//                                              at   59     60     61     62     63     64     66     68    rate
//   written one behind the other
//     5000 of 64 KiB, at multiples of it         116.4  118.8  112.5  110.8  109.1  107.6  104.5  102.2   68
//     5000 of 64 KiB                             116.3  120.1  112.5  110.8  109.1  107.5  104.7  102.4   66
//     4096 of 32 KiB                              49.5   48.7   48.0   47.3   46.7   46.0   44.9   44.4   66
//     4500 of 32 896 bytes                        55.0   54.2   53.5   52.8   52.3   51.5   50.2   50.7   66 (one process at 68: 53.0)
//     9000 of 16 KiB                              54.7   53.8   53.0   52.4   51.6   51.0   49.8   50.1   66 (52.6)
//     3000 of 64 to 128 KiB                      105.9  104.2  102.6  101.0   99.6   98.4   96.3   94.2   66
//   elsewhere
//     12 000 of 64 KiB, at multiples of it       274.1  273.6  265.0  260.7  256.9  254.0  250.2  246.0   66
//     7000 of 64 KiB                             161.5  159.1  157.5  155.4  153.9  152.5  164.3  171.6   63
//     6000 of 110 720 bytes                      233.1  231.3  231.4  225.6  224.3  221.6  224.3  257.6   63 (one at 66: 233.7)
//     4000 of 73 728 bytes                       106.2  104.9  103.6  102.3  102.4  107.3  114.9  116.5   60
//     2500 of 90 to 200 KiB                      137.6  128.7  126.7  125.2  123.8  124.6  124.6  134.8   60
//     4308 of 68 KiB                             108.3  106.9  105.5  104.0  106.8  114.9  119.2  120.3   60
//     16 384 of 32 KiB                           192.9  199.1  209.4  212.8  213.6  214.2  214.8  215.7   59
//     16 384 of 16 KiB                           100.2  104.0  105.7  106.6  107.0  107.4  107.8  108.4   59
//     8000 of 24 576 bytes                        73.2   73.0   77.2   80.4   81.4   81.4   81.5   81.6   59
//     8000 of 24 064 bytes                        71.6   71.5   75.0   78.2   79.6   79.9   80.0   80.0   59
//     6000 of 33 280 bytes                        73.8   73.2   75.1   78.8   80.9   81.6   81.8   82.0   59
//   read one behind the other, a read part of 30/64 of the period
//     16 384 of 32 KiB                           189.8  201.8  200.2  184.0  182.8  192.5  202.0  204.7   62
//     16 384 of 16 KiB                            97.2   98.7   98.7   93.9   93.6   97.4  100.2  101.4   62
//     8000 of 28 032 bytes                        81.9   80.8   79.7   78.6   77.8   78.5   85.4   87.4   62 (with even parts 80.7 at best)
//     9000 of 14 080 bytes                        48.1   47.6   46.8   46.3   45.5   45.2   47.0   50.0   62 (46.9)
//
// Short segments that are read in order are written more slowly than they are read, hence their longer write part; it does nothing for the others.
// Segments of one length that fill their pieces less than 75 % go in windows only where they would take three held launches (2500 of 33 333 bytes in two
// 31.8, in windows 32.1; of 20 000 bytes, 61 % full, nothing is better than none).
// At addresses off the lines, segments of several lengths in places without an order: 58 and, less than 85 % full, 57.  us back to back, before / at
//                                      before   54     56     57     58     60     62
//     8192 of up to 70 000 bytes        117.2  114.3  112.0  108.0  110.7  117.2  118.9    (79 % full; 57 on another machine)
//     8192 of up to 100 000             166.3  160.8  156.5     -   154.4  156.1  164.6
//     8192 of up to 131 072             215.3  208.8  204.1     -   201.9  200.3  214.5    (195.3 on the other)
//     8192 of up to 50 000               85.8   85.5   86.9     -    84.4   86.1   86.7    (73 %: left as it was)
//     4000 of up to 70 000 (2 held)      53.3   56.6   55.3     -    53.7   53.7   55.9
//     4000 of up to 131 072 (3 held)     98.5  102.5   99.6     -    98.5   94.7   92.9
// so only those that are not held.  Written in order they are the quicker without windows up to gaps of some 64 KiB, in which a launch still finds rows of HBM open; read in
// order only without a gap.  us without / in windows, 8700 of up to 70 000 bytes, 290 MB, gaps of 1 to 4096 / 20 000 / 60 000 / 200 000: written in order 107 / 114, 110 / 114, 114 / 114,
// 119 / 115, read too 100 / 114, 105 / 114, 114 / 114, 117 / 115, read alone 116 / 115, 118 / 114, 120 / 115, 123 / 115; 6700 of up to 131 072, 420 MB, 153 / 160, 155 / 159,
// 159 / 160, 166 / 160, read too 143 / 159, 148 / 159, 151 / 159, 160 / 162, read alone 167 / 161, 170 / 160, 171 / 162, 173 / 161.
uint32_t XcopyEngine::PieceWindowRate(const BatchStats &stats, const uint64_t *src, const uint64_t *dst, const uint64_t *len, uint32_t n, uint32_t count, uint32_t units,
                                      bool unordered, uint32_t &reading) const
{
    constexpr uint64_t kLessFullBytes = 24000;
    constexpr uint32_t kShortReading = 30;
    constexpr uint64_t kOddPercent = 75;
    constexpr uint64_t kOddGapBytes = 64ull << 10;
    if (unordered || units != kDeepUnits || !WindowsApply(stats.total, MFRT_ROUTE_HBM, kPieceWindowMinBytes)) {
        return 0;
    }
    const uint32_t rate = tuning_.windowMBps / 68;
    const uint64_t mean = stats.total / n;
    const uint64_t percent = stats.total * 100 / (static_cast<uint64_t>(count) * (kDeepUnits * kUnitBytes));
    const bool equal = stats.total == stats.longest * n;
    const bool onGrid = equal && ((stats.addressBits | stats.lengthBits) & (kWindowLongBlockBytes - 1)) == 0;
    const bool longBlocks = mean >= kWindowLongBlockBytes;
    if (!OnLines(stats)) {
        const bool holds = !equal && mean < kHeldOddBytes && count > 2 * kHeldMaxPieces && percent >= kOddPercent;
        return holds && !InOrder(dst, len, n, kOddGapBytes) && !InOrder(src, len, n) ? rate * (percent >= 85 ? 58 : 57) : 0;
    }
    if (InOrder(dst, len, n)) {
        return onGrid ? rate * 68 : equal || (longBlocks && percent >= 85) ? rate * 66 : 0;
    }
    if (onGrid) {
        return rate * 66;
    }
    if (percent < 85 && !(equal && (percent >= 75 || (mean >= kLessFullBytes && count > 2 * kHeldMaxPieces)))) {
        return 0;
    }
    if (longBlocks) {
        return rate * (percent >= 95 ? 63 : 60);
    }
    if (percent >= 85 && InOrder(src, len, n)) {
        reading = kShortReading;
        return rate * 62;
    }
    return rate * 59;
}

// In how many launches, each of as many pieces as are held, a list of more goes out; 1 where one that holds nothing is as fast.  Back to back,
// us in one launch / so: pages of 32 KiB gathered 121 / 138 / 213 MB 43.4 / 41.8, 49.1 / 47.3, 75.7 / 74.2 (but 311 MB 110.2 / 110.5 and 360 MB
// 125.7 / 127.8); segments of 50 000 bytes at random places 130 / 150 MB 53.3 / 48.9, 61.1 / 56.1, of 24 000 132 / 168 MB 54.3 / 50.2, 69.0 / 63.8, of
// 33 333, 68 % full, 153 MB 62.8 / 57.7, of 20 000, 61 %, 122 / 180 MB 50.8 / 52.5, 74.3 / 79.8; ragged ones at odd addresses of up to 63 000 / 100 000 /
// 120 000 / 200 000 bytes 49.7 / 47.5, 62.2 / 58.5, 73.6 / 69.2, 148 / 145, of up to 45 000 58.0 / 62.9: the host writes those no faster than the GPU
// copies them, and the second launch is 4 us of its time.  The ratio over 125 to 450 MB in two to four launches, lengths of one size and ragged ones of 30 000 to
// 900 000 bytes: at random places 0.92 to 0.99, at odd addresses from 640 000 bytes on 0.98 to 1.02; read in order 0.93 to 1.00, at odd addresses from
// 400 000 on 0.98 to 1.06; written in order, where the one launch finds the rows of HBM open, in two launches of nearly full pieces 0.94 to 1.00, of others 1.00
// to 1.04, in three or four 1.00 to 1.07, at odd addresses from 400 000 bytes on 1.00 to 1.08.
// Every launch has a slot of its own, so half of them are left for other calls.
uint32_t XcopyEngine::HeldLaunches(const BatchStats &stats, const uint64_t *src, const uint64_t *dst, const uint64_t *len, uint32_t n, bool unordered) const
{
    constexpr uint64_t kDeepBytes = static_cast<uint64_t>(kDeepUnits) * kUnitBytes;
    if (unordered || tuning_.unitsOverride != 0 || !tuning_.deepHold || stats.deepPieces <= kHeldMaxPieces ||
        stats.deepPieces > kSlots / 2 * kHeldMaxPieces || stats.total < stats.deepPieces * kDeepBytes / 100 * 65) {
        return 1;
    }
    const uint64_t mean = stats.total / n;
    const bool equal = stats.total == stats.longest * n;
    if (mean < (equal ? kDeepBytes : kHeldLaunchBytes) || mean >= kWindowSliceMinAlignedSegmentBytes) {
        return 1;
    }
    // A launch ends with a segment, so a share that surely fits is less than a launch holds by what that one may exceed it.
    const uint64_t over = DeepOver(stats.addressBits);
    const uint64_t longest = DeepPiecesOf(stats.longest, over);
    if (longest > kHeldMaxPieces / 4) {
        return 1;
    }
    const uint32_t pieces = static_cast<uint32_t>(stats.deepPieces);
    const uint32_t room = static_cast<uint32_t>(equal ? kHeldMaxPieces / longest * longest : kHeldMaxPieces + 1 - longest);
    const uint32_t fewest = (pieces + kHeldMaxPieces - 1) / kHeldMaxPieces;
    uint32_t parts = (pieces + room - 1) / room;
    if (parts != fewest) {
        const uint64_t share = (pieces + fewest - 1) / fewest;
        uint64_t taken = 0;
        uint64_t most = 0;
        for (uint32_t i = 0; i < n; ++i) {
            taken = (taken < share || len[i] == 0 ? taken : 0) + DeepPiecesOf(len[i], over);
            most = std::max(most, taken);
        }
        parts = most <= kHeldMaxPieces ? fewest : parts;
    }
    uint32_t reading = 0;
    const bool odd = (stats.addressBits & (kUnitBytes - 1)) != 0;
    const bool refused = InOrder(dst, len, n) ? parts > 2 || stats.total < stats.deepPieces * kDeepBytes / 100 * 92
                                                      : parts > 2 && odd && mean < 3 * kDeepBytes;
    if (parts > kSlots / 2 || refused || (odd && mean >= kHeldOddBytes) ||
        (OnLines(stats) && PieceWindowRate(stats, src, dst, len, n, pieces, kDeepUnits, false, reading) != 0) || HoldForPieces(stats, n, pieces / parts, kDeepUnits, false) == 0) {
        return 1;
    }
    return parts;
}

// The same number of pieces to each of them, up to a segment.  (What the whole list's lengths and addresses rule out for none of its
// segments holds for each part.)
int XcopyEngine::SubmitHeld(const uint64_t *src, const uint64_t *dst, const uint64_t *len, uint32_t n, const BatchStats &stats, uint32_t parts,
                            void *stream, void *mask, uint32_t maskValue)
{
    const uint64_t share = (stats.deepPieces + parts - 1) / parts;
    const uint64_t over = DeepOver(stats.addressBits);
    const uint64_t longest = DeepPiecesOf(stats.longest, over);
    const bool equal = stats.total == stats.longest * n;
    for (uint32_t at = 0; at < n;) {
        uint64_t bytes = 0;
        uint64_t pieces = 0;
        uint32_t end = at;
        if (equal) {
            end = static_cast<uint32_t>(std::min<uint64_t>(n, at + (share + longest - 1) / longest));
            bytes = (end - at) * stats.longest;
            pieces = (end - at) * longest;
        }
        while (end < n && (pieces < share || len[end] == 0)) {
            bytes += len[end];
            pieces += DeepPiecesOf(len[end++], over);
        }
        BatchStats part = stats;
        part.total = bytes;
        part.deepPieces = pieces;
        const int ret = SubmitPieces(src + at, dst + at, len + at, end - at, part, kDeepUnits, stream, end == n ? mask : nullptr, maskValue, false);
        if (ret != BM_OK) {
            return ret;
        }
        at = end;
    }
    return BM_OK;
}

// A wave has its descriptor after two loads from HBM (kTableHoldNanos), and then waits as one of a launch of pieces does.
void XcopyEngine::TablePaceFor(uint32_t &holdNanos, uint32_t &holdMoreNanos, uint32_t &windowMBps) const
{
    const bool alone = g_leasesOut.load(std::memory_order_relaxed) <= 1;
    const bool rule = tuning_.holdNanos < 0 && !tuning_.holdCalibratedOff;
    const int32_t base = tuning_.holdNanos > 0 ? tuning_.holdNanos : kTableHoldNanos + tuning_.holdDeltaNanos;
    holdNanos = alone && tuning_.deepHold && (rule || tuning_.holdNanos > 0) && base > 0 ? static_cast<uint32_t>(base) : 0;
    holdMoreNanos = holdNanos != 0 && rule ? kTableHoldMoreNanos : 0;
    windowMBps = WindowsApply(kDeepMaxBytes, MFRT_ROUTE_HBM, kDeepMaxBytes) ? tuning_.windowMBps / 17 * 15 : 0;
}

bool XcopyEngine::DeepHoldApplies(uint64_t bytes, uint32_t n, int route, bool unordered) const
{
    return route == MFRT_ROUTE_HBM && !unordered && tuning_.holdNanos != 0 && tuning_.unitsOverride == 0 && tuning_.deepHold &&
           bytes > kDeepMinBytes && n != 0 && bytes <= (n == 1 && !tuning_.holdCalibratedOff ? kHeldSingleBytes : kDeepMaxBytes) && bytes / n >= kDeepMinSegmentBytes &&
           g_leasesOut.load(std::memory_order_relaxed) <= 1;
}

bool XcopyEngine::WindowsApply(uint64_t bytes, int route, uint64_t minBytes) const
{
    // Two such launches at a time would each cut their periods for the whole chip's rate, so a second thread with a
    // stream of its own switches the form off, as it does for the largest held launches.
    return route == MFRT_ROUTE_HBM && bytes >= minBytes && tuning_.windowMBps != 0 && tuning_.unitsOverride == 0 &&
           windowsAvailable_ && g_leasesOut.load(std::memory_order_relaxed) <= 1;
}

bool XcopyEngine::SingleSubmitter() const
{
    return g_leasesOut.load(std::memory_order_relaxed) <= 1;
}

int XcopyEngine::Submit(const uint64_t *src, const uint64_t *dst, const uint64_t *len, uint32_t n, int route,
                        void *stream, void *mask, uint32_t maskValue, bool unordered)
{
    return SubmitOne(src, dst, len, n, route, stream, mask, maskValue, unordered, true);
}

// A batch of up to kInlineSegs segments that moves twice kWindowPieceBytes and more, submitted as consecutive runs of
// kWindowPieceBytes to twice that, one windowed launch each.  Runs end at segment ends where the segments are short and
// inside a segment, at a multiple of 1 MiB from its start, where one is long.
int XcopyEngine::SubmitInPieces(const uint64_t *src, const uint64_t *dst, const uint64_t *len, uint32_t n, uint64_t total, int route,
                                void *stream, void *mask, uint32_t maskValue)
{
    const uint64_t pieces = total / kWindowPieceBytes;
    const uint64_t target = (total + pieces - 1) / pieces;
    constexpr uint64_t kCutUnit = 1ull << 20;
    std::vector<uint64_t> ps;
    std::vector<uint64_t> pd;
    std::vector<uint64_t> pl;
    uint64_t inPiece = 0;
    uint64_t left = total;
    auto flush = [&](bool last) -> int {
        if (ps.empty()) {
            return BM_OK;
        }
        const int ret = SubmitOne(ps.data(), pd.data(), pl.data(), static_cast<uint32_t>(ps.size()), route, stream, last ? mask : nullptr,
                                  maskValue, false, false);
        ps.clear();
        pd.clear();
        pl.clear();
        inPiece = 0;
        return ret;
    };
    for (uint32_t i = 0; i < n; ++i) {
        uint64_t at = 0;
        while (at < len[i]) {
            uint64_t take = len[i] - at;
            const uint64_t room = target > inPiece ? target - inPiece : 0;
            // what is left behind this piece must still make a launch of its own, else it stays with this one
            if (take > room && left - room >= kWindowPieceBytes) {
                const uint64_t cut = room / kCutUnit * kCutUnit;
                if (take >= 16 * kCutUnit && cut != 0 && take - cut >= kCutUnit) {
                    take = cut;
                } else if (inPiece != 0 && room < take / 2) {
                    const int ret = flush(false);      // the segment starts the next piece whole
                    if (ret != BM_OK) {
                        return ret;
                    }
                    continue;
                }
            }
            ps.push_back(src[i] + at);
            pd.push_back(dst[i] + at);
            pl.push_back(take);
            at += take;
            inPiece += take;
            left -= take;
            if (inPiece >= target && left >= kWindowPieceBytes) {
                const int ret = flush(false);
                if (ret != BM_OK) {
                    return ret;
                }
            }
        }
    }
    return flush(true);
}

// maySlice: a table of long segments may be cut into launches of kInlineSegs segments; a slice is submitted
// with false, so that one that cannot take the kernel-argument form (a segment of 4 GiB and more is cut into
// pieces, which can carry it past kInlineSegs rows) goes to the table form instead of being sliced again.
int XcopyEngine::SubmitOne(const uint64_t *src, const uint64_t *dst, const uint64_t *len, uint32_t n, int route,
                           void *stream, void *mask, uint32_t maskValue, bool unordered, bool maySlice)
{
    if (!Started()) {
        MF_FAIL(BM_NOT_INITIALIZED, "xcopy engine not started");
    }
    if (mfrt_bind_thread() != 0) {
        MF_FAIL(BM_ERROR, "cannot make the GPU current on this thread");
    }
    ThreadCtx &ctx = t_ctx;
    const uint32_t cu = mfrt_cu_count();
    InlinePlan plan;
    if (stream == nullptr) {
        // An unordered batch that can travel in the kernel arguments is handed to one of the submit threads in turn, where
        // the caller asked for them: launched there in order on the submitter's stream, beside whatever the others launch.
        const uint32_t fanCount = tuning_.unorderedStreams < kFanStreams ? tuning_.unorderedStreams : kFanStreams;
        if (unordered && fanCount >= 2 && n <= kInlineSegs && mask == nullptr && route == MFRT_ROUTE_HBM) {
            uint64_t total = 0;
            for (uint32_t i = 0; i < n; ++i) {
                total += len[i];
            }
            const uint32_t fanUnits = ChooseUnits(total, cu, route, tuning_);
            if (total <= kFanMaxBytes && BuildInlineDirect(src, dst, len, n, fanUnits, plan)) {
                ThreadLease &lease = ctx.Lease();
                if (lease.stream == nullptr && ThreadStream() == nullptr) {
                    MF_FAIL(BM_ERROR, "cannot create the thread's stream");
                }
                const uint32_t w = lease.fanCursor % fanCount;
                Submitter *sub = Submitters().Get(w);
                if (sub != nullptr) {
                    lease.fanCursor = w + 1;
                    if (plan.nchunk != 0) {
                        const uint32_t grid = GridFor(plan.nchunk, cu, route, tuning_);
                        const uint32_t hold = tuning_.holdOnSideStreams ? HoldFor(plan, grid, route, false) : 0;
                        lease.fanTicket[w] = sub->Push(plan, route, grid, hold);
                        lease.fanDirty |= 1u << w;
                        g_launches.fetch_add(1, std::memory_order_relaxed);
                        NotePending(lease.stream, total);   // the thread's next wait covers the submitters' streams
                    }
                    return BM_OK;
                }
            }
        }
        stream = ThreadStream();
        if (stream == nullptr) {
            MF_FAIL(BM_ERROR, "cannot create the thread's stream");
        }
    }
    bool inlined = false;
    uint32_t units = 0;
    bool oversized = false;      // a run the 32-bit length of the inline table cannot hold is possible
    bool windowed = false;
    uint32_t windowRate = tuning_.windowMBps;
    uint64_t queuedBytes = 0;
    if (n <= 4 * kInlineSegs) {  // small enough that a failed attempt costs next to nothing
        uint64_t total = 0;
        uint64_t addressBits = 0;      // low bits any source or destination address has set
        uint64_t apartBits = 0;        // low bits in which a source differs from its destination
        for (uint32_t i = 0; i < n; ++i) {
            total += len[i];
            addressBits |= src[i] | dst[i];
            apartBits |= src[i] ^ dst[i];
        }
        queuedBytes = total;
        oversized = total > 0xFFFFFFFFull;
        units = ChooseUnits(total, cu, route, tuning_);
        // Large HBM copies of one submitter: 16 KiB chunks for the kernel that alternates between read and write windows, from where
        // held stores end (XcopyWindowKernel has the figures).
        const bool aligned = (addressBits & (kWindowAlignBytes - 1)) == 0;
        const bool apart = (apartBits & (kUnitBytes - 1)) != 0;
        windowed = !unordered && WindowsApply(total, route, kDeepMaxBytes + 1) && !DeepHoldApplies(total, n, route, unordered);
        // Segments whose sources and destinations agree modulo 16 hold a higher rate, as their chunks are cut on the destinations' lines; long
        // ones that all start on cache lines, in source and destination, the highest, and shifted ones a little more than the general one.
        // Back to back, us, at 7.2 / 7.3 / 7.4 / 7.5 TB/s: one segment of 370 MB 110.0 / 108.8 / 107.9 / 107.0, 900 MB 269 / 266 / 264 / 262 (512 MiB
        // at 7.5 151 to 155, at 7.6 158 to 162); 128 x 9 MB 355 / 348 / 348 / 350, 128 x 2.4 MB 91.9 / 92.1 / 91.8 / 101.9; the column-parallel part of 28
        // layers with its rectangles 3986 / 3955 / 3952 / 3958; off a line 300 MB 89.0 / 87.7 / 87.1 / 86.1, 900 MB 271 / 269 / 262 / 262.  Shifted, at
        // 6.8 / 7.0 / 7.2 / 7.3: 200 MB 63.4 / 62.1 / 61.0 / 61.2, 900 MB 282 / 278 / 276 / 281, 100 of 2 MB on average 35.4 / 35.2 / 36.2 / 36.8, of 4 MB
        // 131 / 129 / 135 / 144.
        const bool longSegments = windowed && total / n >= kWindowLongSegmentBytes;
        if (longSegments && maySlice && total >= 2 * kWindowPieceBytes) {
            // A windowed launch that loses its schedule runs the rest of its bytes at the rate without windows, and the longer
            // it runs the likelier that is: launches of kWindowPieceBytes to twice that, each with a schedule of its own, hold
            // a target the whole copy in one launch does not (2 GiB at 7.4 TB/s on 4096 waves: 7.1 TB/s on average in four launches,
            // 6.6 to 6.8 in one).  Only long segments are worth it: 896 segments of some 10 MB in launches of 64 or 96
            // segments (600 to 900 MB) were no faster than in launches of 128.
            return SubmitInPieces(src, dst, len, n, total, route, stream, mask, maskValue);
        }
        if (aligned && longSegments && tuning_.windowLongMBps != 0) {
            windowRate = tuning_.windowLongMBps;
        } else if (tuning_.windowAlignedMBps != 0) {
            windowRate = apart ? std::min(tuning_.windowMBps / 34 * 35, tuning_.windowAlignedMBps) : tuning_.windowAlignedMBps;
        }
        if (windowed) {
            units = mfk_xcopy_window_units();
        }
        const bool deep = !windowed && DeepHoldApplies(total, n, route, unordered);
        if (deep && n != 1 && (apartBits & (kUnitBytes - 1)) != 0 && mfrt_stream_capturing(stream) == 0) {
            // as pieces: sixteen loads per lane of aligned units and what shifts them, with the table of the kernel arguments, take
            // more registers than sixteen waves per CU have (42 MB 17.5 us with straddling loads); one segment has no table
            const int ret = SubmitPieces(src, dst, len, n, StatsOf(src, dst, len, n), kDeepUnits, stream, mask, maskValue, unordered);
            if (ret != kNotLaunched) {
                return ret;
            }
        }
        inlined = BuildInlineDirect(src, dst, len, n, deep ? kDeepUnits : units, plan);
        if (inlined && deep && HoldNanosFor(plan.nchunk, plan.nchunk, kDeepUnits, plan.first[1] == kNoChunk) == 0) {
            inlined = BuildInlineDirect(src, dst, len, n, units, plan);   // ragged enough to exceed the waves that hold: the usual chunks
        }
    }
    if (!inlined && oversized) {
        // a run of 4 GiB and more may have made the one-pass attempt give up: the general inline path cuts it into pieces
        NormalizeSegments(src, dst, len, n, kInlinePiece, ctx.segs);
        units = windowed ? mfk_xcopy_window_units() : ChooseUnits(ctx.segs.totalBytes, cu, route, tuning_);
        inlined = BuildInlinePlan(ctx.segs, units, plan);
    }
    if (inlined && windowed) {
        const int err = mfk_xcopy_windowed(&plan, windowRate, mask, maskValue, stream);
        if (err != 0) {
            MF_FAIL(BM_ERROR, "xcopy launch failed: " << mfrt_error_string(err));
        }
        g_launches.fetch_add(1, std::memory_order_relaxed);
        NotePending(stream, queuedBytes);
        return BM_OK;
    }
    if (inlined) {
        const uint32_t grid = GridFor(plan.nchunk, cu, route, tuning_);
        // a completion word is stored by a launch of its own behind the copy, which an unordered copy would not hold back
        int err = mfk_xcopy_inline(&plan, route, grid, mask, maskValue, stream, unordered && mask == nullptr ? 1 : 0,
                                   HoldFor(plan, grid, route, unordered));
        if (err != 0) {
            MF_FAIL(BM_ERROR, "xcopy launch failed: " << mfrt_error_string(err));
        }
        g_launches.fetch_add(1, std::memory_order_relaxed);
        NotePending(stream, queuedBytes);
        return BM_OK;
    }

    // Beyond the kernel arguments descriptors are built in a pinned slot, which is sized for n segments; merging can only make
    // them fewer.  A graph has no use for a slot.
    if (mfrt_stream_capturing(stream) != 0) {
        return SubmitRecorded(src, dst, len, n, route, stream, mask, maskValue);
    }
    {
        const BatchStats stats = StatsOf(src, dst, len, n);
        const uint64_t total = stats.total;
        queuedBytes = total;
        // A table of long segments between HBM addresses is cut into launches of kInlineSegs segments, each of which
        // then takes the form with read and write windows: the few extra launches cost microseconds, the windows
        // gain 8 % (896 segments, 8.5 GB: 2.55 ms in seven launches against 2.78 ms in one).  Segments on cache lines
        // are worth it from 1 MiB each, 128 MiB a launch (1024 x 1 MiB 327 against 361 us, 1024 x 2 MiB 658 against
        // 753 to 772 us, 512 x 3 MiB 458 against 588 us; 1024 x 512 KiB, 64 MiB a launch, the same either way).  Tables
        // themselves were measured under windows three times, with a search of the whole prefix, with the division and
        // group map, and with full periods at rates from 6.0 to 7.1 TB/s, and are left without them: 262 144
        // pages of 32 KiB at random places lose 7 to 12 % (3.23 to 3.45 against 3.04 ms; the third time 2.93 to 3.38
        // against 2.89 to 3.06), 4096 pages take 58 to 60 instead of 46.5 to 49 us, 16 384 ragged segments lose 3 %, and
        // the 896 long segments in one windowed table launch are no faster than in seven launches of the kernel-argument form.
        if (maySlice && n > kInlineSegs && route == MFRT_ROUTE_HBM && !unordered && tuning_.windowMBps != 0 && windowsAvailable_ &&
            tuning_.unitsOverride == 0 &&
            total / n >= ((stats.addressBits & (kWindowAlignBytes - 1)) == 0 && tuning_.windowAlignedMBps != 0 ? kWindowSliceMinAlignedSegmentBytes
                                                                                                         : kWindowSliceMinSegmentBytes) &&
            g_leasesOut.load(std::memory_order_relaxed) <= 1) {
            for (uint32_t at = 0; at < n; at += kInlineSegs) {
                const uint32_t m = n - at < kInlineSegs ? n - at : kInlineSegs;
                const bool last = at + m == n;
                const int ret = SubmitOne(src + at, dst + at, len + at, m, route, stream, last ? mask : nullptr, maskValue, false,
                                          true);
                if (ret != BM_OK) {
                    return ret;
                }
            }
            return BM_OK;
        }
        units = ChooseUnits(total, cu, route, tuning_);
        if (route == MFRT_ROUTE_HBM) {
            const uint32_t parts = HeldLaunches(stats, src, dst, len, n, unordered);
            if (parts > 1) {
                return SubmitHeld(src, dst, len, n, stats, parts, stream, mask, maskValue);
            }
            const int ret = SubmitPieces(src, dst, len, n, stats, units, stream, mask, maskValue, unordered);
            if (ret != kNotLaunched) {
                return ret;
            }
        }
        if (route == MFRT_ROUTE_TO_HOST && tuning_.unitsOverride == 0) {
            // Four accesses per lane, whose loads from HBM are in flight together: with one the walk over a table's chunks is too
            // slow for the link (K and V blocks of four requests 638 us, 669 with one; 256 workgroups with one 639).
            units = kDeepUnits;
        }
        // Many short segments: a chunk size that holds the longest of them gives every segment exactly
        // one chunk, which is the equal-count form below (no prefix, no search).
        if (tuning_.unitsOverride == 0 && stats.longest != 0) {
            for (uint32_t u = units; u <= 4 * kXcopyThreads; u *= 2) {
                if (stats.longest <= static_cast<uint64_t>(u) * kUnitBytes - kUnitBytes) {
                    units = u;
                    break;
                }
            }
        }
    }
    // Slot layout: triples | prefix | group map.  The map's size follows from the chunk count, which is bounded
    // here by one chunk per segment plus one per full chunk of payload.
    const uint64_t tripleBytes = 24ull * n;
    const uint64_t prefixBytes = RoundUp(4ull * (n + 1), 8);
    const uint64_t chunkBound = static_cast<uint64_t>(n) + queuedBytes / (static_cast<uint64_t>(units) * kUnitBytes);
    const uint32_t groupCapacity = static_cast<uint32_t>(
        std::min<uint64_t>(GroupCapacityFor(n), (chunkBound >> kGroupShiftMin) + 2));
    const uint64_t slotBytes = RoundUp(tripleBytes + prefixBytes + 4ull * groupCapacity, kUnitBytes);
    StagingSlot *slot = nullptr;
    ThreadLease &lease = ctx.Lease();
    int ret = AcquireSlot(lease, slotBytes, stream, slot);
    if (ret != BM_OK) {
        return ret;
    }
    uint64_t *triples = static_cast<uint64_t *>(slot->host);
    uint32_t *first = reinterpret_cast<uint32_t *>(static_cast<uint8_t *>(slot->host) + tripleBytes);
    uint32_t count = 0;
    ChunkPattern pattern;
    const uint64_t nchunk = BuildTableDirect(src, dst, len, n, units, triples, first, count, &pattern);
    if (nchunk >= kNoChunk) {
        MF_FAIL(BM_INVALID_PARAM, "batch too large for one launch: " << nchunk << " chunks");
    }
    if (count == 0) {   // nothing but empty segments
        InlinePlan empty;
        SegList none;
        (void)BuildInlinePlan(none, kXcopyThreads, empty);
        int err = mfk_xcopy_inline(&empty, route, 1, mask, maskValue, stream, 0, 0);
        return err == 0 ? BM_OK : BM_ERROR;
    }

    const uint32_t grid = GridFor(nchunk, cu, route, tuning_);
    TablePlan table{};
    table.nseg = count;
    table.nchunk = static_cast<uint32_t>(nchunk);
    table.units = units;
    int err = 0;
    // Chunk counts that repeat (pages of one size, K and V blocks in turn): a workgroup finds its descriptor by
    // a division and a few comparisons, so the only thing it needs from the table is that one descriptor, which it
    // can read straight out of the pinned slot.  No upload launch, nothing serial in front of the copy.
    // Over the link a few workgroups walk all the chunks, and a descriptor fetch across the link it saturates would be in every
    // one of their steps: those tables are uploaded (K and V blocks of four requests to the host: 638 us, 681 from the slot and
    // on 4 KiB chunks).
    if (pattern.period != 0 && route == MFRT_ROUTE_HBM) {
        table.triples = triples;
        table.pattern = pattern;
        err = mfk_xcopy_table(&table, route, grid, mask, maskValue, stream);
        g_launches.fetch_add(1, std::memory_order_relaxed);
    } else {
        // Ragged segments: prefix and group map go to HBM with the triples (with them in host memory every
        // step of the lookup is a link round trip: 16 384 ragged segments 135 us against 74).  The upload is
        // launched without a barrier: the slot's device half is free (AcquireSlot has waited for its last
        // reader), so it may run while the caller's earlier copies still do; the table launch behind it waits
        // for both.
        // A pattern needs the triples only.
        uint32_t *group = reinterpret_cast<uint32_t *>(static_cast<uint8_t *>(slot->host) + tripleBytes + prefixBytes);
        uint64_t usedBytes = RoundUp(24ull * count, kUnitBytes);
        if (pattern.period != 0) {
            table.pattern = pattern;
        } else {
            table.groupShift = BuildGroupMap(first, count, group, groupCapacity);
            usedBytes = RoundUp(tripleBytes + prefixBytes + 4ull * (GroupCount(nchunk, table.groupShift) + 1), kUnitBytes);
        }
        ret = EnsureDevice(*slot, slotBytes);
        if (ret != BM_OK) {
            return ret;
        }
        const uint64_t hostAddr = reinterpret_cast<uint64_t>(slot->host);
        const uint64_t devAddr = reinterpret_cast<uint64_t>(slot->dev);
        InlinePlan stagePlan;
        if (!BuildInlineDirect(&hostAddr, &devAddr, &usedBytes, 1, kXcopyThreads, stagePlan)) {
            MF_FAIL(BM_INVALID_PARAM, "descriptor table of " << usedBytes << " bytes is too large");
        }
        err = mfk_xcopy_inline(&stagePlan, MFRT_ROUTE_FROM_HOST, stagePlan.nchunk, nullptr, 0, stream,
                               tuning_.stageUnordered ? 1 : 0, 0);
        if (err != 0) {
            MF_FAIL(BM_ERROR, "descriptor staging launch failed: " << mfrt_error_string(err));
        }
        const uint8_t *devBase = static_cast<const uint8_t *>(slot->dev);
        table.triples = reinterpret_cast<const uint64_t *>(devBase);
        table.first = reinterpret_cast<const uint32_t *>(devBase + tripleBytes);
        table.group = reinterpret_cast<const uint32_t *>(devBase + tripleBytes + prefixBytes);
        err = mfk_xcopy_table(&table, route, grid, mask, maskValue, stream);
        g_launches.fetch_add(2, std::memory_order_relaxed);
    }
    if (err != 0) {
        // an earlier launch may still be reading the slot: keep it reserved until the stream has passed this point
        (void)MarkQueued(lease, slot, stream, true);
        MF_FAIL(BM_ERROR, "xcopy table launch failed: " << mfrt_error_string(err));
    }
    NotePending(stream, queuedBytes);
    return MarkQueued(lease, slot, stream, false);
}

// A batch that becomes part of a graph: launches of kInlineSegs segments, whose descriptors are copied into the graph with their
// arguments.  (Every run fits the kernel arguments: it has at most kInlineSegs segments of at most kInlinePiece once merged and cut.)
int XcopyEngine::SubmitRecorded(const uint64_t *src, const uint64_t *dst, const uint64_t *len, uint32_t n, int route, void *stream,
                                void *mask, uint32_t maskValue)
{
    SegList segs;
    NormalizeSegments(src, dst, len, n, kInlinePiece, segs);
    uint32_t at = 0;
    do {
        const uint32_t m = segs.Size() - at < kInlineSegs ? segs.Size() - at : kInlineSegs;
        const int ret = SubmitOne(segs.src.data() + at, segs.dst.data() + at, segs.len.data() + at, m, route, stream,
                                  at + m == segs.Size() ? mask : nullptr, maskValue, false, false);
        if (ret != BM_OK) {
            return ret;
        }
        at += m;
    } while (at < segs.Size());
    return BM_OK;
}

// A batch between HBM addresses in one launch of pieces; kNotLaunched where their list would outgrow the batch.
int XcopyEngine::SubmitPieces(const uint64_t *src, const uint64_t *dst, const uint64_t *len, uint32_t n, const BatchStats &stats, uint32_t units,
                              void *stream, void *mask, uint32_t maskValue, bool unordered)
{
    const uint64_t total = stats.total;
    if (tuning_.unitsOverride != 0) {
        units = units <= kXcopyThreads ? kXcopyThreads : units <= 2 * kXcopyThreads ? 2 * kXcopyThreads : kDeepUnits;
    } else {
        units = DeepHoldApplies(total, n, MFRT_ROUTE_HBM, unordered) ? kDeepUnits : PieceUnits(stats, n, unordered);
    }
    // A few segments of gigabytes would make a list of millions of pieces, megabytes that take the host longer to write than a chunk
    // prefix takes the GPU to read.
    const uint64_t bound = PieceBound(total, n, units);
    if (bound > std::max<uint64_t>(kPieceListMin, 2ull * n) || bound > kPieceMaxCount) {
        return kNotLaunched;
    }
    ThreadLease &lease = t_ctx.Lease();
    StagingSlot *slot = nullptr;
    const int ret = AcquireSlot(lease, bound * sizeof(Piece), stream, slot);
    if (ret != BM_OK) {
        return ret;
    }
    Piece *pieces = static_cast<Piece *>(slot->host);
    const uint32_t count = BuildPieces(src, dst, len, n, units, pieces);
    if (count == 0) {   // nothing but empty segments
        InlinePlan empty;
        SegList none;
        (void)BuildInlinePlan(none, kXcopyThreads, empty);
        return mfk_xcopy_inline(&empty, MFRT_ROUTE_HBM, 1, mask, maskValue, stream, 0, 0) == 0 ? BM_OK : BM_ERROR;
    }
    const uint32_t hold = HoldForPieces(stats, n, count, units, unordered);
    uint32_t reading = 0;
    const uint32_t rate = hold != 0 ? 0 : PieceWindowRate(stats, src, dst, len, n, count, units, unordered, reading);
    const bool own = stream == lease.stream;
    // Reporting costs the GPU the atomics of every wave (200 x 128 KiB 9.9 us with an event, 10.4 so, 2000 x 40 000 34.0 / 37.4), the
    // event costs the host: for batches that the GPU copies in less time than the host needs for the next (4 us and some ns a segment).
    const bool reports = !own && rate == 0 && total <= kReportBytes + kReportSegmentBytes * n;
    if (mask == nullptr && (own ? HasDoneWord(lease) : reports && HasReadMarks(lease))) {
        const uint32_t seq = own ? lease.startSeq + 1 : slot->readSeq + 1;
        const int failed = mfk_xcopy_pieces_reported(pieces, count, total, units, hold, rate, reading, own ? StartedWord(lease) : ReadWord(lease, *slot), seq,
                                                     own ? nullptr : ReadCounter(lease, *slot), stream);
        if (failed != 0) {
            (void)MarkQueued(lease, slot, stream, true);
            MF_FAIL(BM_ERROR, "xcopy launch failed: " << mfrt_error_string(failed));
        }
        (own ? lease.startSeq : slot->readSeq) = seq;
        slot->startSeq = own ? seq : 0;
        slot->state = own ? StagingSlot::kFollowed : StagingSlot::kReported;
        g_launches.fetch_add(1, std::memory_order_relaxed);
        NotePending(stream, total);
        return BM_OK;
    }
    void *event = EventOfLaunch(lease, *slot, stream);
    const int err = rate != 0 ? mfk_xcopy_pieces_windowed(pieces, count, total, rate, reading, mask, maskValue, stream, event)
                              : mfk_xcopy_pieces(pieces, count, total, units, mask, maskValue, stream, hold, event);
    if (err != 0) {
        (void)MarkQueued(lease, slot, stream, true);   // the launch may have gone out with only the word behind it failing
        MF_FAIL(BM_ERROR, "xcopy launch failed: " << mfrt_error_string(err));
    }
    g_launches.fetch_add(1, std::memory_order_relaxed);
    NotePending(stream, total);
    return MarkQueued(lease, slot, stream, false, event != nullptr);
}

int XcopyEngine::SubmitDeviceTable(const void *triples, uint32_t n, int route, void *stream, void *mask,
                                   uint32_t maskValue)
{
    if (!Started()) {
        MF_FAIL(BM_NOT_INITIALIZED, "xcopy engine not started");
    }
    if (mfrt_bind_thread() != 0) {
        MF_FAIL(BM_ERROR, "cannot make the GPU current on this thread");
    }
    if (stream == nullptr) {
        stream = ThreadStream();
        if (stream == nullptr) {
            MF_FAIL(BM_ERROR, "cannot create the thread's stream");
        }
    }
    if (n == 0) {
        InlinePlan empty;
        SegList none;
        (void)BuildInlinePlan(none, kXcopyThreads, empty);
        int err = mfk_xcopy_inline(&empty, route, 1, mask, maskValue, stream, 0, 0);
        return err == 0 ? BM_OK : BM_ERROR;
    }
    // Calls that become nodes of a graph have lists of their own, for a graph may be replayed beside plain calls.  They are made by the
    // thread's first plain call whichever way that goes: the recorded one may have more segments, or another thread may submit by then.
    // (A call that needs no list goes out without room for them.)
    ThreadLease &lease = t_ctx.Lease();
    int ret = BM_OK;
    if (lease.graphRests == nullptr && mfrt_stream_capturing(stream) == 0) {
        ret = EnsureRestLists(lease.graphRests, kSlots, kRestGraphCapacity);
        if (ret != BM_OK && ret != BM_MALLOC_FAILED) {
            return ret;
        }
    }
    // Up to kPlannedSegments segments one launch plans and copies.  Where it may not pace itself for the whole chip, because other
    // threads submit too, only the shorter ones.
    uint32_t hold = 0;
    uint32_t holdMore = 0;
    uint32_t windows = 0;
    const bool own = route == MFRT_ROUTE_HBM && tuning_.unitsOverride == 0 && tuning_.deviceTableWgPerCu == 0;
    if (own) {
        TablePaceFor(hold, holdMore, windows);
    }
    if (own && n <= (windows != 0 ? kPlannedSegments : 64 * kPlannedShortRun)) {
        const int err = mfk_xcopy_planned(triples, n, hold, holdMore, windows, mask, maskValue, stream);
        if (err != 0) {
            MF_FAIL(BM_ERROR, "xcopy launch of a device table failed: " << mfrt_error_string(err));
        }
        g_launches.fetch_add(1, std::memory_order_relaxed);
        NotePending(stream, ~0ull);   // sizes unknown here: the next wait sleeps on the stream
        return BM_OK;
    }
    // The list of long segments belongs to a slot: the next call of another stream gets another one.
    StagingSlot *slot = nullptr;
    const bool recorded = mfrt_stream_capturing(stream) != 0;
    ret = ret == BM_OK ? EnsureRestLists(lease.graphRests, kSlots, kRestGraphCapacity) : ret;
    if (ret == BM_OK && !recorded) {
        ret = AcquireSlot(lease, 0, stream, slot);
        ret = ret == BM_OK ? EnsureRestLists(slot->rest, 1, kRestCapacity) : ret;
    }
    if (ret != BM_OK) {
        return ret;
    }
    void *list = recorded ? static_cast<uint8_t *>(lease.graphRests) + lease.graphCursor++ % kSlots * RestListStride(kRestGraphCapacity)
                          : slot->rest;
    void *event = recorded ? nullptr : EventOfLaunch(lease, *slot, stream);
    const uint32_t cu = mfrt_cu_count();
    const uint32_t units = ChooseUnits(0, cu, route, tuning_);   // sizes are only known on the GPU
    const uint32_t capacity = recorded ? kRestGraphCapacity : kRestCapacity;
    // Where the launch may go in windows all workgroups but those that then copy start only to look and leave, through the few places
    // the others leave them.  us with four a segment and up to 1024 a CU / with up to 192: 16 384 pages scattered of 4 KiB 31.4 / 30.2, of
    // 8 KiB 58.2 / 56.7, of 16 KiB 109.2 / 106.4, 16 080 segments of 2 KiB 25.8 / 22.6, of 6 KiB 50.6 / 47.4, 40 000 of up to 9 KB 86.6 / 84.2,
    // 16 384 of 2 to 14 KB 58.0 / 58.4, at odd addresses 64.8 / 64.3, of up to 262 KB 925 / 928; with up to 128 a CU 60.2 and 932.
    constexpr uint32_t kSampledPerCu = 192;
    const auto gridOf = [&](uint32_t segments) {
        const uint32_t grid = DeviceTableGrid(segments, cu, route, tuning_);
        return windows != 0 && segments > kPlannedSegments ? std::min(grid, kSampledPerCu * (cu == 0 ? 256 : cu)) : grid;
    };
    int err = 0;
    for (uint32_t at = 0; at < n && err == 0; ) {
        const uint32_t m = n - at < capacity ? n - at : capacity;
        const bool last = m == n - at;
        err = mfk_xcopy_direct(static_cast<const uint64_t *>(triples) + 3ull * at, m, units, route, gridOf(m),
                               DeviceTableRestGrid(cu, route, tuning_), list, capacity, windows, last ? mask : nullptr, maskValue, stream,
                               last ? event : nullptr);
        g_launches.fetch_add(err == 0 ? 2 : 0, std::memory_order_relaxed);
        at += m;
    }
    if (err != 0) {
        if (!recorded) {
            (void)MarkQueued(lease, slot, stream, true);   // the first launch writes the list
        }
        MF_FAIL(BM_ERROR, "xcopy launch of a device table failed: " << mfrt_error_string(err));
    }
    NotePending(stream, ~0ull);   // sizes unknown here: the next wait sleeps on the stream
    return recorded ? BM_OK : MarkQueued(lease, slot, stream, false, event != nullptr);
}

#ifndef MF_RT_HIDDEN
int XcopyEngine::SubmitDeviceTableStatic(const void *triples, uint32_t n, int route, void *stream)
{
    if (!Started()) {
        MF_FAIL(BM_NOT_INITIALIZED, "xcopy engine not started");
    }
    if (n > MFK_STATIC_TABLE_SEGMENTS) {
        MF_FAIL(BM_INVALID_PARAM, "table of " << n << " segments exceeds the " << MFK_STATIC_TABLE_SEGMENTS
                << " the statically allocated scratch holds; split the table or use mf_xcopy_device_table");
    }
    if (n == 0) {
        return BM_OK;
    }
    if (mfrt_bind_thread() != 0) {
        MF_FAIL(BM_ERROR, "cannot make the GPU current on this thread");
    }
    const uint32_t cu = mfrt_cu_count();
    const uint32_t units = ChooseUnits(0, cu, route, tuning_);   // sizes are only known on the GPU
    const int err = mfk_xcopy_table_static(triples, n, units, route, DeviceTableGrid(n, cu, route, tuning_),
                                           DeviceTableRestGrid(cu, route, tuning_), stream);
    if (err != 0) {
        MF_FAIL(BM_ERROR, "static-scratch table launch failed (" << err << ")");
    }
    g_launches.fetch_add(2, std::memory_order_relaxed);
    NotePending(stream, ~0ull);
    return BM_OK;
}
#endif

}  // namespace mf
