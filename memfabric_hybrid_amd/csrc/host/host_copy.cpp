#include "host_copy.h"

#include <cstring>
#include <thread>

#if defined(__x86_64__)
#include <emmintrin.h>
#endif

namespace mf {
namespace {

inline void CpuRelax()
{
#if defined(__x86_64__) || defined(__i386__)
    __builtin_ia32_pause();
#else
    std::this_thread::yield();
#endif
}

constexpr int kSpinRounds = 2000;   // about 100 us of polling between the pieces of one transfer

}  // namespace

HostCopyHelper &HostCopyHelper::Instance()
{
    static HostCopyHelper *helper = new HostCopyHelper();
    return *helper;
}

void HostCopyHelper::StreamCopy(void *dst, const void *src, size_t len)
{
    uint8_t *to = static_cast<uint8_t *>(dst);
    const uint8_t *from = static_cast<const uint8_t *>(src);
#if defined(__x86_64__)
    const size_t head = (0 - reinterpret_cast<uintptr_t>(to)) & 63;
    if (len >= 4096) {
        std::memcpy(to, from, head);
        to += head;
        from += head;
        len -= head;
        for (; len >= 64; len -= 64, to += 64, from += 64) {
            const __m128i *s = reinterpret_cast<const __m128i *>(from);
            __m128i *d = reinterpret_cast<__m128i *>(to);
            const __m128i a = _mm_loadu_si128(s);
            const __m128i b = _mm_loadu_si128(s + 1);
            const __m128i c = _mm_loadu_si128(s + 2);
            const __m128i e = _mm_loadu_si128(s + 3);
            _mm_stream_si128(d, a);
            _mm_stream_si128(d + 1, b);
            _mm_stream_si128(d + 2, c);
            _mm_stream_si128(d + 3, e);
        }
        _mm_sfence();       // what is stored next is seen behind it
    }
#endif
    std::memcpy(to, from, len);
}

void HostCopyHelper::Run(const Share &share)
{
    for (size_t i = share.begin.piece; i < share.count && i <= share.end.piece; ++i) {
        const size_t from = i == share.begin.piece ? share.begin.offset : 0;
        const size_t to = i == share.end.piece ? share.end.offset : share.tasks[i].len;
        if (to > from) {
            uint8_t *dst = static_cast<uint8_t *>(share.tasks[i].dst) + from;
            const uint8_t *src = static_cast<const uint8_t *>(share.tasks[i].src) + from;
            if (share.pastCaches) {
                StreamCopy(dst, src, to - from);
            } else {
                std::memcpy(dst, src, to - from);
            }
        }
    }
}

void HostCopyHelper::Loop(Worker *worker)
{
    uint64_t seen = 0;
    for (;;) {
        bool posted = false;
        for (int i = 0; i < kSpinRounds; ++i) {
            if (worker->seq.load(std::memory_order_acquire) != seen) {
                posted = true;
                break;
            }
            CpuRelax();
        }
        if (!posted) {
            std::unique_lock<std::mutex> lock(worker->m);
            worker->sleeping.store(true, std::memory_order_seq_cst);
            worker->cv.wait(lock, [&] { return worker->seq.load(std::memory_order_seq_cst) != seen; });
            worker->sleeping.store(false, std::memory_order_seq_cst);
        }
        seen = worker->seq.load(std::memory_order_acquire);   // one share is outstanding at most: the caller waits for it
        if (worker->part != nullptr) {
            worker->part(worker->context);
        } else {
            Run(worker->share);
        }
        worker->done.store(seen, std::memory_order_release);
    }
}

bool HostCopyHelper::HasWorkers()
{
    while (started_ < kWorkers && !unavailable_) {
        try {
            std::thread(&HostCopyHelper::Loop, this, &workers_[started_]).detach();
            ++started_;
        } catch (...) {
            unavailable_ = true;
        }
    }
    return started_ != 0;
}

void HostCopyHelper::Post(uint32_t w)
{
    Worker &worker = workers_[w];
    tickets_[w] = worker.seq.fetch_add(1, std::memory_order_seq_cst) + 1;
    if (worker.sleeping.load(std::memory_order_seq_cst)) {
        std::lock_guard<std::mutex> lock(worker.m);
        worker.cv.notify_one();
    }
}

void HostCopyHelper::Join(uint32_t w)
{
    for (int spins = 0; workers_[w].done.load(std::memory_order_acquire) != tickets_[w]; ++spins) {
        if (spins < kSpinRounds) {
            CpuRelax();
        } else {
            std::this_thread::yield();   // the helper has not been scheduled: do not hold the core it may need
        }
    }
}

bool HostCopyHelper::Begin(Part part, void *context)
{
    if (!owner_.try_lock()) {
        return false;
    }
    if (!HasWorkers()) {
        owner_.unlock();
        return false;
    }
    for (uint32_t w = 0; w < started_; ++w) {
        workers_[w].part = part;
        workers_[w].context = context;
        Post(w);
    }
    return true;
}

void HostCopyHelper::End(bool begun)
{
    if (!begun) {
        return;
    }
    for (uint32_t w = 0; w < started_; ++w) {
        Join(w);
        workers_[w].part = nullptr;
    }
    owner_.unlock();
}

void HostCopyHelper::CopySet(const Task *tasks, size_t count, bool pastCaches)
{
    size_t total = 0;
    for (size_t i = 0; i < count; ++i) {
        total += tasks[i].len;
    }
    auto alone = [&]() {
        for (size_t i = 0; i < count; ++i) {
            std::memcpy(tasks[i].dst, tasks[i].src, tasks[i].len);
        }
    };
    if (total < kSplitMin || !owner_.try_lock()) {
        alone();
        return;
    }
    std::lock_guard<std::mutex> owner(owner_, std::adopt_lock);
    if (!HasWorkers()) {
        alone();
        return;
    }
    // Equal shares by bytes; a cut inside a piece is moved down to a multiple of 4096 so that every
    // share stays page-aligned relative to the piece.  Share 0 is the caller's.
    const uint32_t parts = started_ + 1;
    Cut cuts[kWorkers + 2];
    cuts[parts] = Cut{count, 0};
    size_t piece = 0;
    size_t before = 0;      // bytes of the pieces in front of `piece`
    for (uint32_t p = 1; p < parts; ++p) {
        const size_t at = total / parts * p;
        while (piece < count && before + tasks[piece].len <= at) {
            before += tasks[piece].len;
            ++piece;
        }
        cuts[p] = piece < count ? Cut{piece, (at - before) & ~static_cast<size_t>(4095)} : Cut{count, 0};
    }
    Share shares[kWorkers + 1];
    for (uint32_t p = 0; p < parts; ++p) {
        shares[p] = Share{tasks, count, cuts[p], cuts[p + 1], pastCaches};
    }
    for (uint32_t w = 0; w < started_; ++w) {
        workers_[w].share = shares[w + 1];
        Post(w);
    }
    Run(shares[0]);
    for (uint32_t w = 0; w < started_; ++w) {
        Join(w);
    }
    shared_.fetch_add(1, std::memory_order_relaxed);
    pastCaches_.fetch_add(pastCaches ? 1 : 0, std::memory_order_relaxed);
}

}  // namespace mf
