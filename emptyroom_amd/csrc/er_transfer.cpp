// er_transfer.cpp -- see er_transfer.h.
#include "er_transfer.h"

#include <algorithm>
#include <cstdint>
#include <cstring>
#include <map>
#if defined(__x86_64__)
#include <immintrin.h>
#endif

namespace er {

namespace {

constexpr size_t kSlot = 2 << 20;     // bytes of a slot (37 us of the link)
constexpr int kSlots = 8;
constexpr size_t kPiece = 256 << 10;  // bytes copied at a time
// Arrays of this size and more usually are fresh pages, huge ones where the
// system gives them, and the page faults take longer than the copy: three
// threads help, slots follow the array's 2 MiB pages and one thread copies a
// whole slot, since threads that fault on one page each clear it (64 MB into
// fresh pages by 8 threads: 1.3 ms in pieces of 2 MiB, 2.2 ms in pieces of 256
// KiB).  Alone / with threads: 12 MB 399 / 393 us, 20 MB 793 / 607, 40 MB 3154 /
// 1872, and the caller then reads the array as fast as before.  (Uploads do not
// go through threads: the caller's next write to what several threads have read
// takes its lines back from their caches, 24 MB of it 15 ms.)
constexpr size_t kFreshMin = 16 << 20;
constexpr long kThreads = 3;

void pause() {
#if defined(__x86_64__)
    _mm_pause();
#else
    std::this_thread::yield();
#endif
}

}  // namespace

// One copy: chunk c (of a slot's size) goes through slot c % kSlots, in pieces
// handed out in order; a piece may be copied once its chunk is ready.
struct Transfer::Job {
    char *host;
    size_t bytes, first, piece;  // first: bytes of chunk 0
    char *const *slot = nullptr;
    long chunks, per_chunk, pieces;
    std::atomic<long> next{0}, ready{0};
    std::atomic<long> done[kSlots] = {};
    std::atomic<bool> abort{false};

    Job(void *h, size_t n) : host((char *)h), bytes(n) {
        const bool fresh = n >= kFreshMin;
        first = std::min(n, fresh ? kSlot - (size_t)((uintptr_t)h % kSlot) : kSlot);
        piece = fresh ? kSlot : kPiece;
        per_chunk = (long)(kSlot / piece);
        chunks = 1 + (long)((n - first + kSlot - 1) / kSlot);
        pieces = chunks * per_chunk;  // some of the first and last chunk's are empty
    }
    size_t begin(long c) const { return c == 0 ? 0 : first + (size_t)(c - 1) * kSlot; }
    size_t chunk_bytes(long c) const {
        return c == 0 ? first : std::min(kSlot, bytes - begin(c));
    }
    void copy(long p) {
        const long c = p / per_chunk;
        const size_t off = (size_t)(p % per_chunk) * piece, len = chunk_bytes(c);
        if (off < len) {
            const size_t n = std::min(piece, len - off);
            std::memcpy(host + begin(c) + off, slot[c % kSlots] + off, n);
        }
        done[c % kSlots].fetch_add(1, std::memory_order_release);
    }
    // a helping thread: every piece it can get
    void run() {
        for (;;) {
            const long p = next.fetch_add(1);
            if (p >= pieces) return;
            while (ready.load(std::memory_order_acquire) <= p / per_chunk) {
                if (abort.load()) return;
                pause();
            }
            copy(p);
        }
    }
    // the caller, which makes chunks ready: at most one piece that already is
    void help() {
        long p = next.load();
        if (p < pieces && p / per_chunk < ready.load() && next.compare_exchange_strong(p, p + 1))
            copy(p);
        else
            pause();
    }
    // every piece of chunk c has been copied
    bool emptied(long c) const {
        return done[c % kSlots].load(std::memory_order_acquire) >=
               (c / kSlots + 1) * per_chunk;
    }
};

// One event per slot for the length of a copy: the runtime keeps an event's last
// stream and looks at it again, so an event must not outlive that stream.
struct Events {
    hipEvent_t ev[kSlots] = {};
    bool make(int n) {
        for (int k = 0; k < n; k++)
            if (hipEventCreateWithFlags(&ev[k], hipEventDisableTiming) != hipSuccess) {
                (void)hipGetLastError();
                return false;
            }
        return true;
    }
    ~Events() {
        for (hipEvent_t e : ev)
            if (e) (void)hipEventDestroy(e);
    }
};

Transfer::~Transfer() {
    {
        std::lock_guard<std::mutex> lk(mu_);
        stop_ = true;
    }
    cv_.notify_all();
    for (std::thread &t : threads_) t.join();
    for (char *p : slot_) (void)hipHostFree(p);
    if (small_) (void)hipHostFree(small_);
}

std::shared_ptr<Transfer> Transfer::of_device(int device) {
    static std::mutex mu;
    static std::map<int, std::weak_ptr<Transfer>> known;
    std::lock_guard<std::mutex> lk(mu);
    std::shared_ptr<Transfer> t = known[device].lock();
    if (!t) known[device] = t = std::make_shared<Transfer>();
    return t;
}

// The small buffer (chunks = 0), or slots and threads for a copy of so many
// chunks; what is there stays.
bool Transfer::ensure(long chunks, bool threads) {
    if (chunks == 0 && !small_ && hipHostMalloc((void **)&small_, kBuffer) != hipSuccess) {
        (void)hipGetLastError();
        small_ = nullptr;
        return false;
    }
    slot_.reserve(kSlots);
    while ((long)slot_.size() < std::min<long>(kSlots, chunks)) {
        void *p = nullptr;
        if (hipHostMalloc(&p, kSlot) != hipSuccess) {
            (void)hipGetLastError();
            return false;
        }
        slot_.push_back((char *)p);
    }
    const long cores = std::max(1l, (long)std::thread::hardware_concurrency());
    try {
        while (threads && (long)threads_.size() < std::min(kThreads, cores - 1))
            threads_.emplace_back([this] { work(); });
    } catch (...) {
        // as many helpers as the system gives; the caller copies too
    }
    return true;
}

void Transfer::work() {
    std::unique_lock<std::mutex> lk(mu_);
    unsigned long seen = 0;
    for (;;) {
        cv_.wait(lk, [&] { return stop_ || (job_ && count_ != seen); });
        if (stop_) return;
        Job *j = job_;
        seen = count_;
        active_++;
        lk.unlock();
        j->run();
        lk.lock();
        active_--;
        if (active_ == 0) cv_.notify_all();
    }
}

void Transfer::start(Job *job) {
    {
        std::lock_guard<std::mutex> lk(mu_);
        job_ = job;
        count_++;
    }
    cv_.notify_all();
}

void Transfer::finish() {
    std::unique_lock<std::mutex> lk(mu_);
    job_ = nullptr;
    cv_.wait(lk, [&] { return active_ == 0; });
}

hipError_t Transfer::out(void *host, const void *dev, size_t bytes, hipStream_t s) {
    std::unique_lock<std::mutex> lk(busy_, std::defer_lock);
    if (bytes <= kSmall && lk.try_lock() && ensure(0, false)) {
        hipError_t e = hipMemcpyAsync(small_, dev, bytes, hipMemcpyDeviceToHost, s);
        if (e == hipSuccess) e = hipStreamSynchronize(s);
        if (e == hipSuccess) std::memcpy(host, small_, bytes);
        return e;
    }
    Job job(host, bytes);
    Events events;
    // what the stream still computes is waited for first: the slots belong to every
    // context of the device, and the helping threads poll
    if (bytes > kSmall) {
        const hipError_t e = hipStreamSynchronize(s);
        if (e != hipSuccess) return e;
    }
    if (bytes <= kSmall || !lk.try_lock() || !ensure(job.chunks, bytes >= kFreshMin) ||
        !events.make((int)std::min<long>(kSlots, job.chunks))) {
        hipError_t e = hipMemcpyAsync(host, dev, bytes, hipMemcpyDeviceToHost, s);
        return e == hipSuccess ? hipStreamSynchronize(s) : e;
    }
    job.slot = slot_.data();
    hipError_t e = hipSuccess;
    auto issue = [&](long c) {
        const int k = (int)(c % kSlots);
        e = hipMemcpyAsync(slot_[k], (const char *)dev + job.begin(c), job.chunk_bytes(c),
                           hipMemcpyDeviceToHost, s);
        if (e == hipSuccess) e = hipEventRecord(events.ev[k], s);
    };
    for (long c = 0; c < std::min<long>(kSlots, job.chunks) && e == hipSuccess; c++) issue(c);
    if (bytes >= kFreshMin) start(&job);
    // chunks the link has brought are handed out, emptied slots refilled, in turn
    long arrived = 0, issued = std::min<long>(kSlots, job.chunks);
    while (arrived < job.chunks && e == hipSuccess) {
        bool idle = true;
        if (arrived < issued) {
            e = hipEventQuery(events.ev[arrived % kSlots]);
            if (e == hipSuccess) {
                job.ready.store(++arrived, std::memory_order_release);
                idle = false;
            } else if (e == hipErrorNotReady) {
                e = hipSuccess;
            }
        }
        if (e == hipSuccess && issued < job.chunks && job.emptied(issued - kSlots)) {
            issue(issued++);
            idle = false;
        }
        if (idle) job.help();
    }
    if (e == hipSuccess)
        for (long c = std::max(0L, job.chunks - kSlots); c < job.chunks; c++)
            while (!job.emptied(c)) job.help();
    else job.abort.store(true);
    finish();
    if (e != hipSuccess) (void)hipStreamSynchronize(s);  // no copy into the ring is left
    return e;
}

hipError_t Transfer::in(void *dev, const void *host, size_t bytes, hipStream_t s, Staged *hold) {
    char *pinned = nullptr;
    std::unique_lock<std::mutex> lk;
    if (bytes <= kSmall) lk = small(&pinned);
    if (!pinned) return hipMemcpyAsync(dev, host, bytes, hipMemcpyHostToDevice, s);
    std::memcpy(pinned, host, bytes);
    hold->lk_ = std::move(lk);
    hold->s_ = s;
    return hipMemcpyAsync(dev, pinned, bytes, hipMemcpyHostToDevice, s);
}

Transfer::Staged::~Staged() {
    if (lk_.owns_lock()) (void)hipStreamSynchronize(s_);
}

std::unique_lock<std::mutex> Transfer::small(char **p) {
    *p = nullptr;
    std::unique_lock<std::mutex> lk(busy_, std::defer_lock);
    if (lk.try_lock() && ensure(0, false)) *p = small_;
    else if (lk.owns_lock()) lk.unlock();
    return lk;
}

}  // namespace er
