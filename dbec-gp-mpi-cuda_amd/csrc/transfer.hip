// transfer.hip - fields between device memory and host arrays (transfer.hpp).
//
// The caller's arrays are pageable, often fresh from the allocator.  The
// runtime's own pageable copy takes them through one staging thread, and a
// new page costs its first writer a fault: 134 MB (256^3 FP64) took 12.7 ms,
// the mixed form with its conversion by one thread 24 ms.  Here pieces of up
// to 2 MiB go through pinned slots, and for arrays past 32 MiB (below that the
// allocator hands out touched pages) the caller and kWorkers threads copy or
// convert between the slots and the array while the copy engine moves the next
// pieces: 3.4 and 2.5 ms.  The mixed form moves 4 bytes a value over the bus.
//
// Slots and threads outlive a call: at most kMaxSlots and kWorkers per process,
// shared by all threads and contexts (a slot is in use by one call at a time),
// given back when the last context ends.  A call that finds no slot, or a small
// field, goes the plain way.  The caller never waits for a thread as such, only
// for pieces that one has taken: on a host whose CPUs are busy (another
// library's spinning workers) waiting for seven threads to get a time slice
// cost 4 ms a call.
#include "transfer.hpp"

#include <algorithm>
#include <atomic>
#include <condition_variable>
#include <cstring>
#include <functional>
#include <memory>
#include <mutex>
#include <new>
#include <thread>
#include <vector>

namespace dbec {

namespace {

constexpr size_t kPiece = size_t(2) << 20;  // bytes of a slot, the largest piece; a field goes in 16 pieces or
constexpr size_t kPieceMin = size_t(256) << 10;  // more down to this size
// Device bytes up to which the plain way is kept, in us plain / staged by the
// caller alone: fetch FP64 128^3 (16 MB) 1010 / 693, 96^3 (6.8 MB) 417 / 402,
// 96x16x192 complex (4.5 MB) 275 / 358, mixed 96^3 (3.5 MB) 381 / 300, 64^3
// complex (2 MB) 200 / 189, 96x64x64 phi (1.5 MB) 147 / 149, 64^3 phi (1 MB)
// 100 / 112; store 128^3 FP64 486 / 580, 96^3 mixed 213 / 315, 80x96x160
// complex mixed (9.8 MB) 668 / 574.
constexpr size_t kFetch64 = size_t(6) << 20, kFetch32 = size_t(3) << 19;
constexpr size_t kStore64 = size_t(32) << 20, kStore32 = size_t(4) << 20;
constexpr size_t kOneThread = size_t(32) << 20;  // host bytes the caller moves alone
constexpr int kWorkers = 7, kSlotsPerCall = 16, kMaxSlots = 32;

struct Slot {
    void *mem = nullptr;
    hipEvent_t ev = nullptr;
    int device = -1;
};

std::mutex g_mu;
std::vector<Slot> g_free;
int g_slots = 0, g_users = 0;

void destroy(Slot &s) {
    if (s.ev) (void)hipEventDestroy(s.ev);
    if (s.mem) (void)hipHostFree(s.mem);
    s = Slot();
}

// Up to `want` slots of the device: its free ones, new ones up to the pool's
// bound, then free ones of other devices (the memory serves every device, an
// event only its own).  Fewer, or none, where all are in use or memory is short.
std::vector<Slot> acquire(int device, int want) {
    std::vector<Slot> got;
    got.reserve(want);
    std::lock_guard<std::mutex> lk(g_mu);
    for (size_t i = g_free.size(); i-- > 0 && (int)got.size() < want;)
        if (g_free[i].device == device) {
            got.push_back(g_free[i]);
            g_free.erase(g_free.begin() + (long)i);
        }
    while ((int)got.size() < want && g_slots < kMaxSlots) {
        Slot s;
        s.device = device;
        if (hipHostMalloc(&s.mem, kPiece, hipHostMallocPortable) != hipSuccess ||
            hipEventCreateWithFlags(&s.ev, hipEventDisableTiming) != hipSuccess) {
            destroy(s);
            (void)hipGetLastError();
            break;
        }
        ++g_slots;
        got.push_back(s);
    }
    while ((int)got.size() < want && !g_free.empty()) {
        Slot s = g_free.back();
        g_free.pop_back();
        (void)hipEventDestroy(s.ev);
        s.ev = nullptr;
        s.device = device;
        if (hipEventCreateWithFlags(&s.ev, hipEventDisableTiming) != hipSuccess) {
            s.ev = nullptr;
            destroy(s);
            --g_slots;
            (void)hipGetLastError();
            break;
        }
        got.push_back(s);
    }
    return got;
}

void give_back(std::vector<Slot> &v) {
    std::lock_guard<std::mutex> lk(g_mu);
    for (Slot &s : v) {
        bool kept = g_users > 0;
        if (kept) {
            try {
                g_free.push_back(s);
            } catch (const std::bad_alloc &) {
                kept = false;
            }
        }
        if (!kept) {
            destroy(s);
            --g_slots;
        }
    }
    v.clear();
}

// The pieces 0..n-1 of one call: taken in order by whoever is free, work(i)
// returns the first error.  The closure may refer to the caller's frame: it is
// entered only with a piece that the caller still waits for.
struct Task {
    std::function<hipError_t(size_t)> work;
    size_t n = 0;
    int device = 0;
    std::atomic<size_t> next{0}, done{0};
    std::atomic<int> err{(int)hipSuccess};

    void take_all() {
        bool set = false;
        for (size_t i; (i = next.fetch_add(1)) < n; done.fetch_add(1, std::memory_order_release)) {
            hipError_t e = hipSuccess;
            if (!set) e = hipSetDevice(device);
            set = true;
            if (e == hipSuccess && err.load() == (int)hipSuccess) e = work(i);
            if (e != hipSuccess) {
                int none = (int)hipSuccess;
                err.compare_exchange_strong(none, (int)e);
            }
        }
    }
};

class Workers {
public:
    // Runs the task on the pool's threads and this one, until every piece is
    // done.  Never throws: copies may be on their way to the caller's slots.
    void run(const std::shared_ptr<Task> &t, bool alone) noexcept {
        if (!alone) {
            {
                std::lock_guard<std::mutex> lk(mu_);
                try {
                    tasks_.push_back(t);
                    while ((int)threads_.size() < kWorkers)
                        threads_.emplace_back([this, g = generation_] { loop(g); });
                } catch (const std::exception &) {  // fewer threads, or the caller alone, do the same work
                }
            }
            cv_.notify_all();
        }
        t->take_all();
        if (!alone) {
            std::lock_guard<std::mutex> lk(mu_);
            tasks_.erase(std::remove(tasks_.begin(), tasks_.end(), t), tasks_.end());
        }
        while (t->done.load(std::memory_order_acquire) < t->n) std::this_thread::yield();
    }
    // Ends the threads; a later run starts new ones.
    void stop() {
        std::vector<std::thread> th;
        {
            std::lock_guard<std::mutex> lk(mu_);
            th.swap(threads_);
            ++generation_;
        }
        cv_.notify_all();
        for (auto &t : th) t.join();
    }

private:
    // born: generation_ when the thread was made.  It may get the lock for the
    // first time only after stop() has passed (the caller moves every piece
    // itself then), and must end all the same.
    void loop(unsigned born) {
        std::unique_lock<std::mutex> lk(mu_);
        while (born == generation_) {
            if (tasks_.empty()) {
                cv_.wait(lk);
                continue;
            }
            const std::shared_ptr<Task> t = tasks_.front();
            lk.unlock();
            t->take_all();
            lk.lock();
            if (!tasks_.empty() && tasks_.front() == t) tasks_.erase(tasks_.begin());
        }
    }
    std::mutex mu_;
    std::condition_variable cv_;
    std::vector<std::shared_ptr<Task>> tasks_;
    std::vector<std::thread> threads_;
    unsigned generation_ = 0;
};

// Never destroyed: a thread of the host program may still be in a call while
// the process ends.  In static storage: the end of a context must not throw.
Workers &workers() {
    alignas(Workers) static unsigned char mem[sizeof(Workers)];
    static Workers *w = new (mem) Workers;
    return *w;
}

// The task of n pieces; `work` outlives its run.  Made before the transfer's
// first copy, after which nothing may throw.
template <typename F>
std::shared_ptr<Task> make_task(int device, size_t n, F &work) {
    auto t = std::make_shared<Task>();
    t->n = n;
    t->device = device;
    Task *raw = t.get();
    t->work = [&work, raw](size_t i) { return work(i, raw->err); };
    return t;
}
hipError_t run_task(const std::shared_ptr<Task> &t, size_t host_bytes) {
    workers().run(t, host_bytes <= kOneThread);
    return (hipError_t)t->err.load();
}

struct Pieces {
    size_t n, per, count;  // values, values per piece, pieces
    Pieces(size_t n_, size_t el)
        : n(n_), per(std::min(kPiece, std::max(kPieceMin, n_ * el / 16)) / el), count((n_ + per - 1) / per) {}
    size_t len(size_t i) const { return std::min(per, n - i * per); }
};

// Flags of the pieces whose copy has been queued (their slot's event recorded).
using Flags = std::vector<std::atomic<int>>;

bool wait_queued(const Flags &f, size_t i, const std::atomic<int> &err) {
    while (!f[i].load(std::memory_order_acquire)) {
        if (err.load() != (int)hipSuccess) return false;
        std::this_thread::yield();
    }
    return true;
}

hipError_t fetch_staged(const dbec_ctx *c, double *dst, const char *src, size_t n, bool f32, std::vector<Slot> &slots) {
    const size_t el = f32 ? sizeof(float) : sizeof(double);
    const Pieces pc(n, el);
    const size_t R = slots.size();
    Flags queued(pc.count);
    const auto queue = [&](size_t i) {
        Slot &s = slots[i % R];
        hipError_t e = hipMemcpyAsync(s.mem, src + i * pc.per * el, pc.len(i) * el, hipMemcpyDeviceToHost, c->stream);
        if (e == hipSuccess) e = hipEventRecord(s.ev, c->stream);
        if (e == hipSuccess) queued[i].store(1, std::memory_order_release);
        return e;
    };
    // the worker of piece i queues piece i + R into the slot it has emptied:
    // a piece waits only for one that a worker has taken before it
    const auto piece = [&](size_t i, std::atomic<int> &err) {
        if (!wait_queued(queued, i, err)) return hipSuccess;
        const Slot &s = slots[i % R];
        hipError_t r = hipEventSynchronize(s.ev);
        if (r != hipSuccess) return r;
        double *out = dst + i * pc.per;
        const size_t m = pc.len(i);
        if (f32) {
            const float *in = static_cast<const float *>(s.mem);
            for (size_t k = 0; k < m; ++k) out[k] = (double)in[k];
        } else {
            std::memcpy(out, s.mem, m * sizeof(double));
        }
        return i + R < pc.count ? queue(i + R) : hipSuccess;
    };
    const std::shared_ptr<Task> task = make_task(c->device, pc.count, piece);
    hipError_t e = hipSuccess;
    for (size_t i = 0; i < std::min(R, pc.count) && e == hipSuccess; ++i) e = queue(i);
    if (e == hipSuccess) e = run_task(task, n * sizeof(double));
    const hipError_t w = hipStreamSynchronize(c->stream);
    return e != hipSuccess ? e : w;
}

hipError_t store_staged(const dbec_ctx *c, char *dst, const double *src, size_t n, bool f32, std::vector<Slot> &slots) {
    const size_t el = f32 ? sizeof(float) : sizeof(double);
    const Pieces pc(n, el);
    const size_t R = slots.size();
    Flags queued(pc.count);
    const auto piece = [&](size_t i, std::atomic<int> &err) {
        Slot &s = slots[i % R];
        if (i >= R) {  // the slot's last copy has left it
            if (!wait_queued(queued, i - R, err)) return hipSuccess;
            const hipError_t r = hipEventSynchronize(s.ev);
            if (r != hipSuccess) return r;
        }
        const double *in = src + i * pc.per;
        const size_t m = pc.len(i);
        if (f32) {
            float *out = static_cast<float *>(s.mem);
            for (size_t k = 0; k < m; ++k) out[k] = (float)in[k];
        } else {
            std::memcpy(s.mem, in, m * sizeof(double));
        }
        hipError_t r = hipMemcpyAsync(dst + i * pc.per * el, s.mem, m * el, hipMemcpyHostToDevice, c->stream);
        if (r == hipSuccess) r = hipEventRecord(s.ev, c->stream);
        if (r == hipSuccess) queued[i].store(1, std::memory_order_release);
        return r;
    };
    const hipError_t e = run_task(make_task(c->device, pc.count, piece), n * sizeof(double));
    const hipError_t w = hipStreamSynchronize(c->stream);
    return e != hipSuccess ? e : w;
}

// run(slots) where the field is past `plain` bytes and slots are to be had (done: it ran).
template <typename F>
hipError_t staged(const dbec_ctx *c, size_t n, size_t el, size_t plain, F &&run, bool &done) {
    done = false;
    if (n * el <= plain) return hipSuccess;
    std::vector<Slot> slots;
    hipError_t e = hipSuccess;
    try {
        slots = acquire(c->device, (int)std::min(Pieces(n, el).count, (size_t)kSlotsPerCall));
        if (slots.empty()) return hipSuccess;
        done = true;
        e = run(slots);
    } catch (const std::bad_alloc &) {  // only ever before the first copy: the plain way
        done = false;
    }
    give_back(slots);
    return e;
}

}  // namespace

hipError_t fetch_field(const dbec_ctx *c, double *dst, const void *src, size_t n, bool f32) {
    bool done;
    hipError_t e = staged(c, n, f32 ? sizeof(float) : sizeof(double), f32 ? kFetch32 : kFetch64, [&](std::vector<Slot> &s) {
        return fetch_staged(c, dst, static_cast<const char *>(src), n, f32, s);
    }, done);
    if (done) return e;
    if (!f32) return fetch_plain(c, dst, static_cast<const double *>(src), n);
    std::vector<float> f(n);
    e = hipMemcpyAsync(f.data(), src, n * sizeof(float), hipMemcpyDeviceToHost, c->stream);
    if (e == hipSuccess) e = hipStreamSynchronize(c->stream);
    if (e == hipSuccess)
        for (size_t i = 0; i < n; i++) dst[i] = f[i];
    return e;
}

hipError_t fetch_plain(const dbec_ctx *c, double *dst, const double *src, size_t n) {
    const hipError_t e = hipMemcpyAsync(dst, src, n * sizeof(double), hipMemcpyDeviceToHost, c->stream);
    return e != hipSuccess ? e : hipStreamSynchronize(c->stream);
}

hipError_t store_field(const dbec_ctx *c, void *dst, const double *src, size_t n, bool f32) {
    bool done;
    hipError_t e = staged(c, n, f32 ? sizeof(float) : sizeof(double), f32 ? kStore32 : kStore64, [&](std::vector<Slot> &s) {
        return store_staged(c, static_cast<char *>(dst), src, n, f32, s);
    }, done);
    if (done) return e;
    if (!f32) {
        e = hipMemcpyAsync(dst, src, n * sizeof(double), hipMemcpyHostToDevice, c->stream);
        return e != hipSuccess ? e : hipStreamSynchronize(c->stream);
    }
    std::vector<float> f(src, src + n);
    e = hipMemcpyAsync(dst, f.data(), n * sizeof(float), hipMemcpyHostToDevice, c->stream);
    return e != hipSuccess ? e : hipStreamSynchronize(c->stream);
}

void staging_user(int change) {
    {
        std::lock_guard<std::mutex> lk(g_mu);
        g_users += change;
        if (g_users > 0) return;
        for (Slot &s : g_free) {
            destroy(s);
            --g_slots;
        }
        g_free.clear();
    }
    workers().stop();
}

}  // namespace dbec
