// Host paths of libdbec_hip without a device: this program defines the HIP
// entry points that the library imports (the dynamic linker prefers the
// program's own), with device memory in host memory, copies to and from pinned
// memory left pending until somebody waits for them, and kernels that only
// leave their name.  test_host_paths.py builds it and runs one scenario a
// process; a scenario ends with "ok", or with what went wrong.
#include <dlfcn.h>
#include <hip/hip_runtime_api.h>
#include <pthread.h>
#include <unistd.h>

#include <atomic>
#include <climits>
#include <cstdio>
#include <cstdlib>
#include <cstring>
#include <deque>
#include <map>
#include <mutex>
#include <new>
#include <set>
#include <string>
#include <thread>
#include <vector>

#include "dbec.h"

namespace {

thread_local int in_fake = 0;              // allocations of the stand-in itself never fail
std::atomic<bool> short_of_memory{false};  // allocations fail while a fetched piece is pending
std::atomic<int> pending_fetches{0};
std::atomic<int> thread_delay_us{0};
std::atomic<int> pinned_live{0}, freed_in_flight{0};
std::atomic<int> allocs{0};  // host and device memory, events
std::atomic<int> staged_copies[16];
std::atomic<int> copies{0};

struct Enter {
    Enter() { ++in_fake; }
    ~Enter() { --in_fake; }
};

struct Op {
    void *dst;
    const void *src;
    size_t n;
};
struct Stream {
    int device;
    std::deque<Op> ops;
    size_t queued = 0, ended = 0;
};
struct Event {
    int device;
    Stream *stream = nullptr;
    size_t at = 0;
};
struct Fake {
    std::mutex mu;
    std::map<char *, size_t> pinned;
    std::set<Stream *> streams;
    std::map<const void *, std::string> kernels;
    std::map<std::string, unsigned> launched;  // mangled name -> threads per workgroup
};
Fake &fake() {  // also reached from the library's initialisers, before this program's
    static Fake *f = new Fake;
    return *f;
}
thread_local int device = 0;
struct Config {
    dim3 g, b;
    size_t shm;
    hipStream_t s;
};
thread_local Config config;

bool is_pinned(const void *p) {
    auto &m = fake().pinned;
    auto it = m.upper_bound(const_cast<char *>(static_cast<const char *>(p)));
    if (it == m.begin()) return false;
    --it;
    return static_cast<const char *>(p) < it->first + it->second;
}
void drain(Stream *s, size_t upto) {  // mu held
    while (!s->ops.empty() && s->ended < upto) {
        const Op o = s->ops.front();
        s->ops.pop_front();
        std::memcpy(o.dst, o.src, o.n);
        if (is_pinned(o.dst)) --pending_fetches;
        ++s->ended;
    }
}

}  // namespace

void *operator new(size_t n) {
    if (!in_fake && short_of_memory && pending_fetches > 0) throw std::bad_alloc();
    if (!in_fake) ++allocs;
    if (void *p = std::malloc(n ? n : 1)) return p;
    throw std::bad_alloc();
}
void operator delete(void *p) noexcept { std::free(p); }
void operator delete(void *p, size_t) noexcept { std::free(p); }

// Threads start as late as the scenario asks for, as they do on a busy host.
extern "C" int pthread_create(pthread_t *t, const pthread_attr_t *a, void *(*f)(void *), void *arg) {
    using Fn = int (*)(pthread_t *, const pthread_attr_t *, void *(*)(void *), void *);
    static const Fn real = reinterpret_cast<Fn>(dlsym(RTLD_NEXT, "pthread_create"));
    struct Late {
        void *(*f)(void *);
        void *arg;
    };
    auto *l = static_cast<Late *>(std::malloc(sizeof(Late)));
    *l = {f, arg};
    return real(t, a, [](void *p) -> void * {
        const Late l = *static_cast<Late *>(p);
        std::free(p);
        if (const int us = thread_delay_us) usleep((useconds_t)us);
        return l.f(l.arg);
    }, l);
}

extern "C" {

struct uint3_;
void **__hipRegisterFatBinary(const void *) {
    static void *module = nullptr;
    return &module;
}
void __hipUnregisterFatBinary(void **) {}
void __hipRegisterFunction(void **, const void *host, char *, const char *name, unsigned, uint3_ *, uint3_ *, dim3 *,
                           dim3 *, int *) {
    Enter in;
    fake().kernels[host] = name;
}
void __hipRegisterVar(void **, void *, char *, char *, int, size_t, int, int) {}
hipError_t __hipPushCallConfiguration(dim3 g, dim3 b, size_t shm, hipStream_t s) {
    config = {g, b, shm, s};
    return hipSuccess;
}
hipError_t __hipPopCallConfiguration(dim3 *g, dim3 *b, size_t *shm, hipStream_t *s) {
    *g = config.g, *b = config.b, *shm = config.shm, *s = config.s;
    return hipSuccess;
}
hipError_t hipLaunchKernel(const void *f, dim3, dim3 b, void **, size_t, hipStream_t) {
    Enter in;
    std::lock_guard<std::mutex> lk(fake().mu);
    fake().launched[fake().kernels[f]] = b.x * b.y * b.z;
    return hipSuccess;
}
hipError_t hipFuncSetAttribute(const void *, hipFuncAttribute, int) { return hipSuccess; }

hipError_t hipGetDeviceCount(int *n) { return *n = 16, hipSuccess; }
hipError_t hipGetDevice(int *d) { return *d = device, hipSuccess; }
hipError_t hipSetDevice(int d) {
    if (d < 0 || d >= 16) return hipErrorInvalidDevice;
    return device = d, hipSuccess;
}
hipError_t hipMemGetInfo(size_t *fr, size_t *tot) { return *fr = *tot = size_t(256) << 30, hipSuccess; }
hipError_t hipGetLastError() { return hipSuccess; }
const char *hipGetErrorString(hipError_t) { return "stand-in error"; }
hipError_t hipMalloc(void **p, size_t n) {
    ++allocs;
    return (*p = std::calloc(n, 1)) ? hipSuccess : hipErrorOutOfMemory;
}
hipError_t hipFree(void *p) { return std::free(p), hipSuccess; }
hipError_t hipGetSymbolAddress(void **p, const void *) {
    static char *mem = static_cast<char *>(std::calloc(DBEC_NOALLOC_SCRATCH_BYTES, 1));
    return *p = mem, hipSuccess;
}
hipError_t hipHostMalloc(void **p, size_t n, unsigned) {
    Enter in;
    if (!(*p = std::calloc(n, 1))) return hipErrorOutOfMemory;
    std::lock_guard<std::mutex> lk(fake().mu);
    fake().pinned[static_cast<char *>(*p)] = n;
    ++allocs, ++pinned_live;
    return hipSuccess;
}
hipError_t hipHostFree(void *p) {
    Enter in;
    std::lock_guard<std::mutex> lk(fake().mu);
    for (Stream *s : fake().streams)
        for (const Op &o : s->ops)
            if (o.dst == p || o.src == p) {
                ++freed_in_flight;
                return hipSuccess;  // the memory stays, so the pending copy is harmless here
            }
    fake().pinned.erase(static_cast<char *>(p));
    --pinned_live;
    return std::free(p), hipSuccess;
}
hipError_t hipStreamCreate(hipStream_t *s) {
    Enter in;
    auto *n = new Stream;
    n->device = device;
    std::lock_guard<std::mutex> lk(fake().mu);
    fake().streams.insert(n);
    return *s = reinterpret_cast<hipStream_t>(n), hipSuccess;
}
hipError_t hipStreamSynchronize(hipStream_t h) {
    Enter in;
    std::lock_guard<std::mutex> lk(fake().mu);
    auto *s = reinterpret_cast<Stream *>(h);
    return drain(s, s->queued), hipSuccess;
}
hipError_t hipStreamDestroy(hipStream_t h) {
    (void)hipStreamSynchronize(h);
    Enter in;
    std::lock_guard<std::mutex> lk(fake().mu);
    fake().streams.erase(reinterpret_cast<Stream *>(h));
    return delete reinterpret_cast<Stream *>(h), hipSuccess;
}
hipError_t hipMemcpyAsync(void *dst, const void *src, size_t n, hipMemcpyKind, hipStream_t h) {
    Enter in;
    std::lock_guard<std::mutex> lk(fake().mu);
    auto *s = reinterpret_cast<Stream *>(h);
    const bool to = is_pinned(dst), from = is_pinned(src);
    ++copies;
    if (to || from) ++staged_copies[s->device];
    if (to) ++pending_fetches;
    s->ops.push_back({dst, src, n});
    ++s->queued;
    if (!to && !from) drain(s, s->queued);  // pageable: the call waits
    return hipSuccess;
}
hipError_t hipMemsetAsync(void *p, int v, size_t n, hipStream_t h) {
    (void)hipStreamSynchronize(h);
    return std::memset(p, v, n), hipSuccess;
}
hipError_t hipEventCreateWithFlags(hipEvent_t *ev, unsigned) {
    Enter in;
    auto *n = new Event;
    n->device = device;
    ++allocs;
    return *ev = reinterpret_cast<hipEvent_t>(n), hipSuccess;
}
hipError_t hipEventCreate(hipEvent_t *ev) { return hipEventCreateWithFlags(ev, 0); }
hipError_t hipEventDestroy(hipEvent_t ev) { return delete reinterpret_cast<Event *>(ev), hipSuccess; }
hipError_t hipEventRecord(hipEvent_t ev, hipStream_t h) {
    std::lock_guard<std::mutex> lk(fake().mu);
    auto *e = reinterpret_cast<Event *>(ev);
    auto *s = reinterpret_cast<Stream *>(h);
    if (e->device != s->device) return hipErrorInvalidHandle;
    e->stream = s;
    e->at = s->queued;
    return hipSuccess;
}
hipError_t hipEventSynchronize(hipEvent_t ev) {
    Enter in;
    std::lock_guard<std::mutex> lk(fake().mu);
    auto *e = reinterpret_cast<Event *>(ev);
    if (e->stream) drain(e->stream, e->at);
    return hipSuccess;
}
hipError_t hipEventQuery(hipEvent_t ev) { return hipEventSynchronize(ev); }
hipError_t hipEventElapsedTime(float *ms, hipEvent_t, hipEvent_t) { return *ms = 1.f, hipSuccess; }
hipError_t hipStreamWaitEvent(hipStream_t, hipEvent_t ev, unsigned) { return hipEventSynchronize(ev); }
hipError_t hipStreamBeginCapture(hipStream_t, hipStreamCaptureMode) { return hipErrorNotSupported; }
hipError_t hipStreamEndCapture(hipStream_t, hipGraph_t *) { return hipErrorNotSupported; }
hipError_t hipGraphInstantiate(hipGraphExec_t *, hipGraph_t, hipGraphNode_t *, char *, size_t) {
    return hipErrorNotSupported;
}
hipError_t hipGraphLaunch(hipGraphExec_t, hipStream_t) { return hipErrorNotSupported; }
hipError_t hipGraphDestroy(hipGraph_t) { return hipSuccess; }
hipError_t hipGraphExecDestroy(hipGraphExec_t) { return hipSuccess; }

}  // extern "C"

namespace {

#define CHECK(c)                                                                       \
    do {                                                                               \
        if (!(c)) {                                                                    \
            std::printf("line %d: %s\n", __LINE__, #c);                                \
            std::fflush(stdout);                                                       \
            std::_Exit(1);                                                             \
        }                                                                              \
    } while (0)

dbec_ctx *create(long nx, long ny, long nz, dbec_mode mode, dbec_prec prec, int dev = 0) {
    dbec_params p;
    std::memset(&p, 0, sizeof p);
    p.nx = nx, p.ny = ny, p.nz = nz;
    p.dx = p.dy = p.dz = 0.2;
    p.dt = 0.002;
    p.vgamma = p.vnu = p.vlambda = 1.0;
    p.cutoff = 4.0;
    p.par = 2.0;
    p.device = dev;
    dbec_ctx *c = nullptr;
    CHECK(dbec_create(&p, mode, prec, nullptr, &c) == DBEC_OK);
    return c;
}

void round_trip(dbec_ctx *c, size_t n, int seed) {
    std::vector<double> a(n), b(n, -1.0);
    for (size_t i = 0; i < n; ++i) a[i] = (double)((i * 2654435761u + (size_t)seed * 40503u) & 0xfffff);  // floats hold it
    CHECK(dbec_set_psi(c, a.data()) == DBEC_OK);
    CHECK(dbec_get_psi(c, b.data()) == DBEC_OK);
    CHECK(std::memcmp(a.data(), b.data(), n * sizeof(double)) == 0);
}

// 40 MiB of host doubles: past the bound from which the pool's threads help
constexpr long BX = 160, BY = 128, BZ = 128;
constexpr size_t BIG = 2 * size_t(BX * BY * BZ);

// The last context ends before the threads that its transfer started have run.
void late_threads() {
    for (int k = 0; k < 3; ++k) {
        dbec_ctx *c = create(BX, BY, BZ, DBEC_REAL, DBEC_FP64);
        thread_delay_us = 400000;
        round_trip(c, BIG, k);
        CHECK(dbec_destroy(c) == DBEC_OK);
        thread_delay_us = 0;
        CHECK(pinned_live == 0);
    }
}

// Contexts come and go in several threads, whose transfers share pool and slots.
void callers() {
    thread_delay_us = 2000;
    std::vector<std::thread> th;
    for (int t = 0; t < 4; ++t)
        th.emplace_back([t] {
            for (int k = 0; k < 3; ++k) {
                dbec_ctx *c = create(BX, BY, BZ, DBEC_REAL, (t & 1) ? DBEC_MIXED : DBEC_FP64);
                round_trip(c, BIG, 10 * t + k);
                round_trip(c, BIG, 10 * t + k + 5);
                CHECK(dbec_destroy(c) == DBEC_OK);
            }
        });
    for (auto &t : th) t.join();
    CHECK(pinned_live == 0);
    CHECK(freed_in_flight == 0);
}

// No memory is to be had once the first pieces are on their way.
void memory() {
    for (int big = 0; big < 2; ++big)
        for (dbec_prec prec : {DBEC_FP64, DBEC_MIXED}) {
            const long nx = big ? BX : 48;  // 40 and 12 MiB of host doubles
            const size_t n = 2 * size_t(nx * BY * BZ);
            dbec_ctx *c = create(nx, BY, BZ, DBEC_REAL, prec);
            std::vector<double> a(n), b(n, -1.0);
            for (size_t i = 0; i < n; ++i) a[i] = (double)(i & 0xffff);
            CHECK(dbec_set_psi(c, a.data()) == DBEC_OK);
            short_of_memory = true;
            CHECK(dbec_get_psi(c, b.data()) == DBEC_OK);
            CHECK(freed_in_flight == 0);
            short_of_memory = false;
            CHECK(std::memcmp(a.data(), b.data(), n * sizeof(double)) == 0);
            CHECK(dbec_destroy(c) == DBEC_OK);
            CHECK(pinned_live == 0);
        }
}

// Contexts on more devices than the slots' bound would serve at once.
void devices() {
    std::vector<dbec_ctx *> c;
    for (int d = 0; d < 5; ++d) c.push_back(create(64, BY, BZ, DBEC_REAL, DBEC_FP64, d));
    for (int k = 0; k < 2; ++k)
        for (int d = 0; d < 5; ++d) {
            const int before = staged_copies[d];
            round_trip(c[d], 2 * size_t(64 * BY * BZ), d + k);
            CHECK(staged_copies[d] > before);
            CHECK(pinned_live <= 32 + 5);  // the slots, and each context's scalars
        }
    for (dbec_ctx *x : c) CHECK(dbec_destroy(x) == DBEC_OK);
    CHECK(pinned_live == 0);
}

// The largest extract that the no-allocation entry point takes: 8 MiB.
void noalloc() {
    dbec_ctx *c = create(64, BY, BZ, DBEC_IMAG, DBEC_FP64);
    CHECK(dbec_density_count(c, DBEC_DEN_XYZ, 1, 1, 1) * (long)sizeof(double) == DBEC_NOALLOC_SCRATCH_BYTES);
    std::vector<double> out(DBEC_NOALLOC_SCRATCH_BYTES / sizeof(double));
    const int before = allocs;
    for (int kind = DBEC_DEN_X; kind <= DBEC_DEN_XYZ; ++kind)
        CHECK(dbec_density_noalloc(c, kind, 1, 1, 1, out.data()) == DBEC_OK);
    CHECK(allocs == before);
    CHECK(dbec_destroy(c) == DBEC_OK);
}

// Output steps as large as they come: one sample per axis.
void long_steps() {
    dbec_ctx *c = create(16, 32, 16, DBEC_IMAG, DBEC_FP64);
    for (long o : {1000L, LONG_MAX - 20, LONG_MAX})
        for (int kind = DBEC_DEN_X; kind <= DBEC_DEN_XYZ; ++kind) {
            CHECK(dbec_density_count(c, kind, o, o, o) == 1);
            double out[2] = {-1.0, -1.0};
            CHECK(dbec_density(c, kind, o, o, o, out) == DBEC_OK);
            CHECK(out[0] == 0.0 && out[1] == -1.0);
            out[0] = -1.0;
            CHECK(dbec_density_noalloc(c, kind, o, o, o, out) == DBEC_OK);
            CHECK(out[0] == 0.0 && out[1] == -1.0);
        }
    CHECK(dbec_destroy(c) == DBEC_OK);
}

// Threads per workgroup of the kernel `name` in a call of three steps, 0 if it
// did not run.
unsigned launched(const char *name) {
    for (auto &k : fake().launched)
        if (k.first.find(std::to_string(std::strlen(name)) + name) != std::string::npos) return k.second;
    return 0;
}
void steps(long nx, long ny, long nz, dbec_mode mode, dbec_prec prec) {
    dbec_ctx *c = create(nx, ny, nz, mode, prec);
    fake().launched.clear();
    CHECK(dbec_step(c, 3, 0.0, 0.0, nullptr) == DBEC_OK);
    CHECK(dbec_destroy(c) == DBEC_OK);
}
bool fused() { return launched("k_plane_fwd") || launched("k_plane_inv") || launched("k_sweepz_zfwd"); }

// The kernels of a step's end and the next one's start.
void fuse(bool on) {
    for (dbec_mode mode : {DBEC_IMAG, DBEC_REAL})
        for (dbec_prec prec : {DBEC_FP64, DBEC_MIXED})
            for (long ny : {64, 160}) {  // a grid of the plane kernels, and one past them
                steps(64, ny, 64, mode, prec);
                CHECK(fused() == on);
                CHECK((launched("k_plane_fwd") > 0) == (on && ny == 64));
                CHECK((launched("k_sweep_z") && launched("k_zfwd")) || on);
            }
}

// Bounds on the z sweep's rows, from the environment: threads per workgroup of
// the fused kernel of complex lines, or 0 for the two kernels in its place.
void rows(dbec_prec prec, unsigned want) {
    steps(96, 160, 256, DBEC_REAL, prec);
    CHECK(launched("k_sweepz_zfwd") == want);
    CHECK(want || (launched("k_sweep_z") && launched("k_zfwd")));
}

// Whole or half tiles of complex rows: whole ones where the launch needs no
// more rounds of the chip with them.
void tiles() {
    const struct {
        long nx, ny, nz;
        bool half[2];  // FP64, mixed
    } cases[] = {{16, 160, 16, {false, false}},  {320, 512, 16, {true, false}},  {192, 160, 64, {false, false}},
                 {256, 320, 64, {true, false}},  {48, 160, 160, {false, false}}, {64, 160, 160, {true, false}},
                 {16, 160, 256, {false, false}}, {80, 160, 256, {true, true}},   {48, 160, 320, {false, false}},
                 {80, 160, 320, {true, true}},   {16, 160, 512, {true, false}}};
    for (auto &k : cases)
        for (dbec_prec prec : {DBEC_FP64, DBEC_MIXED}) {
            steps(k.nx, k.ny, k.nz, DBEC_REAL, prec);
            CHECK(launched("k_sweepz_zfwd") > 0);
            bool half = false;  // the kernel's last template argument
            for (auto &n : fake().launched)
                half |= n.first.find("k_sweepz_zfwd") != std::string::npos && n.first.find("Lb1EEEv") != std::string::npos;
            CHECK(half == k.half[prec]);
        }
}

// The 3-D extract of a small grid is one launch and one copy in either precision.
void one_slab() {
    for (dbec_prec prec : {DBEC_FP64, DBEC_MIXED})
        for (long n : {16L, 64L}) {
            dbec_ctx *c = create(n, n, n, DBEC_IMAG, prec);
            std::vector<double> out((size_t)(n * n * n));
            const int before = copies;
            CHECK(dbec_density(c, DBEC_DEN_XYZ, 1, 1, 1, out.data()) == DBEC_OK);
            CHECK(copies == before + 1);
            CHECK(dbec_destroy(c) == DBEC_OK);
        }
}

// The tuner times the mixed potential's own kernels where they are not the step's.
void tuned() {
    const auto ran = [](const char *what) {
        for (auto &k : fake().launched)
            if (k.first.find(what) != std::string::npos) return true;
        return false;
    };
    dbec_ctx *c = create(384, 384, 16, DBEC_IMAG, DBEC_MIXED);
    for (const char *k : {"k_xconvILi384EfLi1ELb0ENS_7FftPlanI", "k_xconvILi384EfLi2ELb0ENS_7FftPlanI",
                          "k_xconvILi384EfLi1ELb0ENS_8FftPlanBI", "k_xconvILi384EfLi2ELb0ENS_8FftPlanBI",
                          "k_ypassILi384ELin1EfLi1ENS_7FftPlanI", "k_ypassILi384ELin1EfLi2ENS_7FftPlanI",
                          "k_ypassILi384ELin1EfLi1ENS_8FftPlanBI", "k_ypassILi384ELin1EfLi2ENS_8FftPlanBI"})
        CHECK(ran(k));
    CHECK(dbec_destroy(c) == DBEC_OK);
    c = create(48, 64, 64, DBEC_IMAG, DBEC_MIXED);  // the step's convolution takes the planes' rows
    for (const char *k : {"k_xconvILi48EfLi1ELb0E", "k_xconvILi48EfLi2ELb0E", "k_xconvILi48EfLi1ELb1E"}) CHECK(ran(k));
    CHECK(dbec_destroy(c) == DBEC_OK);
}

}  // namespace

int main(int argc, char **argv) {
    alarm(100);
    const std::string s = argc > 1 ? argv[1] : "";
    if (s == "late_threads") late_threads();
    else if (s == "callers") callers();
    else if (s == "memory") memory();
    else if (s == "devices") devices();
    else if (s == "noalloc") noalloc();
    else if (s == "long_steps") long_steps();
    else if (s == "fused") fuse(true);
    else if (s == "unfused") fuse(false);
    else if (s == "rows") rows((dbec_prec)std::atoi(argv[2]), (unsigned)std::atoi(argv[3]));
    else if (s == "tiles") tiles();
    else if (s == "one_slab") one_slab();
    else if (s == "tuned") tuned();
    else return std::printf("no such scenario\n"), 2;
    std::printf("ok\n");
    return 0;
}
