// A stand-in for the HIP runtime, for checks of what the library does on the host: two devices that exist in name only,
// memory that is counted, streams and events that know their device, and one kernel, the one that moves a group of a
// transfer (a scenario that asks for them has the others too, which do what `pretend` says).  Its functions take the place of the real ones because the program that is asked for a symbol first is the
// executable.  Each scenario of main() prints what went wrong and returns non-zero.
#include <dlfcn.h>
#include <errno.h>
#include <hip/hip_runtime_api.h>
#include <pthread.h>
#include <stdio.h>
#include <stdlib.h>
#include <string.h>
#include <sys/mman.h>
#include <sys/resource.h>

#include <algorithm>
#include <chrono>
#include <map>
#include <mutex>
#include <string>
#include <thread>
#include <vector>

#include "comet_hip_rt.h"

namespace {

using Clock = std::chrono::steady_clock;
std::mutex mu;
constexpr int DEVICES = 2;
size_t total[DEVICES] = {288ull << 30, 288ull << 30}, used[DEVICES];
struct Block { size_t bytes; int device; };
std::map<char *, Block> blocks;
struct Stream { int device; bool live; Clock::time_point idle; };
std::vector<Stream *> streams;
struct Event { int device; bool live; Clock::time_point done; };
std::map<const void *, std::string> &kernels()          // asked for before this file's own statics are made
{
    static auto *k = new std::map<const void *, std::string>;
    return *k;
}
thread_local int current = 0;
thread_local hipError_t last = hipSuccess;
thread_local struct { dim3 grid, block; size_t lds; hipStream_t stream; } config;

hipError_t fail(hipError_t e, const char *what)
{
    fprintf(stderr, "fake hip: %s\n", what);
    return last = e;
}
Stream *stream_of(hipStream_t s) { return reinterpret_cast<Stream *>(s); }
Event *event_of(hipEvent_t e) { return reinterpret_cast<Event *>(e); }
bool on_device(const char *p, size_t bytes, int device)
{
    std::lock_guard<std::mutex> lk(mu);
    auto it = blocks.upper_bound(const_cast<char *>(p));
    if (it == blocks.begin())
        return false;
    --it;
    return it->second.device == device && p + bytes <= it->first + it->second.bytes;
}

}  // namespace

static int threads_left = 1 << 20;          // how many more the system has
static bool (*pretend)(const std::string &kernel, void **args) = nullptr;          // false: the launch is refused

extern "C" {

int pthread_create(pthread_t *t, const pthread_attr_t *a, void *(*f)(void *), void *arg)
{
    static const auto real = (int (*)(pthread_t *, const pthread_attr_t *, void *(*)(void *), void *))dlsym(RTLD_NEXT, "pthread_create");
    if (threads_left-- <= 0)
        return EAGAIN;
    return real(t, a, f, arg);
}
void **__hipRegisterFatBinary(const void *) { static void *h; return &h; }
void __hipUnregisterFatBinary(void **) {}
void __hipRegisterFunction(void **, const void *host, char *, const char *name, unsigned, void *, void *, void *, void *, int *)
{
    kernels()[host] = name;
}
void __hipRegisterVar(void **, void *, char *, char *, int, size_t, int, int) {}
hipError_t __hipPushCallConfiguration(dim3 g, dim3 b, size_t lds, hipStream_t s)
{
    config = {g, b, lds, s};
    return hipSuccess;
}
hipError_t __hipPopCallConfiguration(dim3 *g, dim3 *b, size_t *lds, hipStream_t *s)
{
    *g = config.grid;
    *b = config.block;
    *lds = config.lds;
    *s = config.stream;
    return hipSuccess;
}
hipError_t hipGetDeviceCount(int *n) { *n = DEVICES; return hipSuccess; }
hipError_t hipSetDevice(int d) { current = d; return hipSuccess; }
hipError_t hipGetDevice(int *d) { *d = current; return hipSuccess; }
hipError_t hipGetDevicePropertiesR0600(hipDeviceProp_tR0600 *p, int)
{
    memset(p, 0, sizeof *p);
    strcpy(p->gcnArchName, "gfx950");
    p->multiProcessorCount = 256;
    return hipSuccess;
}
hipError_t hipGetSymbolAddress(void **p, const void *) { static char room[16 << 20]; *p = room; return hipSuccess; }
hipError_t hipFuncSetAttribute(const void *, hipFuncAttribute, int) { return hipSuccess; }
int hipGetStreamDeviceId(hipStream_t s) { return stream_of(s)->device; }
hipError_t hipOccupancyMaxActiveBlocksPerMultiprocessor(int *n, const void *, int, size_t) { *n = 1; return hipSuccess; }
const char *hipGetErrorString(hipError_t e) { return e == hipErrorOutOfMemory ? "out of memory" : "fake error"; }
hipError_t hipGetLastError(void) { const hipError_t e = last; last = hipSuccess; return e; }

hipError_t hipMalloc(void **p, size_t bytes)
{
    std::lock_guard<std::mutex> lk(mu);
    if (used[current] + bytes > total[current])
        return last = hipErrorOutOfMemory;
    *p = mmap(nullptr, bytes, PROT_READ | PROT_WRITE, MAP_PRIVATE | MAP_ANONYMOUS | MAP_NORESERVE, -1, 0);
    if (*p == MAP_FAILED)
        return fail(hipErrorOutOfMemory, "mmap");
    used[current] += bytes;
    blocks[(char *)*p] = Block{bytes, current};
    return hipSuccess;
}
hipError_t hipFree(void *p)
{
    std::lock_guard<std::mutex> lk(mu);
    auto it = blocks.find((char *)p);
    if (it == blocks.end())
        return fail(hipErrorInvalidValue, "free of something else");
    used[it->second.device] -= it->second.bytes;
    munmap(p, it->second.bytes);
    blocks.erase(it);
    return hipSuccess;
}
hipError_t hipMemGetInfo(size_t *f, size_t *t)
{
    *t = total[current];
    *f = total[current] - used[current];
    return hipSuccess;
}
hipError_t hipHostMalloc(void **p, size_t bytes, unsigned) { *p = aligned_alloc(4096, (bytes + 4095) & ~4095ull); return hipSuccess; }
hipError_t hipHostFree(void *p) { free(p); return hipSuccess; }

hipError_t hipStreamCreate(hipStream_t *s)
{
    streams.push_back(new Stream{current, true, Clock::now()});
    *s = reinterpret_cast<hipStream_t>(streams.back());
    return hipSuccess;
}
hipError_t hipStreamCreateWithFlags(hipStream_t *s, unsigned) { return hipStreamCreate(s); }
hipError_t hipStreamDestroy(hipStream_t s) { stream_of(s)->live = false; return hipSuccess; }
hipError_t hipStreamSynchronize(hipStream_t s) { std::this_thread::sleep_until(stream_of(s)->idle); return hipSuccess; }
hipError_t hipStreamQuery(hipStream_t s) { return Clock::now() < stream_of(s)->idle ? hipErrorNotReady : hipSuccess; }
hipError_t hipStreamWaitEvent(hipStream_t, hipEvent_t, unsigned) { return hipSuccess; }
hipError_t hipDeviceSynchronize(void)
{
    Clock::time_point until = Clock::now();          // what has been launched by now
    for (Stream *s : streams)
        if (s->live && s->device == current)
            until = std::max(until, s->idle);
    std::this_thread::sleep_until(until);
    return hipSuccess;
}

hipError_t hipEventCreate(hipEvent_t *e) { *e = reinterpret_cast<hipEvent_t>(new Event{current, true, Clock::now()}); return hipSuccess; }
hipError_t hipEventCreateWithFlags(hipEvent_t *e, unsigned) { return hipEventCreate(e); }
hipError_t hipEventDestroy(hipEvent_t e) { event_of(e)->live = false; return hipSuccess; }
hipError_t hipEventRecord(hipEvent_t e, hipStream_t s)
{
    if (!event_of(e)->live || !stream_of(s)->live)
        return fail(hipErrorInvalidHandle, "record of or on what was destroyed");
    if (event_of(e)->device != stream_of(s)->device)
        return fail(hipErrorInvalidHandle, "event recorded on a stream of another device");
    std::lock_guard<std::mutex> lk(mu);
    event_of(e)->done = stream_of(s)->idle;
    return hipSuccess;
}
hipError_t hipEventQuery(hipEvent_t e)
{
    if (!event_of(e)->live)
        return fail(hipErrorInvalidHandle, "query of an event that was destroyed");
    std::lock_guard<std::mutex> lk(mu);
    return Clock::now() < event_of(e)->done ? hipErrorNotReady : hipSuccess;
}
hipError_t hipEventSynchronize(hipEvent_t e) { std::this_thread::sleep_until(event_of(e)->done); return hipSuccess; }
hipError_t hipEventElapsedTime(float *ms, hipEvent_t a, hipEvent_t b)
{
    if (!event_of(a)->live || !event_of(b)->live)
        return fail(hipErrorInvalidHandle, "time between events that were destroyed");
    *ms = 1.0f;
    return hipSuccess;
}
hipError_t hipMemsetAsync(void *p, int v, size_t n, hipStream_t) { memset(p, v, n); return hipSuccess; }
hipError_t hipMemcpyAsync(void *to, const void *from, size_t n, hipMemcpyKind, hipStream_t) { memcpy(to, from, n); return hipSuccess; }

hipError_t hipLaunchKernel(const void *f, dim3, dim3, void **args, size_t, hipStream_t s)
{
    const std::string &name = kernels()[f];
    if (!stream_of(s)->live || stream_of(s)->device != current)
        return fail(hipErrorInvalidHandle, "launch on a stream of another device, or one that was destroyed");
    if (name.find("move_segments") == std::string::npos && pretend)
        return pretend(name, args) ? hipSuccess : fail(hipErrorOutOfMemory, "a launch is refused");
    if (name.find("move_segments") == std::string::npos)
        return fail(hipErrorInvalidValue, ("no such kernel here: " + name).c_str());
    struct Segments { char *dev[12]; uint32_t at[12], bytes[12]; int n; };
    const Segments &p = *static_cast<const Segments *>(args[0]);
    char *pinned = *static_cast<char **>(args[1]);
    for (int i = 0; i < p.n; ++i) {
        if (!on_device(p.dev[i], p.bytes[i], current))
            return fail(hipErrorInvalidValue, "a copy touches memory that is not the device's");
        if (name.find("ILb1E") != std::string::npos)
            memcpy(p.dev[i], pinned + p.at[i], p.bytes[i]);
        else
            memcpy(pinned + p.at[i], p.dev[i], p.bytes[i]);
    }
    return hipSuccess;
}

}  // extern "C"

// from now on the device has something to do
static void busy(int ms)
{
    for (Stream *s : streams)
        s->idle = Clock::now() + std::chrono::milliseconds(ms);
}
static double ms_since(Clock::time_point t) { return std::chrono::duration<double, std::milli>(Clock::now() - t).count(); }

#define REQUIRE(what)                                                                               \
    do {                                                                                            \
        if (!(what)) {                                                                              \
            fprintf(stderr, "line %d: %s (%s)\n", __LINE__, #what, comet_hip_last_error());         \
            return 1;                                                                               \
        }                                                                                           \
    } while (0)

static int there_and_back(size_t bytes, size_t offset)
{
    std::vector<unsigned char> out(bytes), in(bytes, 0);
    for (size_t i = 0; i < bytes; ++i)
        out[i] = (unsigned char)(i * 2654435761u >> 11);
    const int64_t d = comet_hip_malloc((int64_t)(bytes + offset));
    REQUIRE(d != 0);
    REQUIRE(comet_hip_memcpy(d + (int64_t)offset, out.data(), (int64_t)bytes, 0) == 0);
    REQUIRE(comet_hip_memcpy(d + (int64_t)offset, in.data(), (int64_t)bytes, 1) == 0);
    REQUIRE(in == out);
    REQUIRE(comet_hip_free(d) == 0);
    return 0;
}

// the library closed on one device and opened on another
static int another_device()
{
    for (int device : {0, 1, 0}) {
        REQUIRE(comet_hip_init(device) == 0);
        double ms = 0.0;
        REQUIRE(comet_hip_timer_start() == 0 && comet_hip_timer_stop(&ms) == 0 && ms > 0.0);
        for (size_t bytes : {100ul, 700ul << 10, 30ul << 20})
            REQUIRE(there_and_back(bytes, 0) == 0);
        REQUIRE(comet_hip_finalize() == 0);
    }
    return 0;
}

// what fits the device can be had, whatever is kept or rounded
static int whole_device()
{
    const int64_t GiB = 1ll << 30;
    REQUIRE(comet_hip_init(0) == 0);
    for (int turn = 0; turn < 2; ++turn) {
        const int64_t a = comet_hip_malloc(130 * GiB), b = comet_hip_malloc(130 * GiB), c = comet_hip_malloc(20 * GiB),
                      d = comet_hip_malloc(7 * GiB);
        REQUIRE(a && b && c && d);
        for (int64_t p : {a, b, c, d})
            REQUIRE(comet_hip_free(p) == 0);
        const int64_t e = comet_hip_malloc(260 * GiB), f = comet_hip_malloc(27 * GiB + 12345);
        REQUIRE(e && f);
        REQUIRE(comet_hip_malloc(GiB) == 0);
        const int64_t rest = (int64_t)(total[0] - used[0]);          // to the last page
        const int64_t g = comet_hip_malloc(rest - rest % 4096);
        REQUIRE(g);
        for (int64_t p : {e, f, g})
            REQUIRE(comet_hip_free(p) == 0);
    }
    return 0;
}

// freed memory that is kept can be had back for others, and so can memory of a device that the library has left
static int given_back()
{
    REQUIRE(comet_hip_init(0) == 0);
    const size_t before = used[0];
    const int64_t a = comet_hip_malloc(5ll << 30), b = comet_hip_malloc(1000);
    REQUIRE(a && b);
    REQUIRE(comet_hip_free(a) == 0);
    REQUIRE(used[0] >= before + (5ull << 30));
    REQUIRE(comet_hip_release_memory() == 0);
    REQUIRE(used[0] >= before + 1000 && used[0] < before + (1ull << 20));
    REQUIRE(comet_hip_free(b) == 0);
    REQUIRE(comet_hip_release_memory() == 0);
    REQUIRE(used[0] == before);
    return 0;
}

// memory that was had on a device the library has left is given back to that device, not handed out on another
static int block_of_another_device()
{
    REQUIRE(comet_hip_init(0) == 0);
    const int64_t kept = comet_hip_malloc(3 << 20);
    REQUIRE(kept);
    REQUIRE(comet_hip_finalize() == 0);
    REQUIRE(comet_hip_init(1) == 0);
    REQUIRE(comet_hip_free(kept) == 0);
    REQUIRE(there_and_back(3 << 20, 0) == 0);
    REQUIRE(comet_hip_finalize() == 0);
    REQUIRE(used[0] == 0 && used[1] == 0);
    return 0;
}

// one thread waits for the device, another one wants memory
static int memory_while_another_waits()
{
    REQUIRE(comet_hip_init(0) == 0);
    std::vector<char> host(100);
    const int64_t a = comet_hip_malloc(100), b = comet_hip_malloc(5000);
    REQUIRE(a && b);
    for (bool pending : {false, true}) {
        if (pending)
            REQUIRE(comet_hip_free(b) == 0);
        int rc = -1;
        busy(1500);
        const auto t0 = Clock::now();
        std::thread waits([&] { rc = comet_hip_memcpy(a, host.data(), 100, 0); });
        std::this_thread::sleep_for(std::chrono::milliseconds(300));
        const int64_t c = comet_hip_malloc(pending ? 3 << 20 : 1 << 20);
        REQUIRE(c && comet_hip_free(c) == 0);
        const double ms = ms_since(t0);
        waits.join();
        REQUIRE(rc == 0 && ms_since(t0) >= 1490);
        REQUIRE(ms < 1200);
    }
    // what was freed while that thread waited is not free to hand out: the work launched before may use it
    busy(0);
    const int64_t d = comet_hip_malloc(70000);
    REQUIRE(d);
    busy(900);
    std::thread waits([&] { (void)comet_hip_memcpy(a, host.data(), 100, 0); });
    std::this_thread::sleep_for(std::chrono::milliseconds(300));
    busy(2000);                                     // launched after that wait began
    REQUIRE(comet_hip_free(d) == 0);
    waits.join();
    const auto t0 = Clock::now();
    const int64_t e = comet_hip_malloc(70000);
    REQUIRE(e && (e != d || ms_since(t0) > 300));
    return 0;
}

// a copy that has to wait for the device does not keep the CPUs busy meanwhile
static int waiting_is_cheap()
{
    REQUIRE(comet_hip_init(0) == 0);
    const int64_t bytes = 40 << 20;
    std::vector<char> host((size_t)bytes, 1);
    const int64_t d = comet_hip_malloc(bytes);
    REQUIRE(d);
    const auto cpu_ms = [] {
        rusage u;
        getrusage(RUSAGE_SELF, &u);
        return (double)(u.ru_utime.tv_sec + u.ru_stime.tv_sec) * 1e3 + (double)(u.ru_utime.tv_usec + u.ru_stime.tv_usec) / 1e3;
    };
    for (int64_t n : {bytes, (int64_t)1000})
        for (int direction : {0, 1, 0, 1}) {
            REQUIRE(comet_hip_memcpy(d, host.data(), n, direction) == 0);          // what it costs with an idle device
            const double c0 = cpu_ms();
            REQUIRE(comet_hip_memcpy(d, host.data(), n, direction) == 0);
            const double c1 = cpu_ms();
            busy(600);
            const auto t0 = Clock::now();
            REQUIRE(comet_hip_memcpy(d, host.data(), n, direction) == 0);
            REQUIRE(ms_since(t0) >= 590);
            REQUIRE(cpu_ms() - c1 <= 3 * (c1 - c0) + 150);
        }
    return 0;
}

// a process that may have no more threads still copies
static int few_threads(int n)
{
    REQUIRE(comet_hip_init(0) == 0);
    threads_left = n;
    for (int i = 0; i < 3; ++i)
        REQUIRE(there_and_back(30 << 20, 8) == 0);
    threads_left = 1 << 20;
    REQUIRE(there_and_back(30 << 20, 8) == 0);
    return 0;
}

// a masked product of which one row is a workgroup's, drawn by ticket, and one a wavefront's, whose launch is refused: the
// tickets are as they were for the next product
static unsigned long long *tickets_drawn = nullptr;
static bool refuse_light = false;
static bool masked_product_kernels(const std::string &kernel, void **args)
{
    const auto is = [&](const char *name) { return kernel.find(name) != std::string::npos; };
    const auto at = [&](int i) { return *static_cast<int64_t **>(args[i]); };
    if (is("coo_flag"))
        std::fill_n(at(4), *static_cast<int64_t *>(args[0]), 1);
    if (is("scan_one")) {
        int64_t sum = 0;
        for (int i = 0; i < *static_cast<int *>(args[1]); ++i) {
            at(2)[i] = sum;
            sum += at(0)[i];
        }
        at(2)[*static_cast<int *>(args[1])] = sum;
    }
    if (is("pair_parts")) {
        at(10)[0] = 1;
        at(10)[1] = 1ll << 32;
    }
    if (is("pair_dot_heavy")) {
        tickets_drawn = *static_cast<unsigned long long **>(args[6]);
        tickets_drawn[0] += 2;
    }
    if (is("pair_dot_light")) {
        unsigned long long *cleared = *static_cast<unsigned long long **>(args[2]);
        if (cleared && !refuse_light)
            cleared[0] = 0;
        return !refuse_light;
    }
    return true;
}
static int refused_launch()
{
    REQUIRE(comet_hip_init(0) == 0);
    pretend = masked_product_kernels;
    const int64_t pos[] = {0, 3, 6, 9}, crd[] = {0, 1, 2, 0, 1, 2, 0, 1, 2};
    const double val[] = {1, 2, 3, 4, 5, 6, 7, 8, 9};
    const int64_t a = comet_hip_csr_upload_i64(3, 3, pos, crd, val);
    REQUIRE(a != 0);
    for (bool refused : {false, true, false}) {
        refuse_light = refused;
        tickets_drawn = nullptr;
        const int64_t c = comet_hip_spgemm_csr(a, a, a);
        REQUIRE(tickets_drawn && (c == 0) == refused);
        REQUIRE(tickets_drawn[0] == 0);
        REQUIRE(refused || comet_hip_csr_destroy(c) == 0);
    }
    return 0;
}

int main(int, char **argv)
{
    const std::string what = argv[1];
    if (what == "another_device")
        return another_device();
    if (what == "whole_device")
        return whole_device();
    if (what == "given_back")
        return given_back();
    if (what == "block_of_another_device")
        return block_of_another_device();
    if (what == "memory_while_another_waits")
        return memory_while_another_waits();
    if (what == "waiting_is_cheap")
        return waiting_is_cheap();
    if (what == "no_threads")
        return few_threads(0);
    if (what == "two_threads")
        return few_threads(2);
    if (what == "refused_launch")
        return refused_launch();
    fprintf(stderr, "no scenario %s\n", argv[1]);
    return 2;
}
