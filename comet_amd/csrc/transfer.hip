// Copies between host arrays of the caller and device memory.
//
// A copy from or to pageable memory goes through the runtime's own staging buffer with one thread filling it: 29 GB/s
// up and 18 GB/s down on a link that moves 57 GB/s either way from pinned memory.  Here four threads (107 GB/s) fill
// or empty pinned groups of up to four megabytes, and a kernel moves each group across the link - all the arrays of a
// call in the same groups - while the next one is filled.  (Link rate by size of the copy, DMA / kernel: 256 KiB
// 19 / 33 GB/s, 1 MiB 38 / 39, 4 MiB 50 / 52.)  What has to be done to the data anyway - narrowing 64-bit column
// numbers, looking whether they lie inside the matrix - is done on the way through.  Everything on the device is
// ordered on the library's stream.
#include <string.h>

#include <algorithm>
#include <atomic>
#include <chrono>
#include <condition_variable>
#include <functional>
#include <mutex>
#include <system_error>
#include <thread>

#include "common.h"

namespace comet {

namespace {

constexpr size_t SLOT = 4 << 20;           // pinned bytes of a group
constexpr int SLOTS = 3;                   // groups on their way
constexpr size_t UNIT = 256 << 10;         // bytes a thread fills or empties at a time
constexpr size_t ALONE = 512 << 10;        // transfers up to this size are not worth waking the other threads
constexpr int WORKERS = 4;                 // the caller's thread and three more
constexpr int MAX_SEGS = 12;               // parts of arrays in a group

struct Segments {
    char *dev[MAX_SEGS];
    uint32_t at[MAX_SEGS], bytes[MAX_SEGS];          // where the part lies in the group, as far from 16 bytes as in dev; its size
    int n;
};

// Sixteen bytes a lane wherever the device address lies: what is in front of the first and behind the last sixteen goes
// byte by byte.  (An array that did not begin at sixteen bytes went so as a whole: 64 KiB 34.8 us up and 21.2 down
// instead of 16.5, 64 MiB 1.45 and 1.60 ms instead of 1.38.)
template <bool UP>
__global__ __launch_bounds__(256) void move_segments(Segments p, char *pinned)
{
    typedef int v4i __attribute__((ext_vector_type(4)));
    const uint32_t t = blockIdx.x * blockDim.x + threadIdx.x, step = gridDim.x * blockDim.x;
    for (int i = 0; i < p.n; ++i) {
        char *dev = p.dev[i], *pin = pinned + p.at[i];
        const uint32_t bytes = p.bytes[i], before = -(uint32_t)(uintptr_t)dev & 15u, head = before < bytes ? before : bytes;
        const uint32_t units = (bytes - head) / 16;
        for (uint32_t u = t; u < units; u += step)
            if (UP)
                reinterpret_cast<v4i *>(dev + head)[u] = reinterpret_cast<const v4i *>(pin + head)[u];
            else
                reinterpret_cast<v4i *>(pin + head)[u] = reinterpret_cast<const v4i *>(dev + head)[u];
        for (uint32_t r = t; r < bytes - units * 16; r += step) {
            const uint32_t b = r < head ? r : r + units * 16;
            (UP ? dev : pin)[b] = (UP ? pin : dev)[b];
        }
    }
}

// The threads, parked between transfers, and the pinned slots.  Made at the first transfer; the threads are kept for
// the life of the process and take the device of each transfer, the slots and their events go with the device when
// the library is closed.
struct Crew {
    std::mutex mu;
    std::condition_variable start, done;
    uint64_t generation = 0;
    int running = 0, device = 0;
    const std::function<void()> *job = nullptr;
    char *pinned = nullptr;
    hipEvent_t moved[SLOTS];          // the last group in the slot is across
    int threads = 0;                  // how many have been made

    int prepare()
    {
        if (pinned)
            return COMET_HIP_OK;
        char *room = nullptr;
        COMET_HIPCHK(hipHostMalloc((void **)&room, SLOTS * SLOT, hipHostMallocDefault));
        for (hipEvent_t &e : moved)
            COMET_HIPCHK(hipEventCreateWithFlags(&e, hipEventDisableTiming));
        pinned = room;
        return COMET_HIP_OK;
    }
    void release()
    {
        if (!pinned)
            return;
        for (hipEvent_t e : moved)
            (void)hipEventDestroy(e);
        (void)hipHostFree(pinned);
        pinned = nullptr;
    }
    void loop(uint64_t seen)
    {
        int current = -1;
        for (;;) {
            const std::function<void()> *mine;
            int wanted;
            {
                std::unique_lock<std::mutex> lk(mu);
                start.wait(lk, [&] { return generation != seen; });
                seen = generation;
                mine = job;
                wanted = device;
            }
            if (wanted != current) {
                (void)hipSetDevice(wanted);
                current = wanted;
            }
            (*mine)();
            std::lock_guard<std::mutex> lk(mu);
            if (--running == 0)
                done.notify_one();
        }
    }
    // work on this thread and, unless alone, on the others
    void run(bool alone, const std::function<void()> &work)
    {
        if (!alone) {
            std::lock_guard<std::mutex> lk(mu);
            (void)hipGetDevice(&device);
            try {
                for (const uint64_t now = generation; threads < WORKERS - 1; ++threads)
                    std::thread([this, now] { loop(now); }).detach();
            } catch (const std::system_error &) {          // there are no more to be had: with those there are
            }
            job = &work;
            running = threads;
            ++generation;
            start.notify_all();
        }
        work();
        if (!alone) {
            std::unique_lock<std::mutex> lk(mu);
            done.wait(lk, [&] { return running == 0; });
        }
    }
};

std::mutex g_crew_mu;          // one transfer at a time: the next one's copies come after this one's on the stream anyway
Crew *g_crew = new Crew();     // never destroyed: its threads outlive main

// Asking again and again sees the end of a wait at once, and for as long as the copies of a call take - or the short
// product before a download: threads that have to be woken first cost it 60 us - that is worth four CPUs.  After ASKING
// the device is at something long, and naps of a thirtieth of the wait, a millisecond at most, do.
constexpr std::chrono::microseconds ASKING(1000), LONGEST_NAP(1000);
struct Waiting {
    std::chrono::steady_clock::time_point begin = std::chrono::steady_clock::now();
    void pause() const
    {
        const auto waited = std::chrono::steady_clock::now() - begin;
        if (waited > ASKING)
            std::this_thread::sleep_for(std::min<std::chrono::nanoseconds>(waited / 32, LONGEST_NAP));
    }
};

template <typename QUERY>
int wait_for(QUERY query)
{
    const Waiting waiting;
    hipError_t s;
    while ((s = query()) == hipErrorNotReady)
        waiting.pause();
    COMET_HIPCHK(s);
    return COMET_HIP_OK;
}

struct Unit {
    int group;
    const Piece *piece;
    size_t first, count, at;          // elements of the piece, and where they lie in the group
};

int transfer(const std::vector<Piece> &pieces, bool up)
{
    // cut into groups (the first ones smaller: the link starts sooner) and these into units
    std::vector<Segments> groups;
    std::vector<Unit> units;
    std::vector<int> units_in;
    size_t used = SLOT, limit = 0, total = 0;
    for (const Piece &p : pieces) {
        total += p.n * p.elem;
        for (size_t first = 0; first < p.n;) {
            if (used + UNIT > limit || groups.back().n == MAX_SEGS) {
                groups.push_back(Segments());
                groups.back().n = 0;
                units_in.push_back(0);
                used = 0;
                limit = std::min(SLOT, (1 << 20) * groups.size());
            }
            Segments &g = groups.back();
            g.dev[g.n] = (char *)p.dev + first * p.elem;
            const size_t at = used + ((uintptr_t)g.dev[g.n] & 15), count = std::min(p.n - first, (limit - at) / p.elem);
            g.at[g.n] = (uint32_t)at;
            g.bytes[g.n++] = (uint32_t)(count * p.elem);
            const size_t per = std::max<size_t>(1, UNIT / p.elem);
            for (size_t o = 0; o < count; o += per) {
                units.push_back(Unit{(int)groups.size() - 1, &p, first + o, std::min(per, count - o), at + o * p.elem});
                ++units_in.back();
            }
            used = (at + count * p.elem + 15) & ~(size_t)15;
            first += count;
        }
    }
    if (groups.empty())
        return COMET_HIP_OK;
    std::lock_guard<std::mutex> lk(g_crew_mu);
    Crew &crew = *g_crew;
    COMET_CHK(crew.prepare());
    const int ngroups = (int)groups.size();
    // state[g]: 0 not launched, 1 launched, 2 across
    std::vector<std::atomic<int>> state((size_t)ngroups), left((size_t)ngroups);
    for (int g = 0; g < ngroups; ++g) {
        state[(size_t)g] = 0;
        left[(size_t)g] = units_in[(size_t)g];
    }
    std::atomic<size_t> next{0};
    std::atomic<bool> failed{false};
    std::mutex asking;
    const auto launch = [&](int g) {
        const Segments &seg = groups[(size_t)g];
        char *pin = crew.pinned + (size_t)(g % SLOTS) * SLOT;
        const size_t bytes = seg.at[seg.n - 1] + seg.bytes[seg.n - 1];
        const dim3 grid((unsigned)std::min<size_t>(256, (bytes + 4095) / 4096));
        if (up)
            move_segments<true><<<grid, dim3(256), 0, stream()>>>(seg, pin);
        else
            move_segments<false><<<grid, dim3(256), 0, stream()>>>(seg, pin);
        if (hipGetLastError() != hipSuccess || hipEventRecord(crew.moved[g % SLOTS], stream()) != hipSuccess)
            failed = true;
        state[(size_t)g] = 1;
    };
    const auto wait_across = [&](int g) {          // one thread at a time asks the runtime
        const Waiting waiting;
        for (; state[(size_t)g] != 2 && !failed; waiting.pause())
            if (state[(size_t)g] == 1 && asking.try_lock()) {
                if (state[(size_t)g] == 1) {
                    const hipError_t e = hipEventQuery(crew.moved[g % SLOTS]);
                    if (e == hipSuccess)
                        state[(size_t)g] = 2;
                    else if (e != hipErrorNotReady)
                        failed = true;
                }
                asking.unlock();
            }
    };
    const std::function<void()> work = [&] {
        for (size_t u; !failed && (u = next++) < units.size();) {
            const Unit &t = units[u];
            char *pin = crew.pinned + (size_t)(t.group % SLOTS) * SLOT + t.at;
            if (up && t.group >= SLOTS)
                wait_across(t.group - SLOTS);
            if (!up)
                wait_across(t.group);
            if (failed)
                return;
            t.piece->host(pin, t.first, t.count);
            if (--left[(size_t)t.group] == 0) {
                if (up)
                    launch(t.group);
                else if (t.group + SLOTS < ngroups)
                    launch(t.group + SLOTS);
            }
        }
    };
    for (hipEvent_t e : crew.moved)          // the transfer before may still be reading the slots
        COMET_CHK(wait_for([&] { return hipEventQuery(e); }));
    if (!up)
        for (int g = 0; g < SLOTS && g < ngroups; ++g)
            launch(g);
    crew.run(total <= ALONE, work);
    if (failed)
        return set_error(COMET_HIP_ERR_HIP, "copying between host and device failed");
    return COMET_HIP_OK;
}

}  // namespace

int transfer_up(const std::vector<Piece> &pieces) { return transfer(pieces, true); }
int transfer_down(const std::vector<Piece> &pieces) { return transfer(pieces, false); }

void transfer_release()
{
    std::lock_guard<std::mutex> lk(g_crew_mu);
    g_crew->release();
}

Piece plain_up(void *dev, const void *host, size_t bytes)
{
    return Piece{dev, bytes, 1, [host](void *pin, size_t first, size_t count) {
                     memcpy(pin, (const char *)host + first, count);
                 }};
}

Piece plain_down(void *host, const void *dev, size_t bytes)
{
    return Piece{const_cast<void *>(dev), bytes, 1, [host](void *pin, size_t first, size_t count) {
                     memcpy((char *)host + first, pin, count);
                 }};
}

}  // namespace comet
