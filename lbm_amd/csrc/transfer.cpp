// The runtime copies device memory to pageable memory through a buffer of its own, one piece after the
// other on the calling thread, which also takes the page faults of an array that is written for the
// first time: 13-15 GB/s measured on MI355X, where the link itself carries about 50.  Here the copy
// engine fills or empties page-locked slots while several threads do the other side.
// Measured with 8 threads and 2 MiB slots, FP32 384x192x128: moments (154 MB) 15.6 -> 4.5 ms, a D3Q27
// record (1.04 GB) out 97 -> 26.5 ms, in 35 -> 27 ms.  What fits one slot takes one copy on the calling
// thread, also where it goes to several arrays (60x14x5 moments 123 -> 38 us), and spares the runtime's
// page-locking of the caller's array on the way in (60x14x5 record 340 -> 70 us).  The first copies through a
// new pool cost up to 2.3 ms more, as its pages are touched (equilibrium start of 112x84x70 cells, 22 MB in: 3.4
// ms, 1.1 ms from then on; the runtime's copies 1.6 and 1.1 ms).  Slots of 1 MiB halve that, but made a readout
// of 154 MB 0.8 ms slower.
#include "transfer.h"

#include <hip/hip_runtime.h>

#include <algorithm>
#include <atomic>
#include <condition_variable>
#include <cstring>
#include <exception>
#include <mutex>
#include <new>
#include <thread>

namespace lbm_host {

namespace {

constexpr size_t kSlot = 2u << 20;   // bytes of a slot
constexpr int kWorkers = 8;          // threads of a large copy, two slots each

std::mutex g_mu;                     // one copy at a time: the link is one
std::mutex g_users_mu;
int g_users = 0;
char* g_slots = nullptr;             // 2 * kWorkers slots (guarded by g_mu)

struct Job {
    lbm_ctx* c;
    char* dev;
    const HostPart* parts;
    int np;
    bool in;             // host to device
    size_t total, chunks;
    int threads;
    std::atomic<size_t> next{0};
    std::atomic<int> error{hipSuccess};
};

// The threads that take part in large copies beside the calling one.  They stay until the last context goes and
// are joined then: nothing of a thread outlives its contexts.  A copy does not wait for a thread that wakes late
// (other threads of the process may keep all processors busy): it finds the job gone.  Threads started and
// joined by each copy made copies of 16 MB slower than the runtime's beside a spinning OpenMP team.  Never
// destroyed: a program may exit with contexts alive, whose threads then still wait here.
struct Team {
    std::thread th[kWorkers - 1];
    int started = 0;             // guarded by g_mu
    std::mutex mu;
    std::condition_variable wake, idle;
    Job* job = nullptr;
    unsigned long long turn = 0;
    int active = 0;
    bool stop = false;
};
Team& team() {
    alignas(Team) static unsigned char place[sizeof(Team)];
    static Team* const t = new (place) Team;
    return *t;
}

// Everything of the device range's chunk k that a part holds or wants, from or to the slot.
void move_host(const Job& j, size_t k, char* slot) {
    const size_t o = k * kSlot, n = std::min(kSlot, j.total - o);
    for (int q = 0; q < j.np; ++q) {
        const HostPart& p = j.parts[q];
        if (!p.host) continue;
        const size_t lo = std::max(o, p.offset), hi = std::min(o + n, p.offset + p.bytes);
        if (lo >= hi) continue;
        char* h = static_cast<char*>(p.host) + (lo - p.offset);
        if (j.in) std::memcpy(slot + (lo - o), h, hi - lo);
        else std::memcpy(h, slot + (lo - o), hi - lo);
    }
}

hipError_t move_device(const Job& j, size_t k, char* slot) {
    const size_t o = k * kSlot, n = std::min(kSlot, j.total - o);
    if (j.in) return hipMemcpyAsync(j.dev + o, slot, n, hipMemcpyHostToDevice, j.c->stream);
    return hipMemcpyAsync(slot, j.dev + o, n, hipMemcpyDeviceToHost, j.c->stream);
}

// One thread's share: a chunk is on the link in one of its slots while it fills or empties the other.
void work(Job& j, int w) {
    auto bad = [&](hipError_t e) {
        if (e == hipSuccess) return false;
        j.error.store((int)e);
        return true;
    };
    hipEvent_t ev[2] = {nullptr, nullptr};
    for (hipEvent_t& e : ev)
        if (bad(hipEventCreateWithFlags(&e, hipEventDisableTiming))) break;
    size_t held[2] = {0, 0};
    bool busy[2] = {false, false};
    auto slot = [&](int s) { return g_slots + (size_t)(2 * w + s) * kSlot; };
    auto finish = [&](int s) {   // the slot's copy has ended, and what it brought is with the caller
        if (!busy[s]) return;
        busy[s] = false;
        if (!bad(hipEventSynchronize(ev[s])) && !j.in) move_host(j, held[s], slot(s));
    };
    int s = 0;
    while (ev[1] && j.error.load() == hipSuccess) {
        const size_t k = j.next.fetch_add(1);
        if (k >= j.chunks) break;
        if (j.in) {
            finish(s);
            move_host(j, k, slot(s));
        }
        if (bad(move_device(j, k, slot(s))) || bad(hipEventRecord(ev[s], j.c->stream))) break;
        busy[s] = true;
        held[s] = k;
        s ^= 1;
        if (!j.in) finish(s);
    }
    finish(s);
    finish(s ^ 1);
    for (hipEvent_t e : ev)
        if (e) (void)hipEventDestroy(e);
}

void member(Team* t, int w) {
    unsigned long long seen = 0;
    std::unique_lock<std::mutex> lk(t->mu);
    for (;;) {
        t->wake.wait(lk, [&] { return t->stop || (t->job && t->turn != seen); });
        if (t->stop) return;
        seen = t->turn;
        Job& j = *t->job;
        if (w >= j.threads) continue;
        ++t->active;
        lk.unlock();
        // (a thread that cannot take the device leaves its chunks to the others)
        if (hipSetDevice(j.c->device) == hipSuccess) work(j, w);
        lk.lock();
        if (--t->active == 0) t->idle.notify_all();
    }
}

// The job by up to j.threads threads, this one among them.  g_mu is held.
void work_together(Job& j) {
    Team& t = team();
    try {
        for (; t.started < j.threads - 1; ++t.started) t.th[t.started] = std::thread(member, &t, t.started + 1);
    } catch (const std::exception&) {
        // fewer threads than wanted: the others take their chunks
    }
    {
        std::lock_guard<std::mutex> lk(t.mu);
        t.job = &j;
        ++t.turn;
    }
    t.wake.notify_all();
    work(j, 0);
    std::unique_lock<std::mutex> lk(t.mu);
    t.job = nullptr;   // nobody joins any more
    t.idle.wait(lk, [&] { return t.active == 0; });
}

// g_mu is held: no copy is under way.
void dismiss() {
    Team& t = team();
    {
        std::lock_guard<std::mutex> lk(t.mu);
        t.stop = true;
    }
    t.wake.notify_all();
    for (; t.started > 0; --t.started) t.th[t.started - 1].join();
    t.stop = false;
}

// The context's device is the calling thread's current one while this lives, and the caller's own again afterwards.
struct OnDevice {
    int mine = -1, own = -1;
    hipError_t error;
    explicit OnDevice(int d) : mine(d) {
        error = hipGetDevice(&own);
        if (error == hipSuccess && own != mine) error = hipSetDevice(mine);
    }
    ~OnDevice() {
        if (own >= 0 && own != mine) (void)hipSetDevice(own);
    }
};

int copy(lbm_ctx* c, char* dev, const HostPart* parts, int n, bool in) {
    Job j;
    j.c = c;
    j.dev = dev;
    j.parts = parts;
    j.np = n;
    j.in = in;
    j.total = 0;
    for (int q = 0; q < n; ++q)
        if (parts[q].host) j.total = std::max(j.total, parts[q].offset + parts[q].bytes);
    const OnDevice on(c->device);
    HIPCHK(c, on.error);
    // what is queued ends before the slots are taken: others' copies do not wait for this context's steps
    HIPCHK(c, hipStreamSynchronize(c->stream));
    if (j.total == 0) return LBM_OK;
    std::lock_guard<std::mutex> lk(g_mu);
    if (!g_slots && hipHostMalloc((void**)&g_slots, 2 * kWorkers * kSlot, hipHostMallocPortable) != hipSuccess) {
        // no page-locked memory: straight from and to the caller's arrays
        g_slots = nullptr;
        (void)hipGetLastError();
        for (int q = 0; q < n; ++q) {
            char* d = dev + parts[q].offset;
            if (!parts[q].host) continue;
            if (in) HIPCHK(c, hipMemcpyAsync(d, parts[q].host, parts[q].bytes, hipMemcpyHostToDevice, c->stream));
            else HIPCHK(c, hipMemcpyAsync(parts[q].host, d, parts[q].bytes, hipMemcpyDeviceToHost, c->stream));
        }
        HIPCHK(c, hipStreamSynchronize(c->stream));
        return LBM_OK;
    }
    j.chunks = (j.total + kSlot - 1) / kSlot;
    if (j.chunks == 1) {
        if (in) move_host(j, 0, g_slots);
        HIPCHK(c, move_device(j, 0, g_slots));
        HIPCHK(c, hipStreamSynchronize(c->stream));
        if (!in) move_host(j, 0, g_slots);
        return LBM_OK;
    }
    // a thread costs about as much as emptying a slot: one for every two chunks
    j.threads = (int)std::min<size_t>(kWorkers, (j.chunks + 1) / 2);
    work_together(j);
    if (j.error.load() != hipSuccess) {
        (void)hipStreamSynchronize(c->stream);   // nothing still uses the slots
        return hipfail(c, (hipError_t)j.error.load(), in ? "copy to the device" : "copy to the host");
    }
    return LBM_OK;
}

}  // namespace

void transfer_retain() {
    std::lock_guard<std::mutex> lk(g_users_mu);
    ++g_users;
}

void transfer_release() {
    std::lock_guard<std::mutex> lk(g_users_mu);
    if (--g_users > 0) return;
    std::lock_guard<std::mutex> lk2(g_mu);
    dismiss();
    if (g_slots) (void)hipHostFree(g_slots);
    g_slots = nullptr;
}

int copy_out(lbm_ctx* c, const void* dev, const HostPart* parts, int n) {
    return copy(c, const_cast<char*>(static_cast<const char*>(dev)), parts, n, false);
}

int copy_in(lbm_ctx* c, void* dev, const HostPart* parts, int n) { return copy(c, static_cast<char*>(dev), parts, n, true); }

}  // namespace lbm_host
