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
#include <memory>
#include <mutex>
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
    std::atomic<size_t> next{0};
    std::atomic<int> error{hipSuccess};
    // threads that take part; none joins any more once the calling thread has run out of chunks
    std::mutex mu;
    std::condition_variable idle;
    int active = 0;
    bool closed = false;
};

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
    if (bad(hipSetDevice(j.c->device))) return;
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

// A thread of the team.  One that the system starts late (other threads of the process may keep all
// processors busy) finds the job closed, and nobody waits for it: joined threads made copies of 16 MB
// slower than the runtime's beside a spinning OpenMP team.
void join_in(std::shared_ptr<Job> j, int w) {
    {
        std::lock_guard<std::mutex> lk(j->mu);
        if (j->closed) return;
        ++j->active;
    }
    work(*j, w);
    std::lock_guard<std::mutex> lk(j->mu);
    if (--j->active == 0) j->idle.notify_all();
}

int copy(lbm_ctx* c, char* dev, const HostPart* parts, int n, bool in) {
    const std::shared_ptr<Job> job = std::make_shared<Job>();
    Job& j = *job;
    j.c = c;
    j.dev = dev;
    j.parts = parts;
    j.np = n;
    j.in = in;
    j.total = 0;
    for (int q = 0; q < n; ++q)
        if (parts[q].host) j.total = std::max(j.total, parts[q].offset + parts[q].bytes);
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
    const int threads = (int)std::min<size_t>(kWorkers, (j.chunks + 1) / 2);
    try {
        for (int w = 1; w < threads; ++w) std::thread(join_in, job, w).detach();
    } catch (const std::exception&) {
        // fewer threads than wanted: the others take their chunks
    }
    work(j, 0);
    {
        std::unique_lock<std::mutex> lk(j.mu);
        j.closed = true;
        j.idle.wait(lk, [&] { return j.active == 0; });
    }
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
    if (g_slots) (void)hipHostFree(g_slots);
    g_slots = nullptr;
}

int copy_out(lbm_ctx* c, const void* dev, const HostPart* parts, int n) {
    return copy(c, const_cast<char*>(static_cast<const char*>(dev)), parts, n, false);
}

int copy_in(lbm_ctx* c, void* dev, const HostPart* parts, int n) { return copy(c, static_cast<char*>(dev), parts, n, true); }

}  // namespace lbm_host
