// The runtime copies device memory to pageable memory through a buffer of its own, one piece after the
// other on the calling thread, which also takes the page faults of an array that is written for the
// first time: 13-15 GB/s measured on MI355X, where the link itself carries about 50.  Here the copy
// engine fills or empties page-locked slots while several threads do the other side.
// Measured with 2 MiB slots, FP32 384x192x128, the runtime's copies -> these: moments (154 MB) 15.6 -> 4.2 ms, a
// D3Q27 record (1.04 GB) out 97 -> 26.4 ms, in 35 -> 26.8 ms.  What fits one slot takes one copy on the calling
// thread, also where it goes to several arrays (60x14x5 moments 123 -> 38 us), and spares the runtime's page-locking
// of the caller's array on the way in (60x14x5 record 340 -> 70 us).
// Slots are page-locked when a copy first needs them, and no more of them: at most 22 MiB a device.  The
// equilibrium start of a program's only context of 112x84x70 cells (23 MB in, 8 MiB of slots) takes 1.9 ms and its
// later copies 0.7 ms (the runtime's copies 1.6 and 1.1 ms; with 32 MiB at the first copy 2.0 to 3.2 ms); its first
// moments 0.7 ms (the runtime's 1.5).  Slots of 1 MiB made a readout of 154 MB 0.8 ms slower.
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
// Threads of a large copy, two slots each: one for every two chunks, as a thread costs about as much as emptying a
// slot, up to two into the device and five out of it.  Measured on MI355X, ms with 1, 2, 4, 5 and 8: into the device
// 312 MB 12.4, 9.1, 9.1, 9.2, 9.2 (6 MB 0.32 and 0.27 with 1 and 2); out of it into new arrays, whose pages come with
// the first write, 156 MB 13.0, 7.7, 4.9, 4.8, 4.9 (into arrays that have their pages 6.1, 4.3, 4.3, 4.3, 4.3), 1.04 GB
// 26.5, 26.4, 26.5 with 4, 5 and 8 (32 with 3).
constexpr int kWorkers = 5, kWorkersIn = 2;

struct Job {
    lbm_ctx* c;
    char* dev;
    const HostPart* parts;   // one after the other
    int np;
    bool in;             // host to device
    size_t first, total, chunks;   // of the device range: where the parts start, their bytes
    int threads;
    std::atomic<size_t> next{0};
    std::atomic<int> error{hipSuccess};
};

// The threads that take part in large copies beside the calling one.  They stay until the device's last context
// goes and are joined then: nothing of a thread outlives its contexts.  A copy does not wait for a thread that wakes
// late (other threads of the process may keep all processors busy): it finds the job gone.  Threads started and
// joined by each copy made copies of 16 MB slower than the runtime's beside a spinning OpenMP team.
struct Team {
    std::thread th[kWorkers - 1];
    int started = 0;             // guarded by Pool::mu
    std::mutex mu;
    std::condition_variable wake, idle;
    Job* job = nullptr;
    unsigned long long turn = 0;
    int active = 0;
    bool stop = false;
};

// What the copies of one device share.  One large copy at a time: the device's link is one, and another device's
// copies have their own.  A copy that fits a slot goes beside a large one and does not wait for it.
struct Pool {
    std::mutex mu;
    char* slots[2 * kWorkers] = {};
    int pairs = 0;               // threads that there are slots for
    char* blocks[kWorkers] = {}; // what the slots lie in
    int nblocks = 0;
    Team team;
    std::mutex small_mu;
    char* small = nullptr;       // one slot
    std::atomic<int> users{0};   // contexts
};

// nullptr beyond the devices that have one.  Never destroyed: a program may exit with contexts alive, whose
// threads then still wait.
Pool* pool_of(int device) {
    constexpr int kDevices = 64;
    alignas(Pool) static unsigned char place[kDevices * sizeof(Pool)];
    static Pool* const pools = [] {
        for (int d = 0; d < kDevices; ++d) new (place + d * sizeof(Pool)) Pool;
        return reinterpret_cast<Pool*>(place);
    }();
    return device >= 0 && device < kDevices ? pools + device : nullptr;
}

// Chunk k of the parts, from or to the slot.
void move_host(const Job& j, size_t k, char* slot) {
    const size_t o = j.first + k * kSlot, n = std::min(kSlot, j.total - k * kSlot);
    for (int q = 0; q < j.np; ++q) {
        const HostPart& p = j.parts[q];
        const size_t lo = std::max(o, p.offset), hi = std::min(o + n, p.offset + p.bytes);
        if (lo >= hi) continue;
        char* h = static_cast<char*>(p.host) + (lo - p.offset);
        if (j.in) std::memcpy(slot + (lo - o), h, hi - lo);
        else std::memcpy(h, slot + (lo - o), hi - lo);
    }
}

hipError_t move_device(const Job& j, size_t k, char* slot) {
    const size_t o = j.first + k * kSlot, n = std::min(kSlot, j.total - k * kSlot);
    if (j.in) return hipMemcpyAsync(j.dev + o, slot, n, hipMemcpyHostToDevice, j.c->stream);
    return hipMemcpyAsync(slot, j.dev + o, n, hipMemcpyDeviceToHost, j.c->stream);
}

// One thread's share: a chunk is on the link in one of its slots while it fills or empties the other.
void work(Job& j, int w, char* const* slots) {
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
    auto slot = [&](int s) { return slots[2 * w + s]; };
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

void member(Pool* p, int w) {
    Team* const t = &p->team;
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
        if (hipSetDevice(j.c->device) == hipSuccess) work(j, w, p->slots);
        lk.lock();
        if (--t->active == 0) t->idle.notify_all();
    }
}

// The job by up to j.threads threads, this one among them.  p->mu is held.
void work_together(Pool* p, Job& j) {
    Team& t = p->team;
    try {
        for (; t.started < j.threads - 1; ++t.started) t.th[t.started] = std::thread(member, p, t.started + 1);
    } catch (const std::exception&) {
        // fewer threads than wanted: the others take their chunks
    }
    {
        std::lock_guard<std::mutex> lk(t.mu);
        t.job = &j;
        ++t.turn;
    }
    t.wake.notify_all();
    work(j, 0, p->slots);
    std::unique_lock<std::mutex> lk(t.mu);
    t.job = nullptr;   // nobody joins any more
    t.idle.wait(lk, [&] { return t.active == 0; });
}

// No copy is under way: its lock is held.
void dismiss(Team& t) {
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

// Memory of n bytes at p, allocated if there is none yet; false if there is none to be had.
bool page_locked(char*& p, size_t n) {
    if (!p && hipHostMalloc((void**)&p, n, hipHostMallocPortable) != hipSuccess) {
        p = nullptr;
        (void)hipGetLastError();
    }
    return p != nullptr;
}

// Threads that there are slots for, up to n; slots are added where there are fewer.  p->mu is held.
int with_slots(Pool* p, int n) {
    if (p->pairs < n && page_locked(p->blocks[p->nblocks], (size_t)2 * (n - p->pairs) * kSlot)) {
        char* const b = p->blocks[p->nblocks++];
        for (int s = 2 * p->pairs; s < 2 * n; ++s) p->slots[s] = b + (size_t)(s - 2 * p->pairs) * kSlot;
        p->pairs = n;
    }
    return std::min(n, p->pairs);
}

// The parts, one at a time, straight from and to the caller's arrays.
int straight(lbm_ctx* c, char* dev, const HostPart* parts, int n, bool in) {
    for (int q = 0; q < n; ++q) {
        char* d = dev + parts[q].offset;
        if (in) HIPCHK(c, hipMemcpyAsync(d, parts[q].host, parts[q].bytes, hipMemcpyHostToDevice, c->stream));
        else HIPCHK(c, hipMemcpyAsync(parts[q].host, d, parts[q].bytes, hipMemcpyDeviceToHost, c->stream));
    }
    HIPCHK(c, hipStreamSynchronize(c->stream));
    return LBM_OK;
}

// Parts that lie one after the other in the device range, through slots.
int staged(lbm_ctx* c, char* dev, const HostPart* parts, int n, bool in) {
    Job j;
    j.c = c;
    j.dev = dev;
    j.parts = parts;
    j.np = n;
    j.in = in;
    j.first = parts[0].offset;
    j.total = parts[n - 1].offset + parts[n - 1].bytes - j.first;
    if (j.total == 0) return LBM_OK;
    j.chunks = (j.total + kSlot - 1) / kSlot;
    Pool* const p = pool_of(c->device);
    if (p && j.chunks == 1) {
        std::lock_guard<std::mutex> lk(p->small_mu);
        if (page_locked(p->small, kSlot)) {
            if (in) move_host(j, 0, p->small);
            HIPCHK(c, move_device(j, 0, p->small));
            HIPCHK(c, hipStreamSynchronize(c->stream));
            if (!in) move_host(j, 0, p->small);
            return LBM_OK;
        }
    } else if (p) {
        std::lock_guard<std::mutex> lk(p->mu);
        j.threads = with_slots(p, (int)std::min<size_t>(in ? kWorkersIn : kWorkers, (j.chunks + 1) / 2));
        if (j.threads > 0) {
            work_together(p, j);
            if (j.error.load() != hipSuccess) {
                (void)hipStreamSynchronize(c->stream);   // nothing still uses the slots
                return hipfail(c, (hipError_t)j.error.load(), in ? "copy to the device" : "copy to the host");
            }
            return LBM_OK;
        }
    }
    return straight(c, dev, parts, n, in);   // no page-locked memory
}

// Whether the runtime knows the array: page-locked by the caller (or no ordinary memory at all).  From 256 KiB on: below,
// a copy of its own costs more than a slot's share (four fields of 22 KB 55 us straight, 36 us through one slot).
bool known(const HostPart& p) {
    if (p.bytes < (256u << 10)) return false;
    hipPointerAttribute_t a{};
    if (hipPointerGetAttributes(&a, p.host) != hipSuccess) {
        (void)hipGetLastError();
        return false;
    }
    return a.type != hipMemoryTypeUnregistered;
}

int copy(lbm_ctx* c, char* dev, const HostPart* parts, int n, bool in) {
    const OnDevice on(c->device);
    HIPCHK(c, on.error);
    // what is queued ends before the slots are taken: others' copies do not wait for this context's steps
    HIPCHK(c, hipStreamSynchronize(c->stream));
    // Arrays that the runtime knows are the copy engine's own end: a D3Q27 FP32 record of 384x192x128 (1.04 GB) 18.9 ms
    // out and 19.4 ms in where the slots take 26.4 and 27.0, its moments 3.1 and 4.3 ms.  The others go in runs
    // without a gap.
    for (int q = 0, e; q < n; q = e) {
        const HostPart* const r = parts + q;
        e = q + 1;
        if (!r->host) continue;
        const bool own = known(*r);
        while (e < n && parts[e].host && (own || parts[e].offset == parts[e - 1].offset + parts[e - 1].bytes) &&
               known(parts[e]) == own)
            ++e;
        const int rc = own ? straight(c, dev, r, e - q, in) : staged(c, dev, r, e - q, in);
        if (rc) return rc;
    }
    return LBM_OK;
}

}  // namespace

HostResults::HostResults(const lbm_ctx* c) {
    Pool* const pool = pool_of(c->device);
    if (!pool) return;
    lock = std::unique_lock<std::mutex>(pool->small_mu);
    if (page_locked(pool->small, kSlot)) p = pool->small;
}

void transfer_retain(int device) {
    if (Pool* p = pool_of(device)) ++p->users;
}

void transfer_release(int device) {
    Pool* const p = pool_of(device);
    if (!p || --p->users > 0) return;
    {
        std::lock_guard<std::mutex> lk(p->mu);
        if (p->users == 0) {   // (a context may have come meanwhile)
            dismiss(p->team);
            for (; p->nblocks > 0; --p->nblocks) {
                (void)hipHostFree(p->blocks[p->nblocks - 1]);
                p->blocks[p->nblocks - 1] = nullptr;
            }
            p->pairs = 0;
        }
    }
    std::lock_guard<std::mutex> lk(p->small_mu);
    if (p->users != 0) return;
    if (p->small) (void)hipHostFree(p->small);
    p->small = nullptr;
}

int copy_out(lbm_ctx* c, const void* dev, const HostPart* parts, int n) {
    return copy(c, const_cast<char*>(static_cast<const char*>(dev)), parts, n, false);
}

int copy_in(lbm_ctx* c, void* dev, const HostPart* parts, int n) { return copy(c, static_cast<char*>(dev), parts, n, true); }

}  // namespace lbm_host
