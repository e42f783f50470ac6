// CPU check of the copies to and from the caller's arrays (transfer.cpp), linked against the stand-in for the
// HIP runtime below: copies are memory copies on the calling thread, page-locked memory is ordinary memory that
// is counted, events and streams are names.
//
//   transfer_check <case>    prints one JSON line, exits 0 if the case holds
#include <hip/hip_runtime.h>

#include <algorithm>
#include <atomic>
#include <chrono>
#include <cstdio>
#include <cstdlib>
#include <cstring>
#include <functional>
#include <map>
#include <mutex>
#include <random>
#include <string>
#include <thread>
#include <vector>

#include "transfer.h"

using namespace lbm_host;

namespace {

// ---- the stand-in runtime
thread_local int t_device = 0;
std::atomic<int> g_threads_seen{0}, g_threads_ended{0};
struct ThreadState {   // what a runtime keeps per thread, released some time after the thread's function
    bool used = false;
    ~ThreadState() {
        if (!used) return;
        std::this_thread::sleep_for(std::chrono::milliseconds(100));
        ++g_threads_ended;
    }
};
thread_local ThreadState t_state;

std::mutex g_lock_mu;
std::map<void*, size_t> g_locked;
size_t g_locked_bytes = 0;
std::atomic<bool> g_no_lock{false};
std::atomic<int> g_fail_after{-1};   // copies until one fails; -1: none does
std::function<void(const void*, const void*, size_t)> g_on_copy;
const char* g_registered = nullptr;  // the caller's memory that the runtime knows
size_t g_registered_bytes = 0;

}  // namespace

extern "C" {
hipError_t hipSetDevice(int d) {
    if (!t_state.used) {
        t_state.used = true;
        ++g_threads_seen;
    }
    t_device = d;
    return hipSuccess;
}
hipError_t hipGetDevice(int* d) {
    *d = t_device;
    return hipSuccess;
}
hipError_t hipEventCreateWithFlags(hipEvent_t* e, unsigned) {
    *e = reinterpret_cast<hipEvent_t>(std::malloc(1));
    return hipSuccess;
}
hipError_t hipEventDestroy(hipEvent_t e) {
    std::free(e);
    return hipSuccess;
}
hipError_t hipEventRecord(hipEvent_t, hipStream_t) { return hipSuccess; }
hipError_t hipEventSynchronize(hipEvent_t) { return hipSuccess; }
hipError_t hipStreamSynchronize(hipStream_t) { return hipSuccess; }
hipError_t hipGetLastError() { return hipSuccess; }
hipError_t hipPointerGetAttributes(hipPointerAttribute_t* a, const void* p) {
    const char* q = static_cast<const char*>(p);
    std::memset(a, 0, sizeof *a);
    a->type = g_registered && q >= g_registered && q < g_registered + g_registered_bytes ? hipMemoryTypeHost
                                                                                         : hipMemoryTypeUnregistered;
    return hipSuccess;
}
const char* hipGetErrorString(hipError_t) { return "an error"; }
hipError_t hipMemcpyAsync(void* dst, const void* src, size_t n, hipMemcpyKind, hipStream_t) {
    if (g_on_copy) g_on_copy(dst, src, n);
    if (g_fail_after.load() >= 0 && g_fail_after.fetch_sub(1) == 0) return hipErrorUnknown;
    std::memcpy(dst, src, n);
    return hipSuccess;
}
hipError_t hipHostMalloc(void** p, size_t n, unsigned) {
    if (g_no_lock.load()) return hipErrorOutOfMemory;
    std::lock_guard<std::mutex> lk(g_lock_mu);
    *p = std::malloc(n);
    g_locked[*p] = n;
    g_locked_bytes += n;
    return hipSuccess;
}
hipError_t hipHostFree(void* p) {
    std::lock_guard<std::mutex> lk(g_lock_mu);
    g_locked_bytes -= g_locked[p];
    g_locked.erase(p);
    std::free(p);
    return hipSuccess;
}
}

namespace lbm_host {
int hipfail(lbm_ctx*, hipError_t, const char*) { return LBM_EHIP; }
}  // namespace lbm_host

namespace {

constexpr size_t kMB = 1u << 20;

template <class F>
bool until(F f) {
    for (int n = 0; n < 2000 && !f(); ++n) std::this_thread::sleep_for(std::chrono::milliseconds(1));
    return f();
}

std::vector<unsigned char> noise(size_t n, unsigned seed) {
    std::vector<unsigned char> v(n);
    std::mt19937_64 g(seed);
    for (size_t q = 0; q < n; q += 8) {
        const unsigned long long r = g();
        std::memcpy(&v[q], &r, std::min<size_t>(8, n - q));
    }
    return v;
}

// A range of `sizes` one after the other; part q is the caller's unless wanted says otherwise.  Out of the device
// and back in, with guards around every array.
bool round_trip(lbm_ctx* c, const std::vector<size_t>& sizes, unsigned seed, unsigned unwanted) {
    size_t total = 0;
    std::vector<HostPart> parts;
    std::vector<std::vector<unsigned char>> host;
    for (size_t s : sizes) {
        host.emplace_back(s + 128, (unsigned char)0xA5);
        parts.push_back({nullptr, total, s});
        total += s;
    }
    for (size_t q = 0; q < parts.size(); ++q)
        if (!(unwanted >> q & 1)) parts[q].host = host[q].data() + 64;
    std::vector<unsigned char> dev = noise(total, seed);
    const std::vector<unsigned char> before = dev;
    if (copy_out(c, dev.data(), parts.data(), (int)parts.size()) != LBM_OK || dev != before) return false;
    for (size_t q = 0; q < parts.size(); ++q) {
        const unsigned char* h = host[q].data();
        for (int g = 0; g < 64; ++g)
            if (h[g] != 0xA5 || h[64 + sizes[q] + g] != 0xA5) return false;
        if (parts[q].host) {
            if (std::memcmp(h + 64, before.data() + parts[q].offset, sizes[q]) != 0) return false;
        } else if (std::count(h + 64, h + 64 + sizes[q], 0xA5) != (long)sizes[q]) {
            return false;
        }
    }
    if (unwanted) return true;   // what goes in covers the range
    std::vector<unsigned char> to(total + 128, (unsigned char)0x5A);
    if (copy_in(c, to.data() + 64, parts.data(), (int)parts.size()) != LBM_OK) return false;
    for (int g = 0; g < 64; ++g)
        if (to[g] != 0x5A || to[64 + total + g] != 0x5A) return false;
    return std::memcmp(to.data() + 64, before.data(), total) == 0;
}

bool contents(lbm_ctx* c) {
    const std::vector<std::vector<size_t>> sets = {
        {1}, {100, 3, 7}, {2 * kMB}, {2 * kMB + 1}, {5 * kMB, 5 * kMB, 5 * kMB, 5 * kMB, 4},
        {kMB - 4, 3 * kMB + 4, 1}, {70 * kMB + 12345}, {0, 10}};
    for (size_t n = 0; n < sets.size(); ++n)
        for (unsigned unwanted : {0u, 1u, 2u, 5u})
            if (!round_trip(c, sets[n], (unsigned)n, unwanted)) return false;
    return true;
}

// every copy that fails is reported, and the next one is whole
bool errors(lbm_ctx* c) {
    std::vector<unsigned char> host(20 * kMB), dev = noise(host.size(), 3);
    for (size_t n : {kMB, 20 * kMB})
        for (int after : {0, 1, 3, 9}) {
            const HostPart part{host.data(), 0, n};
            if ((size_t)after * 2 * kMB >= n) continue;
            for (bool in : {false, true}) {
                g_fail_after = after;
                const int rc = in ? copy_in(c, dev.data(), &part, 1) : copy_out(c, dev.data(), &part, 1);
                g_fail_after = -1;
                if (rc != LBM_EHIP) return false;
            }
            if (!round_trip(c, {n}, 4, 0)) return false;
        }
    return true;
}

}  // namespace

int main(int argc, char** argv) {
    const std::string name = argc > 1 ? argv[1] : "";
    lbm_ctx c;
    bool ok = false;
    if (name == "contents") {
        transfer_retain(c.device);
        ok = contents(&c);
        transfer_release(c.device);
        ok = ok && g_locked_bytes == 0;
    } else if (name == "no_page_locked_memory") {
        g_no_lock = true;
        transfer_retain(c.device);
        ok = contents(&c);
        g_no_lock = false;
        ok = ok && contents(&c);
        transfer_release(c.device);
    } else if (name == "errors") {
        transfer_retain(c.device);
        ok = errors(&c);
        transfer_release(c.device);
    } else if (name == "device_of_the_caller") {
        // a context on another device than the calling thread's current one: the copies are made with its device
        // current, and the caller finds its own again
        c.device = 1;
        std::atomic<int> wrong{0};
        g_on_copy = [&](const void*, const void*, size_t) { wrong += t_device != 1; };
        transfer_retain(c.device);
        ok = true;
        for (size_t n : {kMB, 20 * kMB}) {
            t_device = 0;
            ok = ok && round_trip(&c, {n}, 6, 0) && t_device == 0;
        }
        transfer_release(c.device);
        ok = ok && wrong == 0 && t_device == 0;
    } else if (name == "devices_side_by_side") {
        // two threads read out contexts on two devices: each copy waits (for a bounded time) until the other is
        // under way
        lbm_ctx d;
        d.device = 1;
        transfer_retain(c.device);
        transfer_retain(d.device);
        std::atomic<unsigned> seen{0};
        std::atomic<bool> together{true};
        g_on_copy = [&](const void*, const void*, size_t) {
            seen |= 1u << t_device;
            if (!until([&] { return seen == 3u; })) together = false;
        };
        std::atomic<int> good{0};
        std::thread other([&] { good += round_trip(&d, {9 * kMB}, 7, 0); });
        good += round_trip(&c, {9 * kMB}, 8, 0);
        other.join();
        transfer_release(c.device);
        transfer_release(d.device);
        ok = good == 2 && together && g_locked_bytes == 0;
    } else if (name == "small_beside_large") {
        // a copy of one slot ends while a large one of the same device is held up
        transfer_retain(c.device);
        std::atomic<bool> large{false}, small{false}, first{true};
        g_on_copy = [&](const void*, const void*, size_t n) {
            if (n != 2 * kMB) return;
            large = true;
            if (!until([&] { return small.load(); })) first = false;
        };
        std::atomic<int> good{0};
        lbm_ctx d;
        std::thread other([&] {
            until([&] { return large.load(); });
            good += round_trip(&d, {kMB}, 7, 0);
            small = true;
        });
        good += round_trip(&c, {20 * kMB}, 8, 0);
        other.join();
        transfer_release(c.device);
        ok = good == 2 && first && g_locked_bytes == 0;
    } else if (name == "arrays_the_runtime_knows") {
        // large ones are the copies' own end, whole, whatever they stand beside; the others go through slots
        transfer_retain(c.device);
        ok = true;
        for (size_t n : {kMB / 4 - 1, kMB / 4, 7 * kMB}) {
            const int own_end = n >= kMB / 4;
            std::vector<unsigned char> own(n), dev = noise(3 * n + 4, 9), back(dev.size()), plain(2 * n + 4);
            g_registered = reinterpret_cast<const char*>(own.data());
            g_registered_bytes = n;
            const HostPart parts[4] = {{plain.data(), 0, n}, {own.data(), n, n}, {plain.data() + n, 2 * n, n},
                                       {plain.data() + 2 * n, 3 * n, 4}};
            std::atomic<int> direct{0}, pageable{0};
            g_on_copy = [&](const void* to, const void* from, size_t bytes) {
                for (const void* p : {to, from}) {
                    if (p == own.data() && bytes == n) ++direct;
                    if (p >= plain.data() && p < plain.data() + plain.size()) ++pageable;
                }
            };
            ok = ok && copy_out(&c, dev.data(), parts, 4) == LBM_OK && direct == own_end && pageable == 0;
            ok = ok && std::memcmp(own.data(), dev.data() + n, n) == 0 && std::memcmp(plain.data(), dev.data(), n) == 0 &&
                 std::memcmp(plain.data() + n, dev.data() + 2 * n, n + 4) == 0;
            ok = ok && copy_in(&c, back.data(), parts, 4) == LBM_OK && direct == 2 * own_end && pageable == 0 && back == dev;
        }
        transfer_release(c.device);
    } else if (name == "page_locked_by_need") {
        // one slot of 2 MiB for what fits one; two slots for each thread that a larger copy takes, the same for all
        // that follow; nothing without contexts
        ok = true;
        for (int rep = 0; rep < 2; ++rep) {
            size_t locked = 0;
            transfer_retain(c.device);
            for (size_t n : {kMB / 10, 2 * kMB}) {
                ok = ok && round_trip(&c, {n}, 10, 0);
                ok = ok && g_locked_bytes <= 2 * kMB;
            }
            ok = ok && round_trip(&c, {3 * kMB}, 11, 0) && g_locked_bytes <= 6 * kMB;
            ok = ok && round_trip(&c, {100 * kMB}, 12, 0);
            locked = g_locked_bytes;
            ok = ok && locked <= 22 * kMB && round_trip(&c, {70 * kMB, 3}, 13, 0) && g_locked_bytes == locked;
            transfer_release(c.device);
            ok = ok && g_locked_bytes == 0;
        }
        // into the device only
        std::vector<unsigned char> to(22 * kMB), from = noise(to.size(), 14);
        const HostPart part{from.data(), 0, from.size()};
        transfer_retain(c.device);
        ok = ok && copy_in(&c, to.data(), &part, 1) == LBM_OK && to == from && g_locked_bytes <= 8 * kMB;
        transfer_release(c.device);
    } else if (name == "threads_end") {
        // no thread that took part in a copy lives on after the last context, nor does its share of the runtime
        for (int n = 0; n < 3; ++n) {
            transfer_retain(c.device);
            ok = round_trip(&c, {32 * kMB}, 5, 0);
            transfer_release(c.device);
            if (t_state.used) g_threads_seen = g_threads_seen.load() - 1, t_state.used = false;   // the caller's own
            ok = ok && g_threads_ended == g_threads_seen;
            if (!ok) break;
        }
    }
    std::printf("{\"case\": \"%s\", \"ok\": %s, \"threads\": %d, \"ended\": %d, \"locked\": %zu}\n", name.c_str(),
                ok ? "true" : "false", g_threads_seen.load(), g_threads_ended.load(), g_locked_bytes);
    return ok ? 0 : 1;
}
