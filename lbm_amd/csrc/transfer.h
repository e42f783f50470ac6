// Arrays of the caller's ordinary (pageable) memory from and to device memory.
#pragma once

#include <cstddef>
#include <mutex>

#include "ctx.h"

namespace lbm_host {

// A piece of a device range: bytes at offset, at host in the caller's memory (nullptr: not wanted).
struct HostPart {
    void* host;
    size_t offset, bytes;
};

// Copies the parts of the device range that starts at dev, in stream order, and returns when they are
// there.  Parts are in ascending order and do not overlap.
int copy_out(lbm_ctx* c, const void* dev, const HostPart* parts, int n);
// The other way; returns when the caller's arrays have been read.  The parts cover the range.
int copy_in(lbm_ctx* c, void* dev, const HostPart* parts, int n);

// Page-locked memory of at least 64 KiB, which kernels may write and the host reads, the calling thread's while this
// lives: what a kernel leaves there needs no copy.  p is nullptr if there is none.  Taken when nothing is queued on the
// context's stream, so that others do not wait for its steps.
struct HostResults {
    explicit HostResults(const lbm_ctx* c);
    HostResults(const HostResults&) = delete;
    void* p = nullptr;

private:
    std::unique_lock<std::mutex> lock;
};

// The page-locked buffers that the copies go through and the threads that take part belong to the device: they come
// with the first copy that needs them and are gone when the call for its last context returns.
void transfer_retain(int device);
void transfer_release(int device);

}  // namespace lbm_host
