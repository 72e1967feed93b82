// Scratch memory of bulk calls, shared by all tables of the process.
//
// A bulk call leases one buffer for the kernels it launches. The lease ends
// with the call, and an event is recorded behind the call's kernels. A buffer
// is handed out again to a call on the same stream, or once that event has
// passed: no stream ever waits for another one's work here, calls on several
// streams or host threads get buffers of their own. Bounded: at most
// kWorkspaceLimit bytes per device; a lease that would exceed it, or that
// finds no device memory, is empty and the caller runs its kernels that need
// no scratch; so does one that would leave less device memory free than it
// takes. Given back: the buffers are freed when the process's last table is
// destroyed, by trim(), where a table's own allocation finds too little memory
// (device_malloc, device_memory_for), and before the bound or the device's
// memory would refuse a larger lease.
//
// Not for calls under stream capture: a graph would keep the buffer's address
// beyond the lease. Beside a capture of another stream the pool allocates and
// frees in the relaxed capture mode, so that the capture stays valid.
#pragma once

#include "base.hpp"

#include <mutex>
#include <new>

namespace warpcore {
namespace detail {

constexpr std::size_t kWorkspaceLimit = std::size_t(16) << 30;
constexpr std::size_t kWorkspaceUnit = std::size_t(1) << 20;   // leases are rounded up to this

class WorkspacePool {
public:
    static WorkspacePool& instance() noexcept {
        // never destroyed: tables may outlive static objects
        alignas(WorkspacePool) static unsigned char place[sizeof(WorkspacePool)];
        static WorkspacePool* pool = ::new (static_cast<void*>(place)) WorkspacePool;
        return *pool;
    }

    struct Buffer {
        void* p = nullptr;
        std::size_t bytes = 0;
        int device = 0;
        hipEvent_t done = nullptr;   // behind the last user's kernels
        hipStream_t stream = nullptr;   // the last user's
        bool leased = false;
        Buffer* next = nullptr;
    };

    WC_H void add_user() noexcept {
        std::lock_guard<std::mutex> lock(mu_);
        ++users_;
    }
    WC_H void remove_user() noexcept {
        std::lock_guard<std::mutex> lock(mu_);
        if (--users_ != 0) return;
        const RelaxedCapture relaxed;
        free_idle(-1);
    }

    // a buffer of at least `bytes` on the current device whose earlier use is
    // over or ordered before what `stream` is given next; null without one
    WC_H Buffer* acquire(std::size_t bytes, hipStream_t stream) noexcept {
        bytes = (bytes + kWorkspaceUnit - 1) / kWorkspaceUnit * kWorkspaceUnit;
        int device = 0;
        if (bytes > kWorkspaceLimit || hipGetDevice(&device) != hipSuccess) return nullptr;
        std::lock_guard<std::mutex> lock(mu_);
        const RelaxedCapture relaxed;
        Buffer* best = nullptr;
        for (Buffer* b = first_; b != nullptr; b = b->next)
            if (!b->leased && b->device == device && b->bytes >= bytes &&
                (best == nullptr || b->bytes < best->bytes) && (ordered(b, stream) || passed(b)))
                best = b;
        if (best != nullptr) {
            // (nothing to wait for unless the handle was given to a new stream)
            if (hipStreamWaitEvent(stream, best->done, 0) != hipSuccess) {
                (void)hipGetLastError();
                return nullptr;
            }
            best->leased = true;
            return best;
        }
        if (held_on(device) + bytes > kWorkspaceLimit) {
            free_idle(device);
            if (held_on(device) + bytes > kWorkspaceLimit) return nullptr;
        }
        Buffer* b = new (std::nothrow) Buffer;
        if (b == nullptr) return nullptr;
        b->bytes = bytes;
        b->device = device;
        if (hipEventCreateWithFlags(&b->done, hipEventDisableTiming) != hipSuccess) {
            (void)hipGetLastError();
            delete b;
            return nullptr;
        }
        if (available_gpu_memory() / 2 < bytes) free_idle(device);
        if (available_gpu_memory() / 2 < bytes || hipMalloc(&b->p, bytes) != hipSuccess) {
            (void)hipGetLastError();
            (void)hipEventDestroy(b->done);
            delete b;
            return nullptr;
        }
        b->leased = true;
        b->next = first_;
        first_ = b;
        return b;
    }
    WC_H void release(Buffer* b, hipStream_t stream) noexcept {
        std::lock_guard<std::mutex> lock(mu_);
        const RelaxedCapture relaxed;
        if (hipEventRecord(b->done, stream) != hipSuccess) {
            (void)hipGetLastError();
            (void)hipStreamSynchronize(stream);   // no event to wait for: the kernels end here
        }
        b->stream = stream;
        b->leased = false;
        if (users_ == 0) free_idle(-1);
    }
    // frees the buffers no call holds, after waiting for the kernels that
    // still use them; the bytes freed, on all devices
    WC_H std::size_t trim() noexcept {
        std::lock_guard<std::mutex> lock(mu_);
        const RelaxedCapture relaxed;
        const std::size_t before = held_on(-1);
        free_idle(-1);
        return before - held_on(-1);
    }
    // bytes held on all devices
    WC_H std::size_t bytes_held() noexcept {
        std::lock_guard<std::mutex> lock(mu_);
        return held_on(-1);
    }

private:
    WC_H static bool ordered(const Buffer* b, hipStream_t stream) noexcept {
        return b->stream == stream && !per_thread_stream(stream);
    }
    WC_H static bool passed(const Buffer* b) noexcept {
        const hipError_t e = hipEventQuery(b->done);
        if (e != hipSuccess && hipPeekAtLastError() == e) (void)hipGetLastError();
        return e == hipSuccess;
    }
    // bytes of one device's buffers, or (-1) of all
    WC_H std::size_t held_on(int device) const noexcept {
        std::size_t held = 0;
        for (const Buffer* b = first_; b != nullptr; b = b->next)
            if (device < 0 || b->device == device) held += b->bytes;
        return held;
    }
    // frees the buffers not leased: one device's whose last use is over, or
    // (-1) all, after waiting for the kernels that still use them
    WC_H void free_idle(int device) noexcept {
        for (Buffer** at = &first_; *at != nullptr;) {
            Buffer* b = *at;
            if (b->leased || (device >= 0 && (b->device != device || !passed(b)))) {
                at = &b->next;
                continue;
            }
            *at = b->next;
            (void)hipEventSynchronize(b->done);
            (void)hipFree(b->p);
            (void)hipEventDestroy(b->done);
            delete b;
        }
    }

    std::mutex mu_;
    Buffer* first_ = nullptr;   // linked in the buffers themselves: a lease allocates nothing that may throw
    std::size_t users_ = 0;
};

// Allocations of the tables themselves, before which idle scratch memory goes
// back: whether the device has `bytes` free, and hipMalloc.
WC_H bool device_memory_for(std::size_t bytes) noexcept {
    return available_gpu_memory() >= bytes ||
           (WorkspacePool::instance().trim() != 0 && available_gpu_memory() >= bytes);
}
template<class T>
WC_H hipError_t device_malloc(T** p, std::size_t bytes) noexcept {
    const hipError_t e = hipMalloc(reinterpret_cast<void**>(p), bytes);
    if (e == hipSuccess || WorkspacePool::instance().trim() == 0) return e;
    (void)hipGetLastError();
    return hipMalloc(reinterpret_cast<void**>(p), bytes);
}

// One bulk call's lease; false when the pool has no buffer for it.
class WorkspaceLease {
public:
    WC_H WorkspaceLease(std::size_t bytes, hipStream_t stream) noexcept
        : buffer_(WorkspacePool::instance().acquire(bytes, stream)), stream_(stream) {}
    WorkspaceLease(const WorkspaceLease&) = delete;
    WorkspaceLease& operator=(const WorkspaceLease&) = delete;
    WC_H ~WorkspaceLease() noexcept {
        if (buffer_ != nullptr) WorkspacePool::instance().release(buffer_, stream_);
    }
    explicit operator bool() const noexcept { return buffer_ != nullptr; }
    void* get() const noexcept { return buffer_ != nullptr ? buffer_->p : nullptr; }

private:
    WorkspacePool::Buffer* buffer_;
    hipStream_t stream_;
};

}  // namespace detail
}  // namespace warpcore
