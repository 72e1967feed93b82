// Scratch memory of bulk calls, shared by all tables of the process.
//
// A bulk call leases one buffer for the kernels it launches. The lease ends
// with the call, whose last kernel writes a mark that the host can read. A buffer
// is handed out again to a call on the same stream, or once that mark is
// there: no stream ever waits for another one's work here, calls on several
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
#include <thread>

namespace warpcore {

namespace kernels {

// Behind a call's other kernels: they are over. (Their writes reached memory
// when they ended; the store alone is for the host.)
__global__ inline void complete(std::uint64_t* word, std::uint64_t seq) {
    __hip_atomic_store(word, seq, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_SYSTEM);
}

}  // namespace kernels

namespace detail {

// The end of some kernels, as the host reads it without a call to the runtime:
// a query of an event, or a wait for one, ends a capture of the stream on which
// the event was recorded, however long before.
struct CompletionMark {
    std::uint64_t* word = nullptr;   // in pinned host memory; it only grows
    std::uint64_t seq = 0;

    WC_H bool passed() const noexcept { return word == nullptr || __atomic_load_n(word, __ATOMIC_ACQUIRE) >= seq; }
    WC_H void wait() const noexcept {
        while (!passed()) std::this_thread::yield();
    }
};

constexpr unsigned kMarkWords = 512;   // of 8 bytes; as many buffers at once at most
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
        CompletionMark done;         // behind the last user's kernels
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
                (best == nullptr || b->bytes < best->bytes) && (ordered(b, stream) || b->done.passed()))
                best = b;
        if (best != nullptr) {
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
        b->done.word = take_word();
        if (b->done.word != nullptr) b->done.seq = *b->done.word;
        if (available_gpu_memory() / 2 < bytes) free_idle(device);
        if (b->done.word == nullptr || available_gpu_memory() / 2 < bytes || hipMalloc(&b->p, bytes) != hipSuccess) {
            (void)hipGetLastError();
            give_word(b->done.word);
            delete b;
            return nullptr;
        }
        b->leased = true;
        b->next = first_;
        first_ = b;
        return b;
    }
    // the end of the kernels enqueued on `stream` so far
    WC_H CompletionMark release(Buffer* b, hipStream_t stream) noexcept {
        std::lock_guard<std::mutex> lock(mu_);
        const RelaxedCapture relaxed;
        ++b->done.seq;
        void* args[] = {&b->done.word, &b->done.seq};
        if (hipLaunchKernel(reinterpret_cast<const void*>(kernels::complete), dim3(1), dim3(1), args, 0, stream) !=
            hipSuccess) {
            (void)hipGetLastError();
            (void)hipStreamSynchronize(stream);   // nobody to write the mark: the kernels end here
            __atomic_store_n(b->done.word, b->done.seq, __ATOMIC_RELEASE);
        }
        b->stream = stream;
        b->leased = false;
        const CompletionMark done = b->done;
        if (users_ == 0) free_idle(-1);
        return done;
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
    // (destroying a stream waits for its work on this runtime, so a new stream
    // that is given an old one's handle is ordered behind it too)
    WC_H static bool ordered(const Buffer* b, hipStream_t stream) noexcept {
        return b->stream == stream && !per_thread_stream(stream);
    }
    // a word of the marks' memory, allocated with the first; null when all are in use
    WC_H std::uint64_t* take_word() noexcept {
        if (words_ == nullptr) {
            if (hipHostMalloc(reinterpret_cast<void**>(&words_), kMarkWords * sizeof(std::uint64_t),
                              hipHostMallocPortable | hipHostMallocCoherent) != hipSuccess) {
                (void)hipGetLastError();
                words_ = nullptr;
                return nullptr;
            }
            for (unsigned w = 0; w < kMarkWords; ++w) words_[w] = 0;
        }
        for (unsigned w = 0; w < kMarkWords; ++w)
            if (!taken_[w]) {
                taken_[w] = true;
                return words_ + w;
            }
        return nullptr;
    }
    WC_H void give_word(std::uint64_t* word) noexcept {
        if (word != nullptr) taken_[word - words_] = false;
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
            if (b->leased || (device >= 0 && (b->device != device || !b->done.passed()))) {
                at = &b->next;
                continue;
            }
            *at = b->next;
            b->done.wait();
            (void)hipFree(b->p);
            give_word(b->done.word);
            delete b;
        }
    }

    std::mutex mu_;
    std::uint64_t* words_ = nullptr;   // marks; kept: trackers read theirs after the buffer is gone
    bool taken_[kMarkWords] = {};
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

// One bulk call's lease; false when the pool has no buffer for it. `end` (may
// be null) becomes the mark behind the call's kernels.
class WorkspaceLease {
public:
    WC_H WorkspaceLease(std::size_t bytes, hipStream_t stream, CompletionMark* end = nullptr) noexcept
        : buffer_(WorkspacePool::instance().acquire(bytes, stream)), stream_(stream), end_(end) {}
    WorkspaceLease(const WorkspaceLease&) = delete;
    WorkspaceLease& operator=(const WorkspaceLease&) = delete;
    WC_H ~WorkspaceLease() noexcept {
        if (buffer_ == nullptr) return;
        const CompletionMark done = WorkspacePool::instance().release(buffer_, stream_);
        if (end_ != nullptr) *end_ = done;
    }
    explicit operator bool() const noexcept { return buffer_ != nullptr; }
    void* get() const noexcept { return buffer_ != nullptr ? buffer_->p : nullptr; }

private:
    WorkspacePool::Buffer* buffer_;
    hipStream_t stream_;
    CompletionMark* end_;
};

}  // namespace detail
}  // namespace warpcore
