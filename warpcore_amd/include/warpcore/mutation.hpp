// Who may modify a table while a bulk insert rewrites it.
//
// The partitioned inserts (partition.hpp) write whole regions of a table
// back with plain stores, so nothing else may modify the table meanwhile;
// every other path claims slots by compare-and-swap and runs beside anything.
// MutationTracker decides which of the two a bulk call takes:
//
// - Every bulk call that modifies the table notes its stream. A call may run
//   exclusively while all of them used that one stream, which then orders
//   them. A second stream, a call under capture (its graph may be replayed at
//   any time), a handle of the per-thread default stream (one handle, many
//   streams: per_thread_stream), and a copy or a view of the table handed out
//   (user kernels may modify the table through the device calls) end that;
//   the calls that follow use the compare-and-swap paths.
// - An exclusive call leaves an event and a mark (CompletionMark) behind its
//   kernels. A later modifying call on another stream waits for the event on
//   the device, and handing out a copy or a view, or noting a call under
//   capture, waits for the mark on the host. So does a call whose wait for
//   the event is refused: that of a stream that is captured by then.
// - init() starts over (it fills the whole table, so a modification still
//   running on another stream would be a race with it already), except for
//   copies, views and graphs, which stay.
#pragma once

#include "base.hpp"
#include "workspace.hpp"

#include <atomic>
#include <mutex>
#include <new>

namespace warpcore {
namespace detail {

class MutationTracker {
    struct State {
        std::atomic<unsigned> holders{1};   // host objects
        std::mutex mu;
        bool any = false;      // `stream` is the one that ordered every modification so far
        bool mixed = false;    // more than one stream since the last init()
        bool shared = false;   // a copy, a view or a graph may modify the table
        hipStream_t stream = nullptr;
        hipEvent_t fence = nullptr;   // behind the last exclusive call
        CompletionMark end;           // the same for the host
        bool fenced = false;
        hipStream_t fence_stream = nullptr;
    };

public:
    WC_H MutationTracker() noexcept : s_(new (std::nothrow) State) {}
    // a shallow copy of the table shares the state, which lives as long as the
    // last of them on the host (a copy may be copied after its table is gone)
    WC_HD MutationTracker(const MutationTracker& o) noexcept : s_(o.s_) {
        hold();
        share();
    }
    WC_H MutationTracker(MutationTracker&& o) noexcept : s_(o.s_) { hold(); }
    MutationTracker& operator=(const MutationTracker&) = delete;
    WC_HD ~MutationTracker() noexcept {
#if !defined(__HIP_DEVICE_COMPILE__)
        if (s_ == nullptr || s_->holders.fetch_sub(1, std::memory_order_acq_rel) != 1) return;
        if (s_->fence != nullptr) (void)hipEventDestroy(s_->fence);
        delete s_;
#endif
    }

    WC_HD void share() const noexcept {
#if !defined(__HIP_DEVICE_COMPILE__)
        if (s_ == nullptr) return;
        std::lock_guard<std::mutex> lock(s_->mu);
        share_locked();
#endif
    }
    WC_H void restart() const noexcept {
        if (s_ == nullptr) return;
        std::lock_guard<std::mutex> lock(s_->mu);
        s_->any = false;
        s_->mixed = false;
    }
    // a modification on `stream` that runs beside others
    WC_H void note(hipStream_t stream) const noexcept {
        if (s_ == nullptr) return;
        std::lock_guard<std::mutex> lock(s_->mu);
        (void)note_locked(stream);
    }

    // One exclusive call: granted() says whether the kernels enqueued while
    // this object lives may assume that nothing else modifies the table.
    // Modifying calls of other host threads wait until it is gone.
    class Exclusive {
    public:
        WC_H Exclusive(const MutationTracker& t, hipStream_t stream) noexcept : s_(t.s_), stream_(stream) {
            if (s_ == nullptr) return;
            s_->mu.lock();
            granted_ = t.note_locked(stream);
            if (granted_ && s_->fence == nullptr &&
                hipEventCreateWithFlags(&s_->fence, hipEventDisableTiming) != hipSuccess) {
                (void)hipGetLastError();
                s_->fence = nullptr;
                granted_ = false;
            }
        }
        Exclusive(const Exclusive&) = delete;
        Exclusive& operator=(const Exclusive&) = delete;
        WC_H ~Exclusive() noexcept {
            if (s_ == nullptr) return;
            if (used_) {
                s_->fenced = true;
                s_->fence_stream = stream_;
                if (hipEventRecord(s_->fence, stream_) != hipSuccess) {   // nothing to wait for on the device
                    (void)hipGetLastError();
                    wait(*s_);
                }
            }
            s_->mu.unlock();
        }
        bool granted() const noexcept { return granted_; }
        void use(const CompletionMark& end) noexcept {   // exclusive kernels were enqueued, which `end` is behind
            used_ = true;
            s_->end = end;
        }

    private:
        State* s_;
        hipStream_t stream_;
        bool granted_ = false, used_ = false;
    };

private:
    WC_HD void hold() const noexcept {
#if !defined(__HIP_DEVICE_COMPILE__)
        if (s_ != nullptr) s_->holders.fetch_add(1, std::memory_order_relaxed);
#endif
    }
    WC_H void share_locked() const noexcept {
        s_->shared = true;
        wait(*s_);
    }
    // the host waits for the last exclusive call's kernels
    WC_H static void wait(State& s) noexcept {
        if (s.fenced) s.end.wait();
        s.fenced = false;
    }
    // whether `stream` orders every modification
    WC_H bool note_locked(hipStream_t stream) const noexcept {
        hipStreamCaptureStatus capture = hipStreamCaptureStatusNone;
        if (hipStreamIsCapturing(stream, &capture) != hipSuccess || capture != hipStreamCaptureStatusNone) {
            (void)hipGetLastError();
            share_locked();
            return false;
        }
        if (s_->fenced && s_->end.passed()) s_->fenced = false;
        if (s_->fenced && s_->fence_stream != stream && hipStreamWaitEvent(stream, s_->fence, 0) != hipSuccess) {
            (void)hipGetLastError();
            wait(*s_);
        }
        if (per_thread_stream(stream) || (s_->any && s_->stream != stream)) s_->mixed = true;
        s_->any = true;
        s_->stream = stream;
        return !s_->mixed && !s_->shared;
    }

    State* s_;
};

}  // namespace detail
}  // namespace warpcore
