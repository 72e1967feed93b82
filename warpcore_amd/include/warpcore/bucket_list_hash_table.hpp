// BucketListHashTable: key -> growing list of value buckets. Drop-in for
// include/warpcore/bucket_list_hash_table.cuh with the value store
// storage::multi_value::BucketListStore (storage.cuh:656-1454).
//
// Keys live in a SingleValueHashTable<Key, handle>; a handle is one 64-bit
// word {state: 2 bits, bucket index, value count, values in the tail
// bucket} updated only by CAS/exchange. Values live in a pool of 8-byte
// cells handed out by atomicAdds on allocation counters. A key's first bucket holds
// min_bucket_size values and has no header; every later bucket is a header
// cell {previous bucket, bucket size} followed by its values, each bucket
// ceil(previous size * grow_factor) cells long, capped at max_bucket_size.
//
// Append (storage.cuh:1113-1284): an uninitialised handle or a full tail
// bucket is first switched to `blocking` by a CAS; the winner allocates the
// bucket, writes the value and publishes the new handle with an exchange;
// other appenders to the same key re-read the handle until it is no longer
// blocking. The winner's allocation path contains no wait, so a blocked
// handle is always released; the re-read loop is also bounded and returns
// unknown_error if that bound is ever reached. Otherwise the CAS bumps the
// count and the tail, and the winner stores the value in its cell.
//
// Allocation: the reference bumps one counter for the whole pool. Device
// atomics on one address are serialised at the memory side (12 ns each on
// MI355X, measured), which bounded inserts at 2.8 G values/s; so pools of
// at least 2^17 cells are cut into up to 256 arenas of at least 2^16 cells,
// each with its own counter on its own 128-byte line. A wavefront allocates
// from its home arena and moves on to the next ones when a request does not
// fit; an allocation fails (out_of_memory) only when it fits in none. A
// smaller pool is one arena and behaves exactly as the reference's.
//
// Values of a key come back tail bucket first (storage.cuh:1292-1345). A
// handle left `full` by an out-of-memory append still yields the values it
// holds; the reference yields none for it while reporting their count.
#pragma once

#include "base.hpp"
#include "defaults.hpp"
#include "engine.hpp"
#include "multi_value_hash_table.hpp"
#include "pair_groups.hpp"
#include "scan.hpp"
#include "single_value_hash_table.hpp"
#include "status.hpp"
#include "tile.hpp"

#include <algorithm>
#include <cmath>
#include <vector>

namespace warpcore {
namespace storage {
namespace multi_value {

namespace detail {

enum class LinkedListState : std::uint32_t { uninitialized = 0, initialized = 1, blocking = 2, full = 3 };

// One 64-bit word: state | index << 2 | count << (2 + IB) | tail << (2 + IB + CB).
template<index_t IB, index_t CB, index_t SB>
struct alignas(8) BucketListHandle {
    std::uint64_t pack;

    static constexpr std::uint64_t mask(index_t bits) noexcept {
        return bits >= 64 ? ~std::uint64_t(0) : (std::uint64_t(1) << bits) - 1;
    }
    WC_HD static constexpr index_t max_bucket_index() noexcept { return mask(IB); }
    WC_HD static constexpr index_t max_value_count() noexcept { return mask(CB); }
    WC_HD static constexpr index_t max_bucket_size() noexcept { return mask(SB); }

    WC_HD static constexpr BucketListHandle make(LinkedListState state, index_t index, index_t count,
                                                 index_t tail) noexcept {
        return BucketListHandle{std::uint64_t(state) | ((std::uint64_t(index) & mask(IB)) << 2) |
                                ((std::uint64_t(count) & mask(CB)) << (2 + IB)) |
                                ((std::uint64_t(tail) & mask(SB)) << (2 + IB + CB))};
    }
    WC_HD constexpr LinkedListState state() const noexcept { return LinkedListState(pack & 3); }
    WC_HD constexpr index_t bucket_index() const noexcept { return (pack >> 2) & mask(IB); }
    WC_HD constexpr index_t value_count() const noexcept { return (pack >> (2 + IB)) & mask(CB); }
    WC_HD constexpr index_t num_values_tail() const noexcept { return (pack >> (2 + IB + CB)) & mask(SB); }
    WC_HD constexpr bool is_uninitialized() const noexcept { return state() == LinkedListState::uninitialized; }
    WC_HD constexpr bool is_initialized() const noexcept { return state() == LinkedListState::initialized; }
    WC_HD constexpr bool is_blocking() const noexcept { return state() == LinkedListState::blocking; }
    WC_HD constexpr bool is_full() const noexcept { return state() == LinkedListState::full; }
};

// A pool cell: a value, or the header {previous bucket, bucket size} of a bucket.
template<class Value, index_t IB, index_t SB>
union alignas(alignof(Value) > 8 ? alignof(Value) : 8) Bucket {
    Value value;
    std::uint64_t info;

    WC_HD static constexpr std::uint64_t make_info(index_t previous, index_t size) noexcept {
        return (std::uint64_t(previous) & BucketListHandle<IB, 1, SB>::mask(IB)) |
               ((std::uint64_t(size) & BucketListHandle<IB, 1, SB>::mask(SB)) << IB);
    }
    WC_HD static constexpr index_t previous_of(std::uint64_t info) noexcept {
        return info & BucketListHandle<IB, 1, SB>::mask(IB);
    }
    WC_HD static constexpr index_t size_of(std::uint64_t info) noexcept {
        return (info >> IB) & BucketListHandle<IB, 1, SB>::mask(SB);
    }
};

// atomic_add(counter, n) of every active lane of the wavefront with one
// atomic: the lanes' amounts follow each other in lane order after the value
// the counter had. The counter ends where one atomic per lane would leave it
// and every lane's range lies below it exactly as one of those atomics would
// have placed some lane's; only which lane gets which range differs. (A bump
// allocator shared by the whole grid serialises its atomics at the memory
// side; this divides them by the lanes allocating together.)
WC_D index_t wave_atomic_add(index_t* counter, index_t n) noexcept {
    const std::uint64_t active = __builtin_amdgcn_read_exec();
    const unsigned lane = lane_id();
    index_t before = 0, total = 0;
    for (std::uint64_t m = active; m != 0; m &= m - 1) {
        const unsigned l = unsigned(__builtin_ctzll(m));
        const index_t v = (index_t(unsigned(__builtin_amdgcn_readlane(int(n >> 32), int(l)))) << 32) |
                          index_t(unsigned(__builtin_amdgcn_readlane(int(n), int(l))));
        if (l < lane) before += v;
        total += v;
    }
    const unsigned leader = unsigned(__builtin_ctzll(active));
    index_t base = 0;
    if (lane == leader) base = warpcore::detail::atomic_add(counter, total);
    base = (index_t(unsigned(__builtin_amdgcn_readlane(int(base >> 32), int(leader)))) << 32) |
           index_t(unsigned(__builtin_amdgcn_readlane(int(base), int(leader))));
    return base + before;
}

// Device half of the store, passed to kernels by value.
template<class Value, index_t IB, index_t CB, index_t SB>
struct BucketListStoreView {
    using handle_type = BucketListHandle<IB, CB, SB>;
    using bucket_type = Bucket<Value, IB, SB>;
    using value_type = Value;
    // re-reads of a blocked handle before an append gives up (unknown_error)
    static constexpr std::uint32_t kMaxBlockedReads = 1u << 24;

    bucket_type* buckets;
    index_t* counters;    // arena a's cells handed out: counters[a * kCounterStride]
    index_t capacity;
    float grow;
    index_t min_size;
    index_t max_size;
    index_t arenas;       // a power of two; every arena but the last holds arena_cells cells
    index_t arena_cells;

    static constexpr index_t kCounterStride = 16;   // 128 bytes between counters

    WC_HD index_t arena_begin(index_t a) const noexcept { return a * arena_cells; }
    WC_HD index_t arena_size(index_t a) const noexcept {
        return a + 1 < arenas ? arena_cells : capacity - a * arena_cells;
    }

    WC_D index_t home_arena() const noexcept {
        return arenas == 1 ? 0 : index_t(blockIdx.x * (blockDim.x >> 6) + (threadIdx.x >> 6)) & (arenas - 1);
    }

    // `n` cells for every active lane, from the wavefront's home arena or
    // the ones after it; the first cell, or ~0 when no arena holds them.
    // Active lanes take part together (a wave-uniform walk over the arenas).
    WC_D index_t allocate(index_t n) const noexcept {
        const index_t home = home_arena();
        for (index_t t = 0; t < arenas; ++t) {
            const index_t a = (home + t) & (arenas - 1);
            const index_t at = wave_atomic_add(counters + a * kCounterStride, n);
            if (at + n <= arena_size(a)) return arena_begin(a) + at;
        }
        return ~index_t(0);
    }

    WC_HD static constexpr index_t head() noexcept { return handle_type::max_bucket_index(); }

    // A new bucket's link (info word) read by appends must be visible
    // before the handle that points to it: an append that cannot size the
    // tail from the count (size_by_count) reads the tail's link with a
    // device-scope atomic load once it sees the handle. (Links that the
    // count sizes are read by later launches only and are plain stores.)
    // Both are written
    // with device-scope atomics, which the memory side performs; the link's
    // exchange returns its old word, and waiting for that word before the
    // handle's exchange is issued orders the two at the memory side for
    // every XCD. Values are plain stores, read only by later launches. (A
    // device-scope fence here writes back and invalidates the L2 of every
    // XCD: 2.3x the whole insert's time.)
    WC_D static void wait_for(std::uint64_t returned) noexcept {
        asm volatile("" ::"v"(unsigned(returned)) : "memory");
    }

    // Size of the bucket that holds value number c (c >= 1) of a key:
    // buckets follow one sequence (min_size, then each the previous one
    // grown by `grow`, at most max_size, computed as the allocation below
    // does), so it is found from the count without reading the bucket's link
    // when the sequence settles within kSizeSteps steps; false otherwise.
    static constexpr int kSizeSteps = 64;
    // counts and sizes of one key: 32 bits where the handle's fields allow
    // (the sequence is computed per append and per bucket walked)
    using small_type = typename std::conditional<(CB < 32 && SB < 32), std::uint32_t, index_t>::type;
    WC_D bool size_by_count(index_t count, index_t& size_out) const noexcept {
        const small_type c = small_type(count);
        small_type size = small_type(min_size), cum = size;
        for (int k = 0; k < kSizeSteps && cum < c; ++k) {
            const small_type next = grown(size);
            if (next == size) break;   // the same size from here on
            size = next;
            cum += size;
            if (k + 1 == kSizeSteps && cum < c) return false;
        }
        size_out = size;
        return true;
    }
    WC_D small_type grown(small_type size) const noexcept {
        return small_type(fminf(float(max_size), ceilf(float(size) * grow)));
    }

    WC_D Status append(handle_type* handle, const Value& value, index_t max_values_per_key) const noexcept {
        return append_from(handle, warpcore::detail::atomic_load_relaxed(&handle->pack), value, max_values_per_key);
    }

    // append with the handle as the caller read it (`seen`); a failed CAS
    // continues from the word it returned
    WC_D Status append_from(handle_type* handle, std::uint64_t seen, const Value& value,
                            index_t max_values_per_key) const noexcept {
        using warpcore::detail::atomic_cas;
        using warpcore::detail::atomic_exch;
        using LS = detail::LinkedListState;
        std::uint64_t* hp = &handle->pack;
        for (std::uint32_t reads = 0; reads < kMaxBlockedReads; ++reads) {
            const handle_type cur{seen};
            if (cur.is_blocking()) {   // another lane is linking a bucket: wait a little
                __builtin_amdgcn_s_sleep(1);
                seen = warpcore::detail::atomic_load_relaxed(hp);
                continue;
            }
            if (cur.is_uninitialized()) {
                const handle_type blocked = handle_type::make(LS::blocking, head(), 0, 0);
                seen = atomic_cas(hp, cur.pack, blocked.pack);
                if (seen != cur.pack) continue;
                const index_t alloc = allocate(min_size);
                if (alloc != ~index_t(0)) {
                    buckets[alloc].value = value;
                    atomic_exch(hp, handle_type::make(LS::initialized, alloc, 1, 1).pack);
                    return Status::none();
                }
                atomic_exch(hp, handle_type::make(LS::full, head(), 0, 0).pack);
                return Status::out_of_memory();
            }
            if (cur.is_full()) return Status::out_of_memory();
            if (cur.value_count() == max_values_per_key) return Status::max_values_for_key_reached();
            index_t tail_size = min_size;
            if (cur.value_count() > min_size && !size_by_count(cur.value_count(), tail_size))
                tail_size = bucket_type::size_of(warpcore::detail::atomic_load_relaxed(&buckets[cur.bucket_index()].info));
            if (cur.num_values_tail() == tail_size) {
                const handle_type blocked =
                    handle_type::make(LS::blocking, cur.bucket_index(), cur.value_count(), cur.num_values_tail());
                seen = atomic_cas(hp, cur.pack, blocked.pack);
                if (seen != cur.pack) continue;
                const index_t new_size = grown(tail_size);
                const index_t alloc = allocate(new_size + 1);
                if (alloc != ~index_t(0)) {
                    buckets[alloc + 1].value = value;
                    const std::uint64_t link = bucket_type::make_info(cur.bucket_index(), new_size);
                    index_t known = 0;
                    if (size_by_count(cur.value_count() + 1, known))
                        buckets[alloc].info = link;   // read only by later launches: a plain store
                    else
                        wait_for(atomic_exch(&buckets[alloc].info, link));   // appends will read this link
                    atomic_exch(hp, handle_type::make(LS::initialized, alloc, cur.value_count() + 1, 1).pack);
                    return Status::none();
                }
                atomic_exch(hp, handle_type::make(LS::full, cur.bucket_index(), cur.value_count(),
                                                  cur.num_values_tail())
                                    .pack);
                return Status::out_of_memory();
            }
            const handle_type next = handle_type::make(LS::initialized, cur.bucket_index(), cur.value_count() + 1,
                                                       cur.num_values_tail() + 1);
            seen = atomic_cas(hp, cur.pack, next.pack);
            if (seen == cur.pack) {
                const index_t j = cur.value_count() + 1 <= min_size ? cur.num_values_tail()
                                                                    : cur.num_values_tail() + 1;
                buckets[cur.bucket_index() + j].value = value;
                return Status::none();
            }
        }
        return Status::unknown_error();
    }

    // State of a handle that the calling lane holds blocked.
    struct Held {
        index_t bucket;
        small_type count, tail, size;   // size of the tail bucket, min_size while there is none
    };
    WC_D Held held(const handle_type& cur) const noexcept {
        Held h{head(), 0, 0, small_type(min_size)};
        if (cur.is_uninitialized()) return h;
        h.bucket = cur.bucket_index();
        h.count = small_type(cur.value_count());
        h.tail = small_type(cur.num_values_tail());
        index_t size = min_size;
        if (h.count > min_size && !size_by_count(h.count, size))
            size = bucket_type::size_of(warpcore::detail::atomic_load_relaxed(&buckets[h.bucket].info));
        h.size = small_type(size);
        return h;
    }
    WC_D static handle_type blocked(const handle_type& cur) noexcept {
        if (cur.is_uninitialized()) return handle_type::make(detail::LinkedListState::blocking, head(), 0, 0);
        return handle_type::make(detail::LinkedListState::blocking, cur.bucket_index(), cur.value_count(),
                                 cur.num_values_tail());
    }

    // The values next(value) gives (until it returns false; `pairs` of them)
    // appended to a held handle, buckets allocated and filled as append_from
    // does value by value, first from the `cells` cells from `run` on;
    // publishes the handle.
    template<class Next>
    WC_D Status fill(std::uint64_t* hp, Held h, const Next& next, small_type pairs, index_t max_values_per_key,
                     index_t run, std::uint32_t cells) const noexcept {
        using LS = detail::LinkedListState;
        Status st = Status::none();
        LS state = LS::initialized;
        const small_type most = small_type(max_values_per_key);
        const small_type first = small_type(min_size);
        index_t known = 0;
        const bool sized = size_by_count(index_t(h.count) + pairs, known);   // then every count before it is
        bucket_type* to = buckets + h.bucket + (h.count > first ? 1 : 0) + h.tail;   // the next value's cell
        small_type room = h.count == 0 ? 0 : h.size - h.tail;
        Value value{};
        while (next(value)) {
            if (h.count == most) {
                st = Status::max_values_for_key_reached();
                break;
            }
            if (room == 0) {
                const bool headed = h.count != 0;
                const small_type larger = headed ? grown(h.size) : first;
                const index_t need = index_t(larger) + (headed ? 1 : 0);
                index_t alloc = run;
                if (need <= cells) {
                    run += need;
                    cells -= std::uint32_t(need);
                } else {
                    alloc = allocate(need);
                }
                if (alloc == ~index_t(0)) {
                    st = Status::out_of_memory();
                    state = LS::full;
                    break;
                }
                to = buckets + alloc;
                if (headed) {
                    const std::uint64_t link = bucket_type::make_info(h.bucket, larger);
                    if (sized) to->info = link;   // read only by later launches: a plain store
                    else wait_for(warpcore::detail::atomic_exch(&to->info, link));   // appends will read this link
                    ++to;
                }
                h.bucket = alloc;
                h.size = room = larger;
            }
            to->value = value;
            ++to;
            --room;
            ++h.count;
        }
        const small_type tail = h.count == 0 ? 0 : h.size - room;
        warpcore::detail::atomic_exch(hp, handle_type::make(state, h.bucket, h.count, tail).pack);
        return st;
    }

    // Appends of several values to one handle, which is blocked once; returns
    // the flags that appends one by one would have joined. No lane waits for
    // another while it holds a handle: a blocked handle is always released.
    template<class Next>
    WC_D Status append_all(handle_type* handle, const Next& next, small_type pairs,
                           index_t max_values_per_key) const noexcept {
        std::uint64_t* hp = &handle->pack;
        std::uint64_t seen = warpcore::detail::atomic_load_relaxed(hp);
        for (std::uint32_t reads = 0; reads < kMaxBlockedReads; ++reads) {
            const handle_type cur{seen};
            if (cur.is_blocking()) {   // another lane is appending: wait a little
                __builtin_amdgcn_s_sleep(1);
                seen = warpcore::detail::atomic_load_relaxed(hp);
                continue;
            }
            if ((cur.is_uninitialized() ? 0 : cur.value_count()) >= max_values_per_key)
                return Status::max_values_for_key_reached();
            if (cur.is_full()) return Status::out_of_memory();
            seen = warpcore::detail::atomic_cas(hp, cur.pack, blocked(cur).pack);
            if (seen == cur.pack) return fill(hp, held(cur), next, pairs, max_values_per_key, 0, 0);
        }
        return Status::unknown_error();
    }

    // append_all of `pairs` values for every lane with `on`; all lanes of the
    // wavefront call this. The lanes that block their handle at the first
    // try have the cells of all their buckets allocated by one atomic, where
    // the wavefront's arena holds them (2^26 pairs over 2^23 keys: the groups
    // pass 3.65 ms, bucket by bucket, an atomic's round trip each, 4.07); the
    // others append on their own after those have published. A lane that would
    // take kMostCells cells or more takes them bucket by bucket, so that a
    // wavefront's sum fits 32 bits for any bucket sizes.
    // (`fresh`: the handle of a key just claimed, taken to be uninitialised.)
    static constexpr std::uint32_t kMostCells = 1u << 20, kWaveCells = 4096;
    template<class Next>
    WC_D Status append_wave(bool on, bool fresh, handle_type* handle, small_type pairs, const Next& next,
                            index_t max_values_per_key) const noexcept {
        Status st = Status::none();
        bool mine = false;
        Held h{head(), 0, 0, small_type(min_size)};
        if (on) {
            handle_type cur = handle_type::make(detail::LinkedListState::uninitialized, head(), 0, 0);
            if (!fresh) cur = handle_type{warpcore::detail::atomic_load_relaxed(&handle->pack)};
            if (!cur.is_blocking() && !cur.is_full() &&
                (cur.is_uninitialized() ? 0 : cur.value_count()) < max_values_per_key) {
                mine = warpcore::detail::atomic_cas(&handle->pack, cur.pack, blocked(cur).pack) == cur.pack;
                if (mine) h = held(cur);
            }
        }
        std::uint32_t cells = 0;
        if (mine) {
            bool headed = h.count != 0;
            small_type size = h.size, room = headed ? size - h.tail : 0;
            const small_type most = small_type(max_values_per_key) - h.count;
            small_type more = most < pairs ? most : pairs;
            while (more > room && cells < kMostCells) {
                more -= room;
                room = size = headed ? grown(size) : small_type(min_size);
                cells = size < kMostCells ? cells + std::uint32_t(size) + (headed ? 1 : 0) : kMostCells;
                headed = true;
            }
            if (cells >= kMostCells) cells = 0;
        }
        std::uint32_t upto = cells;
#pragma unroll
        for (unsigned s = 1; s < 64; s <<= 1) {
            const std::uint32_t o = __shfl_up(upto, s, 64);
            if (warpcore::lane_id() >= s) upto += o;
        }
        const std::uint32_t total = unsigned(__builtin_amdgcn_readlane(int(upto), 63));
        index_t run = ~index_t(0);
        if (total != 0) {   // uniform
            const index_t a = home_arena();
            if (warpcore::lane_id() == 0) {
                // A request that does not fit leaves the arena's last cells to
                // smaller ones, so near the end it is a compare-and-swap (an
                // add would move the counter past them; the counter only
                // grows, so the loop ends). Further off an add is safe: each
                // wavefront of this arena has one at most under way, of
                // kWaveCells at most (2^26 pairs over 2^23 keys: 5.51 ms, with
                // the swap alone 5.61).
                index_t* counter = counters + a * kCounterStride;
                const index_t waves = SDIV(index_t(gridDim.x) * (blockDim.x >> 6), arenas);
                index_t at = warpcore::detail::atomic_load_relaxed(counter);
                if (total <= kWaveCells && at + waves * kWaveCells <= arena_size(a)) {
                    run = arena_begin(a) + warpcore::detail::atomic_add(counter, index_t(total));
                    at = arena_size(a);
                }
                while (at + total <= arena_size(a)) {
                    const index_t seen = warpcore::detail::atomic_cas(counter, at, at + total);
                    if (seen == at) {
                        run = arena_begin(a) + at;
                        break;
                    }
                    at = seen;
                }
            }
            run = (index_t(unsigned(__builtin_amdgcn_readfirstlane(int(run >> 32)))) << 32) |
                  index_t(unsigned(__builtin_amdgcn_readfirstlane(int(run))));
        }
        if (mine)
            st = fill(&handle->pack, h, next, pairs, max_values_per_key, run + (upto - cells),
                      run != ~index_t(0) ? cells : 0u);
        if (on && !mine) st = append_all(handle, next, pairs, max_values_per_key);
        return st;
    }

    // f(value, j) for j < count, lanes of `group` striding over the values
    template<class Func, unsigned G>
    WC_D void for_each(Func&& f, const handle_type& handle, const tile<G>& group) const noexcept {
        for_each_strided(f, handle, group.thread_rank(), G);
    }

    // One lane's walk of a handle's buckets, tail first, put(value, j) for
    // j < count. Bucket sizes come from the value counts (size_by_count), so
    // each bucket costs one round trip: its link and its values are loaded
    // together, B values at a time, before any of them is put.
    template<unsigned B, class Put>
    WC_D void walk_lane(const handle_type& handle, Put& put) const noexcept {
        if ((!handle.is_initialized() && !handle.is_full()) || handle.bucket_index() == head()) return;
        const index_t count = handle.value_count();
        index_t bucket = handle.bucket_index();
        index_t size = handle.num_values_tail();   // values to read in this bucket
        index_t base = 0;                          // values before this bucket, in walk order
        while (true) {
            const bool headed = count - base > min_size;   // not the first, headerless bucket
            const index_t off = headed ? 1 : 0;
            if (size == 0 || bucket + off + size > capacity) return;   // not on a well-formed chain
            const std::uint64_t info = headed ? buckets[bucket].info : 0;
            for (index_t p = 0; p < size; p += B) {
                Value v[B];
#pragma unroll
                for (unsigned b = 0; b < B; ++b)
                    if (p + b < size) v[b] = buckets[bucket + off + p + b].value;
#pragma unroll
                for (unsigned b = 0; b < B; ++b)
                    if (p + b < size) put(v[b], base + p + b);
            }
            base += size;
            if (base >= count || !headed) return;
            bucket = bucket_type::previous_of(info);
            if (bucket == head() || bucket >= capacity) return;
            if (count - base <= min_size) {
                size = min_size;
            } else if (!size_by_count(count - base, size)) {
                size = bucket_type::size_of(buckets[bucket].info);
            }
        }
    }

    // Lane `rank` of `group_size` lanes takes positions rank, rank + group_size,
    // ... of every bucket; all lanes walk the chain together, so each knows
    // which bucket it is in. (The reference advances lane-local and global
    // indices separately, storage.cuh:1310-1343, which for groups of more
    // than one lane mistakes an earlier bucket for the first, headerless one
    // and then follows a value as a link.)
    template<class Func>
    WC_D void for_each_strided(Func& f, const handle_type& handle, index_t rank, index_t group_size) const
        noexcept {
        if ((!handle.is_initialized() && !handle.is_full()) || handle.bucket_index() == head()) return;
        const index_t count = handle.value_count();
        const index_t tail = handle.num_values_tail();
        index_t bucket = handle.bucket_index();
        const index_t offset = count <= min_size ? 0 : 1;
        for (index_t p = rank; p < tail; p += group_size) f(buckets[bucket + offset + p].value, p);
        index_t base = tail;   // values before the current bucket, in walk order
        while (base < count) {
            bucket = bucket_type::previous_of(buckets[bucket].info);
            const bool last = base >= count - min_size;   // the first, headerless bucket
            const index_t size = last ? min_size : bucket_type::size_of(buckets[bucket].info);
            const index_t off = last ? 0 : 1;
            if (size == 0 || bucket == head() || bucket + off + size > capacity) return;   // not on a well-formed chain
            for (index_t p = rank; p < size; p += group_size) f(buckets[bucket + off + p].value, base + p);
            base += size;
        }
    }
};

}  // namespace detail

template<class Value, index_t BucketIndexBits = 32, index_t ValueCounterBits = 20, index_t BucketSizeBits = 10>
class BucketListStore {
    static_assert(checks::is_valid_value_type<Value>(), "Value type must be trivially copyable.");
    static_assert(BucketIndexBits + ValueCounterBits + BucketSizeBits + 2 <= 64,
                  "Too many bits for bucket index and value counter and bucket size.");
    static_assert(BucketIndexBits + BucketSizeBits <= 64, "bucket header does not fit 64 bits");

public:
    using value_type = Value;
    using handle_type = detail::BucketListHandle<BucketIndexBits, ValueCounterBits, BucketSizeBits>;
    using bucket_type = detail::Bucket<Value, BucketIndexBits, BucketSizeBits>;
    using view_type = detail::BucketListStoreView<Value, BucketIndexBits, ValueCounterBits, BucketSizeBits>;
    using index_type = index_t;
    using status_type = Status;
    using tag = tags::dynamic_value_storage;

    WC_HD static constexpr index_type bucket_index_bits() noexcept { return BucketIndexBits; }
    WC_HD static constexpr index_type value_counter_bits() noexcept { return ValueCounterBits; }
    WC_HD static constexpr index_type bucket_size_bits() noexcept { return BucketSizeBits; }
    WC_HD static constexpr index_type head() noexcept { return handle_type::max_bucket_index(); }
    WC_HD static constexpr handle_type uninitialized_handle() noexcept {
        return handle_type::make(detail::LinkedListState::uninitialized, head(), 0, 0);
    }
    WC_HD static constexpr index_type size(const handle_type& handle) noexcept { return handle.value_count(); }

    // storage.cuh:989-1029
    WC_H explicit BucketListStore(index_type max_capacity, float bucket_grow_factor = 1.1f,
                                  index_type min_bucket_size = 1,
                                  index_type max_bucket_size = handle_type::max_bucket_size()) noexcept
        : status_(Status::not_initialized()), capacity_(max_capacity), bucket_grow_factor_(bucket_grow_factor),
          min_bucket_size_(min_bucket_size), max_bucket_size_(max_bucket_size), buckets_(nullptr),
          counters_(nullptr), arenas_(arenas_for(max_capacity)), is_copy_(false) {
        if (capacity_ < handle_type::max_bucket_index() && bucket_grow_factor_ >= 1.0f && min_bucket_size_ >= 1 &&
            max_bucket_size_ >= min_bucket_size_ && max_bucket_size_ <= handle_type::max_bucket_size()) {
            const std::size_t bytes = sizeof(bucket_type) * capacity_ + counter_bytes();
            if (warpcore::detail::device_memory_for(bytes) &&
                (capacity_ == 0 || warpcore::detail::device_malloc(&buckets_, sizeof(bucket_type) * capacity_) == hipSuccess) &&
                warpcore::detail::device_malloc(&counters_, counter_bytes()) == hipSuccess) {
                status_ = Status::none();
                init();
            } else {
                status_ += Status::out_of_memory();
            }
        } else {
            status_ += Status::invalid_configuration();
        }
    }
    WC_HD BucketListStore(const BucketListStore& o) noexcept
        : status_(o.status_), capacity_(o.capacity_), bucket_grow_factor_(o.bucket_grow_factor_),
          min_bucket_size_(o.min_bucket_size_), max_bucket_size_(o.max_bucket_size_), buckets_(o.buckets_),
          counters_(o.counters_), arenas_(o.arenas_), is_copy_(true) {}
    WC_H BucketListStore(BucketListStore&& o) noexcept
        : status_(o.status_), capacity_(o.capacity_), bucket_grow_factor_(o.bucket_grow_factor_),
          min_bucket_size_(o.min_bucket_size_), max_bucket_size_(o.max_bucket_size_), buckets_(o.buckets_),
          counters_(o.counters_), arenas_(o.arenas_), is_copy_(o.is_copy_) {
        o.is_copy_ = true;
    }
    WC_HD ~BucketListStore() noexcept {
#if !defined(__HIP_DEVICE_COMPILE__)
        if (!is_copy_) {
            if (buckets_ != nullptr) (void)hipFree(buckets_);
            if (counters_ != nullptr) (void)hipFree(counters_);
        }
#endif
    }

    // storage.cuh:1063-1090: every cell becomes a header {head, min size};
    // also empties the pool (every arena's counter = 0, by a fill kernel)
    WC_H void init(hipStream_t stream = 0) noexcept {
        if (status_.has_any() || counters_ == nullptr) return;
        if (capacity_ != 0)
            kernels::fill<std::uint64_t><<<warpcore::detail::grid_for(capacity_, 1, 8), block_size(), 0, stream>>>(
                reinterpret_cast<std::uint64_t*>(buckets_), capacity_ * (sizeof(bucket_type) / 8),
                bucket_type::make_info(head(), min_bucket_size_));
        kernels::fill<index_type><<<1, block_size(), 0, stream>>>(counters_, counter_bytes() / sizeof(index_type),
                                                                  index_type(0));
        status_ = Status::none();
    }

    static constexpr index_type kMaxArenas = 256;
    static constexpr index_type kMinArenaCells = index_type(1) << 16;
    // arenas of a pool: the largest power of two up to kMaxArenas leaving
    // every arena at least kMinArenaCells cells
    WC_HD static constexpr index_type arenas_for(index_type cap) noexcept {
        index_type a = 1;
        while (a < kMaxArenas && cap / (2 * a) >= kMinArenaCells) a *= 2;
        return a;
    }
    WC_HD index_type arenas() const noexcept { return arenas_; }
    WC_HD std::size_t counter_bytes() const noexcept {
        return arenas_ == 1 ? sizeof(index_type) : arenas_ * view_type::kCounterStride * sizeof(index_type);
    }

    WC_D status_type append(handle_type* handle, const value_type& value, index_type max_values_per_key) const
        noexcept {
        return view().append(handle, value, max_values_per_key);
    }

    // f(value, j) for j < size(handle), lanes of `group` striding over the
    // values (storage.cuh:1292-1345)
    template<class Func, unsigned G>
    WC_D void for_each(Func&& f, const handle_type& handle, const tile<G>& group) const noexcept {
        view().for_each(f, handle, group);
    }
    template<class Func>
    WC_D void for_each(Func&& f, const handle_type& handle) const noexcept {
        view().for_each(f, handle, tile<1>{});
    }

    WC_HD view_type view() const noexcept {
        return view_type{buckets_, counters_, capacity_, bucket_grow_factor_, min_bucket_size_, max_bucket_size_,
                         arenas_, capacity_ / arenas_};
    }

    WC_HD status_type status() const noexcept { return status_; }
    WC_HD index_type capacity() const noexcept { return capacity_; }
    WC_H index_type bytes_total() const noexcept { return capacity_ * sizeof(bucket_type) + counter_bytes(); }
    // cells handed out: with one arena its counter, as the reference's
    // next_free (it also counts the cells of failed allocations); with
    // several, each arena's counter up to the arena's size (an arena a
    // request did not fit counts as used up to its end)
    WC_H index_type next_free(hipStream_t stream = 0) const noexcept {
        if (counters_ == nullptr) return 0;
        std::vector<index_type> c(counter_bytes() / sizeof(index_type));
        (void)hipMemcpyAsync(c.data(), counters_, counter_bytes(), hipMemcpyDeviceToHost, stream);
        (void)hipStreamSynchronize(stream);
        if (arenas_ == 1) return c[0];
        const view_type v = view();
        index_type n = 0;
        for (index_type a = 0; a < arenas_; ++a) n += std::min(c[a * view_type::kCounterStride], v.arena_size(a));
        return n;
    }
    // storage.cuh:1370-1380
    WC_H float load_factor(hipStream_t stream = 0) const noexcept {
        return float(next_free(stream)) / float(capacity());
    }
    WC_H index_type bytes_occupied(hipStream_t stream = 0) const noexcept {
        return next_free(stream) * sizeof(bucket_type);
    }
    WC_HD float bucket_grow_factor() const noexcept { return bucket_grow_factor_; }
    WC_HD index_type min_bucket_size() const noexcept { return min_bucket_size_; }
    WC_HD index_type max_bucket_size() const noexcept { return max_bucket_size_; }
    WC_HD bool is_copy() const noexcept { return is_copy_; }

private:
    status_type status_;
    index_type capacity_;
    float bucket_grow_factor_;
    index_type min_bucket_size_;
    index_type max_bucket_size_;
    bucket_type* buckets_;
    index_type* counters_;
    index_type arenas_;
    bool is_copy_;
};

}  // namespace multi_value
}  // namespace storage

namespace defaults {
template<class Value> using value_storage_t = storage::multi_value::BucketListStore<Value>;
}  // namespace defaults

namespace detail {

// Device state of a bucket-list table: the key table's view plus the store.
template<class KeyView, class Store>
struct BucketListView {
    using key_type = typename KeyView::key_type;
    using value_type = typename Store::value_type;
    using handle_type = typename Store::handle_type;
    KeyView keys;
    typename Store::view_type store;
    index_t max_values;

    WC_HD static constexpr index_t cg_size() noexcept { return KeyView::cg_size(); }
    WC_HD Status* status_word() const noexcept { return keys.status_word(); }

    template<class Join>
    WC_D Status insert(key_type key_in, const value_type& value_in, const tile<cg_size()>& group,
                       index_t probing_length, Join& join) const noexcept {
        Status status = Status::unknown_error();
        bool published = false;
        const index_t slot = keys.insert_impl(key_in, status, group, probing_length, join,
                                              static_cast<const handle_type*>(nullptr), published);
        if (slot == ~index_t(0)) return status;
        handle_type* handle = &keys.slots[slot].value;
        index_t count = 0;
        if (group.thread_rank() == 0) count = handle_type{atomic_load_relaxed(&handle->pack)}.value_count();
        count = group.shfl(count, 0);
        if (count >= max_values) {
            join(Status::max_values_for_key_reached());
            return status + Status::max_values_for_key_reached();
        }
        status_base_t appended = 0;
        if (group.thread_rank() == 0) {
            const Status a = store.append(handle, value_in, max_values);
            if (a.has_any()) join(a);
            appended = a.base();
        }
        return status + Status::from_base(group.shfl(appended, 0));
    }

    // handle of key_in from the key table (status none when found)
    template<class Join>
    WC_D Status find(key_type key_in, handle_type& handle, const tile<cg_size()>& group, index_t probing_length,
                     Join& join) const noexcept {
        return keys.retrieve(key_in, handle, group, probing_length, join);
    }
};

// Key pass of a bucket-list insert on the lane-owner kernel: finds or
// claims each key's slot in the key table and records the slot of every
// input pair (slot_of; it stays ~0 where the key failed) for the append
// pass. The pair whose compare-and-swap claims a new key also makes that
// key's first append here: its first bucket (min_size cells, from the
// wavefront's arena) gets the pair's value and the handle becomes
// {initialized, bucket, 1, 1}, as the append's uninitialised path leaves
// it; the handle is a plain store, read by the append pass only (a later
// launch), and the pair is marked kSlotAppended. If no arena holds the
// bucket the handle becomes {full, head, 0, 0}, again as that path leaves
// it, and the pair is marked kSlotAppendFailed (the append pass reports its
// out_of_memory).
constexpr std::uint32_t kSlotAppended = ~1u;       // slot_of marks: appended by the key pass,
constexpr std::uint32_t kSlotAppendFailed = ~2u;   // or its allocation failed there

template<class KeyView, class StoreView>
struct BucketListKeyCore : KeyView {
    std::uint32_t* slot_of;
    const typename StoreView::value_type* values;   // the pairs' values, by position
    StoreView store;
    index_t max_values;
    template<class Join>
    WC_D void finish_insert(index_t, const typename KeyView::value_type&, bool, Status&, Join&) const noexcept {}
    WC_D void on_slot(index_t slot, index_t pos, bool claimed) const noexcept {
        if (claimed && max_values > 0) {
            using LS = storage::multi_value::detail::LinkedListState;
            using handle_type = typename KeyView::value_type;
            const index_t at = store.allocate(store.min_size);
            if (at != ~index_t(0)) {
                store.buckets[at].value = values[pos];
                this->slots[slot].value = handle_type::make(LS::initialized, at, 1, 1);
                slot_of[pos] = kSlotAppended;
            } else {
                this->slots[slot].value = handle_type::make(LS::full, StoreView::head(), 0, 0);
                slot_of[pos] = kSlotAppendFailed;
            }
            return;
        }
        slot_of[pos] = std::uint32_t(slot);
    }
};

// Key walk of up to 64 keys of a wavefront: the slot of key `first` + i goes
// to out[i] (it keeps its value where the key failed).
template<class KeyView>
struct BucketListSlotCore : KeyView {
    std::uint32_t* out;
    index_t first;
    template<class Join>
    WC_D void finish_insert(index_t, const typename KeyView::value_type&, bool, Status&, Join&) const noexcept {}
    WC_D void on_slot(index_t slot, index_t pos, bool) const noexcept { out[pos - first] = std::uint32_t(slot); }
};

// Insert of grouped pairs (pair_groups.hpp): a wavefront finds or claims the
// slots of up to 64 keys, then each lane appends all pairs of its key.
// Pair by pair an append costs one memory-side compare-and-swap on the
// handle and another round trip where a bucket is linked; per key of the
// region it is two. The first step of every key's walk reads the region's keys
// in LDS (2.6 ms for the groups pass, with the walks in the table 3.1). 2^26
// pairs over 2^23 keys: key pass 2.1 and appends 4.8 ms pair by pair; sorted
// and grouped 3.4 ms.
template<class KeyView, class StoreView>
struct BucketListGroupCore : KeyView {
    using key_type = typename KeyView::key_type;
    using pair_value_type = typename StoreView::value_type;
    static constexpr unsigned most_region_slots = 1024;
    StoreView store;
    index_t max_values;

    template<unsigned N>
    struct WalkScratch {
        OwnerEntry<key_type, std::uint32_t> entry[N];
        std::uint32_t slot[N];
    };
    struct group_scratch : WalkScratch<kPartThreads> {
        alignas(16) key_type key[most_region_slots];   // keys of the region's slots
        std::uint16_t moved[kPartThreads];       // per wavefront: its keys that go on to their second window
    };
    using rest_scratch = WalkScratch<256>;

    WC_D index_t budget(index_t probing_length) const noexcept {
        return probing_schemes::detail::window_budget(probing_length, KeyView::cg_size(), this->geometry().windows);
    }

    // slots of keys [first, end) of `in`, at most 64, into the wavefront's
    // scratch.slot (~0 for a key that failed)
    template<class Input, unsigned N, class Join>
    WC_D void find_slots(const Input& in, index_t first, index_t end, WalkScratch<N>& scratch, index_t windows,
                         Join& join) const noexcept {
        const unsigned wave = threadIdx.x & ~63u;
        scratch.slot[threadIdx.x] = ~0u;
        wave_sync();
        const BucketListSlotCore<KeyView> core{*this, scratch.slot + wave, first};
        insert_owner_from<BucketListSlotCore<KeyView>, status_handlers::ReturnNothing, std::uint32_t, false,
                          part_spl<BucketListSlotCore<KeyView>>()>(in, first, end, core, windows, nullptr,
                                                                   scratch.entry + wave, join);
        wave_sync();
    }
    WC_D static void wave_sync() noexcept {   // LDS written by the wavefront's other lanes
        __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
        __builtin_amdgcn_wave_barrier();
        __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
    }

    // Keys of a round that a wavefront moves on to their second windows.
    template<class Rec>
    struct MovedInput {
        const PairGroups<Rec>* groups;
        const std::uint16_t* list;
        static constexpr bool skip_first = true;
        WC_D key_type key(index_t i) const noexcept { return groups->key(list[i]); }
        WC_D typename KeyView::value_type value(index_t) const noexcept { return {}; }
        WC_D static index_t position(index_t i) noexcept { return i; }
    };

    // The keys of the region's slots, before its first round: every key's
    // first window lies here, so the walks' first steps read LDS.
    WC_D void begin_region(group_scratch& scratch, index_t w0, unsigned region_windows) const noexcept {
        constexpr unsigned CG = unsigned(KeyView::cg_size());
        const index_t windows = this->geometry().windows;
        const unsigned slots = unsigned(windows - w0 < region_windows ? windows - w0 : region_windows) * CG;
        for (unsigned i = threadIdx.x; i < slots; i += kPartThreads)
            scratch.key[i] = this->slots[w0 * CG + i].key;
    }

    // The lane's key in its first window: the slot, `claimed` if it is new
    // there, or ~0 when the window is full. Claims settle in LDS first, so
    // that one lane asks the table for a slot; a slot that a key of another
    // region took meanwhile, on its way past its own first window, is
    // corrected here and passed by. (A key passes slots that others are still
    // claiming: no call beside this one may insert, or it could put the same
    // key there.)
    WC_D std::uint32_t first_step(key_type key, group_scratch& scratch, index_t w, index_t w0,
                                  bool& claimed) const noexcept {
        constexpr unsigned CG = unsigned(KeyView::cg_size());
        const unsigned at = unsigned(w - w0) * CG;
        unsigned hit = CG, empty = CG;
#pragma unroll
        for (unsigned o = CG; o-- > 0;) {
            const key_type k = scratch.key[at + o];
            if (k == key) hit = o;
            if (KeyView::is_empty_key(k)) empty = o;
        }
        const index_t slot = w * CG;
        if (hit < CG) return std::uint32_t(slot + hit);
        for (unsigned o = empty; o < CG; ++o) {
            const key_type there = scratch.key[at + o];
            if (!KeyView::is_empty_key(there) || !KeyView::is_empty_key(atomic_cas(scratch.key + at + o, there, key)))
                continue;
            const key_type old = atomic_cas(&this->slots[slot + o].key, there, key);
            claimed = old == there;
            if (claimed || old == key) return std::uint32_t(slot + o);
            scratch.key[at + o] = old;
        }
        return ~0u;
    }

    template<class Rec, class Join>
    WC_D void insert_groups(const PairGroups<Rec>& groups, group_scratch& scratch, index_t w0,
                            index_t probing_length, Join& join) const noexcept {
        const std::uint32_t num = groups.groups;
        constexpr std::uint32_t waves = kPartThreads / 64;
        const unsigned wave = threadIdx.x & ~63u;
        const std::uint32_t share = (num + waves - 1) / waves;   // few keys: fewer per wavefront, all at work
        const std::uint32_t per = share < 64 ? share : 64;
        const index_t windows = budget(probing_length);
        for (std::uint32_t g0 = threadIdx.x / 64 * per; g0 < num; g0 += waves * per) {
            const std::uint32_t g = g0 + lane_id();
            bool on = g < (g0 + per < num ? g0 + per : num) && this->ready();
            bool claimed = false;
            unsigned at = 0, end = 0, pairs = 0;
            key_type key{};
            std::uint32_t slot = ~0u;
            if (on) {
                key = groups.key(g);
                at = groups.list[g];
                end = groups.end(g);
                WindowCursor<typename KeyView::probing_scheme_type> c;
                c.begin(key, this->hash_seed(), this->geometry());
                slot = first_step(key, scratch, c.w, w0, claimed);
                if (slot == ~0u) mark_overflow(static_cast<const KeyView&>(*this), std::uint32_t(c.w), std::uint32_t(c.step));
                if (!claimed && slot != ~0u) join(Status::duplicate_key());
                for (unsigned q = at; q < end; ++q) pairs += groups.buf[q].key == key;
                if (pairs > 1) join(Status::duplicate_key());   // all but one found the key
            }
            const std::uint64_t go = __builtin_amdgcn_ballot_w64(on && slot == ~0u);
            if (go != 0) {
                const unsigned mine = lanes_below(go);
                if (on && slot == ~0u) scratch.moved[wave + mine] = std::uint16_t(g);
                wave_sync();
                const MovedInput<Rec> in{&groups, scratch.moved + wave};
                find_slots(in, 0, index_t(__builtin_popcountll(go)), scratch, windows, join);
                if (on && slot == ~0u) slot = scratch.slot[wave + mine];
                wave_sync();
            }
            on = on && slot != ~0u;
            const Status st = store.append_wave(
                on, claimed, &this->slots[on ? slot : 0].value, pairs,
                [&](pair_value_type& v) {
                    while (at < end && groups.buf[at].key != key) ++at;
                    if (at >= end) return false;
                    v = groups.buf[at++].value;
                    return true;
                },
                max_values);
            if (st.has_any()) join(st);
        }
    }

    template<class Input, class Join>
    WC_D void insert_pairs(const Input& in, index_t lo, index_t hi, rest_scratch& scratch, index_t probing_length,
                           Join& join) const noexcept {
        const index_t windows = budget(probing_length);
        for (index_t i0 = lo; i0 < hi; i0 += 64) {
            const index_t i1 = i0 + 64 < hi ? i0 + 64 : hi;
            find_slots(in, i0, i1, scratch, windows, join);
            const std::uint32_t slot = scratch.slot[threadIdx.x];
            wave_sync();
            const index_t i = i0 + lane_id();
            if (i >= i1 || slot == ~0u) continue;
            bool more = true;
            const Status st = store.append_all(
                &this->slots[slot].value,
                [&](pair_value_type& v) {
                    if (!more) return false;
                    v = in.value(i);
                    more = false;
                    return true;
                },
                1, max_values);
            if (st.has_any()) join(st);
        }
    }
};

}  // namespace detail

namespace kernels {

// slot_of of a chunk before its key pass: no slot
__global__ __launch_bounds__(256) inline void bl_clear(std::uint32_t* __restrict__ slot_of, index_t num_in,
                                                       const index_t* __restrict__ num_dev) {
    if (num_dev != nullptr && *num_dev < num_in) num_in = *num_dev;
    const index_t stride = index_t(gridDim.x) * blockDim.x;
    for (index_t i = index_t(blockIdx.x) * blockDim.x + threadIdx.x; i < num_in; i += stride) slot_of[i] = ~0u;
}

// Append pass of a bucket-list insert: one lane per pair, the pair's value
// appended to the handle of the slot the key pass recorded (the appends of
// a wavefront are independent); the pair's status is the key pass's
// (key_status, or none) + the append's (bucket_list_hash_table.cuh:234-339
// per pair).
template<class View, class StatusHandler>
__global__ __launch_bounds__(256) void bl_append(const typename View::value_type* __restrict__ values_in,
                                                 index_t num_in, const std::uint32_t* __restrict__ slot_of,
                                                 const Status* __restrict__ key_status, View view,
                                                 typename StatusHandler::base_type* __restrict__ status_out,
                                                 const index_t* __restrict__ num_dev) {
    using handle_type = typename View::handle_type;
    warpcore::detail::DeferredJoin join;
    if (num_dev != nullptr && *num_dev < num_in) num_in = *num_dev;
    const index_t stride = index_t(gridDim.x) * blockDim.x;
    for (index_t i = index_t(blockIdx.x) * blockDim.x + threadIdx.x; i < num_in; i += stride) {
        const std::uint32_t slot = slot_of[i];
        Status st = key_status != nullptr ? key_status[i] : Status::none();
        if (slot == detail::kSlotAppendFailed) {
            join(Status::out_of_memory());
            st = st + Status::out_of_memory();
        } else if (slot < detail::kSlotAppendFailed) {   // not failed, not appended by the key pass
            handle_type* h = &view.keys.slots[slot].value;
            const std::uint64_t seen = warpcore::detail::atomic_load_relaxed(&h->pack);
            Status a = Status::max_values_for_key_reached();
            if (handle_type{seen}.value_count() < view.max_values)
                a = view.store.append_from(h, seen, values_in[i], view.max_values);
            if (a.has_any()) join(a);
            st = st + a;
        }
        StatusHandler::handle(st, status_out, i);
    }
    join.flush(view.keys.status_word());
}

template<class View, class StatusHandler>
__global__ __launch_bounds__(256) void bl_insert(const typename View::key_type* __restrict__ keys_in,
                                                 const typename View::value_type* __restrict__ values_in,
                                                 index_t num_in, View view, index_t probing_length,
                                                 typename StatusHandler::base_type* __restrict__ status_out) {
    constexpr unsigned CG = unsigned(View::cg_size());
    const tile<CG> group;
    warpcore::detail::DeferredJoin join;
    const warpcore::detail::GroupRange<CG> r;
    for (index_t gid = r.first; gid < num_in; gid += r.stride) {
        const Status st = view.insert(keys_in[gid], values_in[gid], group, probing_length, join);
        if (group.thread_rank() == 0) StatusHandler::handle(st, status_out, gid);
    }
    join.flush(view.status_word());
}

// per-key value counts and their total (gpu_engine.cuh:466-504)
template<class View, class StatusHandler>
__global__ __launch_bounds__(256) void bl_num_values(const typename View::key_type* __restrict__ keys_in,
                                                     index_t num_in, index_t* __restrict__ total_out,
                                                     index_t* __restrict__ num_per_key_out, View view,
                                                     index_t probing_length,
                                                     typename StatusHandler::base_type* __restrict__ status_out) {
    constexpr unsigned CG = unsigned(View::cg_size());
    const tile<CG> group;
    warpcore::detail::DeferredJoin join;
    warpcore::detail::DeferredCount total;
    const warpcore::detail::GroupRange<CG> r;
    for (index_t gid = r.first; gid < num_in; gid += r.stride) {
        typename View::handle_type h{0};
        const Status st = view.find(keys_in[gid], h, group, probing_length, join);
        const index_t num = st.has_any() ? 0 : h.value_count();
        if (group.thread_rank() == 0) {
            if (num_per_key_out != nullptr) num_per_key_out[gid] = num;
            total(num);
            StatusHandler::handle(st, status_out, gid);
        }
    }
    join.flush(view.status_word());
    total.flush(total_out);
}

// gather pass of the two-pass retrieve (gpu_engine.cuh:305-350)
template<class View, class StatusHandler>
__global__ __launch_bounds__(256) void bl_retrieve(const typename View::key_type* __restrict__ keys_in,
                                                   index_t num_in, const index_t* __restrict__ begin_in,
                                                   const index_t* __restrict__ end_in,
                                                   typename View::value_type* __restrict__ values_out, View view,
                                                   index_t probing_length,
                                                   typename StatusHandler::base_type* __restrict__ status_out) {
    using V = typename View::value_type;
    constexpr unsigned CG = unsigned(View::cg_size());
    const tile<CG> group;
    warpcore::detail::DeferredJoin join;
    const warpcore::detail::GroupRange<CG> r;
    for (index_t gid = r.first; gid < num_in; gid += r.stride) {
        const index_t begin = begin_in[gid];
        const index_t room = end_in[gid] - begin;
        V* out = values_out + begin;
        typename View::handle_type h{0};
        Status st = view.find(keys_in[gid], h, group, probing_length, join);
        index_t num = 0;
        if (!st.has_any()) {
            view.store.for_each([=](const V& v, index_t j) { if (j < room) out[j] = v; }, h, group);
            num = h.value_count();
        }
        if (group.thread_rank() == 0) {
            if (num != room) {
                join(Status::invalid_phase_overlap());
                st += Status::invalid_phase_overlap();
            }
            StatusHandler::handle(st, status_out, gid);
        }
    }
    join.flush(view.status_word());
}

// Snapshot retrieve, second step: counts[i] = value count of the handle
// the key lookup wrote to handles[i] (0 for a key it did not find)
template<class Handle>
__global__ __launch_bounds__(256) void bl_counts(const std::uint64_t* __restrict__ handles, index_t num_in,
                                                 index_t* __restrict__ counts) {
    const index_t stride = index_t(gridDim.x) * blockDim.x;
    for (index_t i = index_t(blockIdx.x) * blockDim.x + threadIdx.x; i < num_in; i += stride)
        counts[i] = Handle{handles[i]}.value_count();
}

// Snapshot retrieve, last step: one lane per key walks the buckets of the
// handle in begin_io[i] (kept there by the lookup), replaces it by the key's
// first output position (end - count) and writes the values tail bucket
// first. A lane per key keeps 64 chains in flight per wavefront.
template<class View>
__global__ __launch_bounds__(256) void bl_walk(index_t num_in, index_t* __restrict__ begin_io,
                                               const index_t* __restrict__ end_in,
                                               typename View::value_type* __restrict__ values_out, View view) {
    using V = typename View::value_type;
    using handle_type = typename View::handle_type;
    const index_t stride = index_t(gridDim.x) * blockDim.x;
    for (index_t i = index_t(blockIdx.x) * blockDim.x + threadIdx.x; i < num_in; i += stride) {
        const handle_type h{begin_io[i]};
        const index_t count = h.value_count();
        const index_t begin = end_in[i] - count;
        begin_io[i] = begin;
        V* out = values_out + begin;
        auto put = [=](const V& v, index_t j) { if (j < count) out[j] = v; };
        view.store.template walk_lane<4>(h, put);
    }
}

// sum of the value counts of all keys (bucket_list_hash_table.cuh:805-822)
template<class View>
__global__ __launch_bounds__(256) void bl_total_values(index_t* __restrict__ num_out, View view) {
    const index_t stride = index_t(gridDim.x) * blockDim.x;
    index_t count = 0;
    for (index_t i = index_t(blockIdx.x) * blockDim.x + threadIdx.x; i < view.keys.capacity(); i += stride) {
        const auto s = view.keys.slot_at(i);
        if (view.keys.is_valid_key(s.key)) count += s.value.value_count();
    }
    count = tile<64>::reduce_add(count);
    if (lane_id() == 0 && count) warpcore::detail::atomic_add(num_out, count);
}

}  // namespace kernels

template<class Key, class Value, Key EmptyKey = defaults::empty_key<Key>(),
         Key TombstoneKey = defaults::tombstone_key<Key>(), class ValueStore = defaults::value_storage_t<Value>,
         class ProbingScheme = defaults::probing_scheme_t<Key, 8>>
class BucketListHashTable {
    static_assert(checks::is_value_storage<ValueStore>(), "not a valid storage type");

public:
    using handle_type = typename ValueStore::handle_type;

private:
    using hash_table_type = SingleValueHashTable<Key, handle_type, EmptyKey, TombstoneKey, ProbingScheme>;
    using value_store_type = ValueStore;

public:
    using key_type = Key;
    using value_type = Value;
    using index_type = index_t;
    using status_type = Status;
    using view_type = detail::BucketListView<typename hash_table_type::view_type, ValueStore>;

    WC_HD static constexpr key_type empty_key() noexcept { return EmptyKey; }
    WC_HD static constexpr key_type tombstone_key() noexcept { return TombstoneKey; }
    WC_HD static constexpr bool is_valid_key(key_type key) noexcept {
        return key != empty_key() && key != tombstone_key();
    }
    WC_HD static constexpr index_type cg_size() noexcept { return hash_table_type::cg_size(); }
    WC_HD static constexpr index_type max_bucket_size() noexcept { return handle_type::max_bucket_size(); }

    // bucket_list_hash_table.cuh:106-125
    WC_H explicit BucketListHashTable(index_type key_capacity, index_type value_capacity,
                                      key_type seed = defaults::seed<key_type>(), float grow_factor = 1.1f,
                                      index_type min_bucket_size = 1, index_type max_bucket_size_ = max_bucket_size(),
                                      index_type max_values_per_key = handle_type::max_value_count(),
                                      bool no_init = false) noexcept
        : hash_table_(key_capacity, seed, true),
          value_store_(value_capacity, grow_factor, min_bucket_size, max_bucket_size_),
          max_values_per_key_(std::min(max_values_per_key, handle_type::max_value_count())), is_copy_(false),
          scan_parts_(nullptr) {
        if (warpcore::detail::device_malloc(&scan_parts_, sizeof(index_type) * warpcore::detail::kScanParts) != hipSuccess) {
            scan_parts_ = nullptr;
            join_status(Status::out_of_memory());
        }
        join_status(value_store_.status());
        if (!no_init) init(seed);
    }
    WC_HD BucketListHashTable(const BucketListHashTable& o) noexcept
        : hash_table_(o.hash_table_), value_store_(o.value_store_), max_values_per_key_(o.max_values_per_key_),
          is_copy_(true), scan_parts_(o.scan_parts_) {}
    WC_H BucketListHashTable(BucketListHashTable&& o) noexcept
        : hash_table_(std::move(o.hash_table_)), value_store_(std::move(o.value_store_)),
          max_values_per_key_(o.max_values_per_key_), is_copy_(o.is_copy_), scan_parts_(o.scan_parts_) {
        o.is_copy_ = true;
    }
    WC_HD ~BucketListHashTable() noexcept {
#if !defined(__HIP_DEVICE_COMPILE__)
        if (!is_copy_ && scan_parts_ != nullptr) (void)hipFree(scan_parts_);
        if (!is_copy_ && scratch_ != nullptr) (void)hipFree(scratch_);
#endif
    }

    // :155-171
    WC_H void init(key_type seed, hipStream_t stream = 0) noexcept {
        const status_type status = hash_table_.peek_status(stream);
        if (!status.has_not_initialized()) {
            hash_table_.init(seed, stream);
            value_store_.init(stream);
            hash_table_.table_.init_pairs(empty_key(), ValueStore::uninitialized_handle(), stream);
        }
    }
    WC_H void init(hipStream_t stream = 0) noexcept { init(hash_table_.seed(), stream); }

    // ---- device calls
    WC_D status_type insert(key_type key_in, const value_type& value_in, const tile<cg_size()>& group,
                            index_type probing_length = defaults::probing_length()) const noexcept {
        warpcore::detail::ImmediateJoin join{hash_table_.status_};
        return state().insert(key_in, value_in, group, probing_length, join);
    }
    WC_D status_type retrieve(key_type key_in, value_type* values_out, index_type& num_out,
                              const tile<cg_size()>& group,
                              index_type probing_length = defaults::probing_length()) const noexcept {
        warpcore::detail::ImmediateJoin join{hash_table_.status_};
        handle_type h{0};
        const status_type st = state().find(key_in, h, group, probing_length, join);
        if (!st.has_any()) {
            value_store_.for_each([=](const value_type& v, index_type j) { values_out[j] = v; }, h, group);
            num_out = h.value_count();
        } else {
            num_out = 0;
        }
        return st;
    }
    template<class Func>
    WC_D status_type for_each(Func f, key_type key_in, const tile<cg_size()>& group,
                              index_type probing_length = defaults::probing_length()) const noexcept {
        warpcore::detail::ImmediateJoin join{hash_table_.status_};
        handle_type h{0};
        const status_type st = state().find(key_in, h, group, probing_length, join);
        if (!st.has_any()) value_store_.for_each(f, h, group);
        return st;
    }
    WC_D status_type num_values(key_type key_in, index_type& num_out, const tile<cg_size()>& group,
                                index_type probing_length = defaults::probing_length()) const noexcept {
        warpcore::detail::ImmediateJoin join{hash_table_.status_};
        handle_type h{0};
        const status_type st = state().find(key_in, h, group, probing_length, join);
        num_out = st.has_any() ? 0 : h.value_count();
        return st;
    }

    // ---- host calls
    // :188-292 (status per pair = key-table status + append status)
    template<class StatusHandler = defaults::status_handler_t>
    WC_H void insert(const key_type* keys_in, const value_type* values_in, index_type num_in,
                     hipStream_t stream = 0, index_type probing_length = defaults::probing_length(),
                     typename StatusHandler::base_type* status_out = nullptr) noexcept {
        static_assert(checks::is_status_handler<StatusHandler>(), "not a valid status handler type");
        if (!hash_table_.is_initialized_ || num_in == 0) return;
        using key_view = typename hash_table_type::view_type;
        using key_core = detail::BucketListKeyCore<key_view, typename value_store_type::view_type>;
        // in chunks of the table's scratch, large batches grouped by key first
        if constexpr (warpcore::detail::fixed_step_scheme<typename key_view::probing_scheme_type>::value &&
                      warpcore::detail::owner_insert_capable<key_core>()) {
            // (slot indices below detail::kSlotAppendFailed fit slot_of)
            if (warpcore::detail::owner_inserts() && hash_table_.capacity() < index_type(detail::kSlotAppendFailed) &&
                reserve_scratch(std::min(num_in, insert_chunk))) {
                constexpr bool statuses = !std::is_same<StatusHandler, status_handlers::ReturnNothing>::value;
                const bool wanted = statuses && status_out != nullptr;
                warpcore::detail::MutationTracker::Exclusive exclusive(hash_table_.mutations_, stream);
                index_type done = 0;
                warpcore::detail::CompletionMark end;
                if constexpr (warpcore::detail::part_record<warpcore::detail::PairRecord<key_type, value_type>>())
                    if (!wanted && exclusive.granted())
                        done = insert_grouped(keys_in, values_in, num_in, stream, probing_length, end);
                if (done != 0) exclusive.use(end);
                if (done < num_in) {
                    typename StatusHandler::base_type* out = nullptr;
                    if constexpr (statuses)
                        if (wanted) out = status_out + done;
                    insert_passes<StatusHandler>(keys_in + done, values_in + done, num_in - done, stream,
                                                 probing_length, out, nullptr);
                }
                if (stream == 0) (void)hipStreamSynchronize(stream);
                return;
            }
        }
        hash_table_.mutations_.note(stream);
        kernels::bl_insert<view_type, StatusHandler>
            <<<warpcore::detail::grid_for(num_in, cg_size()), block_size(), 0, stream>>>(
                keys_in, values_in, num_in, state(), probing_length, status_out);
        if (stream == 0) (void)hipStreamSynchronize(stream);
    }

private:
    static constexpr index_type insert_chunk = index_type(1) << 24;

    // The general insert: the key pass on the lane-owner kernel, then one lane
    // per pair appends, in chunks of the table's scratch (each pair's slot and
    // key status). With num_dev the batch is used when *num_dev is not 0.
    template<class StatusHandler>
    WC_H void insert_passes(const key_type* keys_in, const value_type* values_in, index_type num_in,
                            hipStream_t stream, index_type probing_length,
                            typename StatusHandler::base_type* status_out, const index_type* num_dev) noexcept {
        using key_core = detail::BucketListKeyCore<typename hash_table_type::view_type,
                                                   typename value_store_type::view_type>;
        constexpr bool statuses = !std::is_same<StatusHandler, status_handlers::ReturnNothing>::value;
        const index_type cap = std::min(num_in, insert_chunk);
        std::uint32_t* slot_of = scratch_;
        Status* key_status = reinterpret_cast<Status*>(scratch_ + scratch_cap_);
        for (index_type first = 0; first < num_in; first += cap) {
            const index_type n = num_in - first < cap ? num_in - first : cap;
            kernels::bl_clear<<<warpcore::detail::grid_for(n, 1, 8), block_size(), 0, stream>>>(slot_of, n, num_dev);
            const key_core core{hash_table_.state(), slot_of, values_in + first, value_store_.view(),
                                max_values_per_key_};
            Status* ks = statuses && status_out != nullptr ? key_status : nullptr;
            if (ks != nullptr)
                warpcore::detail::launch_insert_owner<key_core, status_handlers::ReturnStatus, false>(
                    keys_in + first, nullptr, n, core, probing_length, ks, stream, num_dev);
            else
                warpcore::detail::launch_insert_owner<key_core, status_handlers::ReturnNothing, false>(
                    keys_in + first, nullptr, n, core, probing_length, nullptr, stream, num_dev);
            typename StatusHandler::base_type* out = nullptr;
            if constexpr (statuses)
                if (status_out != nullptr) out = status_out + first;
            kernels::bl_append<view_type, StatusHandler>
                <<<warpcore::detail::grid_for(n, 1, 32), block_size(), 0, stream>>>(values_in + first, n, slot_of, ks,
                                                                                    state(), out, num_dev);
        }
    }

    WC_HD view_type state() const noexcept {
        return view_type{hash_table_.state(), value_store_.view(), max_values_per_key_};
    }

    // Large batches without statuses, grouped by key within table regions,
    // where nothing else modifies the key table meanwhile; the number of
    // pairs taken (the rest is the general insert's).
    WC_H index_type insert_grouped(const key_type* keys_in, const value_type* values_in, index_type num_in,
                                   hipStream_t stream, index_type probing_length,
                                   warpcore::detail::CompletionMark& end) noexcept {
        using key_view = typename hash_table_type::view_type;
        using core_type = detail::BucketListGroupCore<key_view, typename value_store_type::view_type>;
        using pair_type = detail::PairRecord<key_type, value_type>;
        const key_view keys = hash_table_.state();
        const core_type core{keys, value_store_.view(), max_values_per_key_};
        index_type done = 0;
        while (done < num_in) {
            const index_type n = std::min(num_in - done, warpcore::detail::kPartChunk);
            if (!warpcore::detail::groups_pay<pair_type>(n, keys.geometry(), stream)) break;
            const key_type* k = keys_in + done;
            const value_type* v = values_in + done;
            if (!warpcore::detail::insert_grouped(k, v, n, core, keys, probing_length, stream, end,
                                                  [&](const index_type* count) {
                                                      insert_passes<status_handlers::ReturnNothing>(
                                                          k, v, n, stream, probing_length, nullptr, count);
                                                  }))
                break;
            done += n;
        }
        return done;
    }

public:
    // :333-424, the same two passes as MultiValueHashTable::retrieve
    template<class StatusHandler = defaults::status_handler_t>
    WC_H void retrieve(const key_type* keys_in, index_type num_in, index_type* begin_offsets_out,
                       index_type* end_offsets_out, value_type* values_out, index_type& num_out,
                       hipStream_t stream = 0, index_type probing_length = defaults::probing_length(),
                       typename StatusHandler::base_type* status_out = nullptr) const noexcept {
        static_assert(checks::is_status_handler<StatusHandler>(), "not a valid status handler type");
        if (!hash_table_.is_initialized_) return;
        if (num_in > index_type(std::numeric_limits<int>::max())) {
            join_status(Status::index_overflow(), stream);
            return;
        }
        if (num_in == 0) {
            num_out = 0;
            return;
        }
        if constexpr (warpcore::detail::owner_capable<typename hash_table_type::view_type>()) {
            if (values_out != nullptr && scan_parts_ != nullptr && warpcore::detail::owner_lookups()) {
                retrieve_snapshot<StatusHandler>(keys_in, num_in, begin_offsets_out, end_offsets_out, values_out,
                                                 num_out, stream, probing_length, status_out);
                return;
            }
        }
        num_values(keys_in, num_in, num_out, end_offsets_out, stream, probing_length);
        if (values_out != nullptr) {
            if (scan_parts_ == nullptr) {
                join_status(Status::out_of_memory(), stream);
                num_out = 0;
                return;
            }
            warpcore::detail::device_scan(end_offsets_out, end_offsets_out, num_in, scan_parts_, true, stream);
            kernels::shift_offsets<index_type><<<warpcore::detail::grid_for(num_in, 1, 8), block_size(), 0, stream>>>(
                begin_offsets_out, end_offsets_out, num_in);
            kernels::bl_retrieve<view_type, StatusHandler>
                <<<warpcore::detail::grid_for(num_in, cg_size()), block_size(), 0, stream>>>(
                    keys_in, num_in, begin_offsets_out, end_offsets_out, values_out, state(), probing_length,
                    status_out);
        } else {
            if (status_out != nullptr)
                kernels::handle_all<StatusHandler>
                    <<<warpcore::detail::grid_for(num_in, 1, 8), block_size(), 0, stream>>>(Status::dry_run(),
                                                                                             status_out, num_in);
            join_status(Status::dry_run(), stream);
        }
        if (stream == 0) (void)hipStreamSynchronize(stream);
    }

    // retrieve with the lane-owner key lookup: each key's handle is read once
    // (into begin_offsets_out), its count becomes end_offsets_out, the scan
    // makes the counts end offsets, and one lane per key walks its buckets.
    // Counts and values come from the one handle read, so the two never
    // disagree (no invalid_phase_overlap); statuses are the lookup's.
    template<class StatusHandler>
    WC_H void retrieve_snapshot(const key_type* keys_in, index_type num_in, index_type* begin_offsets_out,
                                index_type* end_offsets_out, value_type* values_out, index_type& num_out,
                                hipStream_t stream, index_type probing_length,
                                typename StatusHandler::base_type* status_out) const noexcept {
        static_assert(sizeof(handle_type) == sizeof(index_type), "handles are kept in the begin offsets");
        // a key the lookup does not find keeps the word 0: an uninitialised handle of no values
        storage::kernels::fill<index_type><<<warpcore::detail::grid_for(num_in, 1, 8), block_size(), 0, stream>>>(
            begin_offsets_out, num_in, index_type(0));
        warpcore::detail::launch_retrieve_owner<typename hash_table_type::view_type, StatusHandler>(
            keys_in, num_in, reinterpret_cast<handle_type*>(begin_offsets_out), hash_table_.state(), probing_length,
            status_out, stream);
        kernels::bl_counts<handle_type><<<warpcore::detail::grid_for(num_in, 1, 8), block_size(), 0, stream>>>(
            reinterpret_cast<const std::uint64_t*>(begin_offsets_out), num_in, end_offsets_out);
        warpcore::detail::device_scan(end_offsets_out, end_offsets_out, num_in, scan_parts_, true, stream);
        kernels::bl_walk<view_type><<<warpcore::detail::grid_for(num_in, 1, 32), block_size(), 0, stream>>>(
            num_in, begin_offsets_out, end_offsets_out, values_out, state());
        num_out = 0;
        (void)hipMemcpyAsync(&num_out, end_offsets_out + (num_in - 1), sizeof(index_type), hipMemcpyDeviceToHost,
                             stream);
        (void)hipStreamSynchronize(stream);
    }

    // :460-488; num_values_out is index_type& (see MultiValueHashTable)
    WC_H void retrieve_all(key_type* keys_out, index_type& num_keys_out, index_type* begin_offsets_out,
                           index_type* end_offsets_out, value_type* values_out, index_type& num_values_out,
                           hipStream_t stream = 0) const noexcept {
        retrieve_all_keys(keys_out, num_keys_out, stream);
        if (keys_out != nullptr)
            retrieve(keys_out, num_keys_out, begin_offsets_out, end_offsets_out, values_out, num_values_out,
                     stream);
        if (stream == 0) (void)hipStreamSynchronize(stream);
    }

    // :495-527; order unspecified
    WC_H void retrieve_all_keys(key_type* keys_out, index_type& num_out, hipStream_t stream = 0) const noexcept {
        if (!hash_table_.is_initialized_) return;
        if (keys_out == nullptr) {
            num_out = hash_table_.size(stream);
            return;
        }
        index_type* tmp = hash_table_.temp_.get();
        (void)hipMemsetAsync(tmp, 0, sizeof(index_type), stream);
        kernels::retrieve_all<typename hash_table_type::view_type>
            <<<warpcore::detail::grid_for(key_capacity(), 1, 8), block_size(), 0, stream>>>(
                keys_out, static_cast<handle_type*>(nullptr), tmp, hash_table_.state());
        (void)hipMemcpyAsync(&num_out, tmp, sizeof(index_type), hipMemcpyDeviceToHost, stream);
        (void)hipStreamSynchronize(stream);
    }

    // :769-803
    template<class StatusHandler = defaults::status_handler_t>
    WC_H void num_values(const key_type* keys_in, index_type num_in, index_type& num_out,
                         index_type* num_per_key_out = nullptr, hipStream_t stream = 0,
                         index_type probing_length = defaults::probing_length(),
                         typename StatusHandler::base_type* status_out = nullptr) const noexcept {
        static_assert(checks::is_status_handler<StatusHandler>(), "not a valid status handler type");
        if (!hash_table_.is_initialized_) return;
        index_type* tmp = hash_table_.temp_.get();
        (void)hipMemsetAsync(tmp, 0, sizeof(index_type), stream);
        if (num_in != 0)
            kernels::bl_num_values<view_type, StatusHandler>
                <<<warpcore::detail::grid_for(num_in, cg_size()), block_size(), 0, stream>>>(
                    keys_in, num_in, tmp, num_per_key_out, state(), probing_length, status_out);
        (void)hipMemcpyAsync(&num_out, tmp, sizeof(index_type), hipMemcpyDeviceToHost, stream);
        (void)hipStreamSynchronize(stream);
    }

    // :805-822
    WC_H index_type num_values(hipStream_t stream = 0) const noexcept {
        if (!hash_table_.is_initialized_) return 0;
        index_type* tmp = hash_table_.temp_.get();
        (void)hipMemsetAsync(tmp, 0, sizeof(index_type), stream);
        kernels::bl_total_values<view_type>
            <<<warpcore::detail::grid_for(key_capacity(), 1, 8), block_size(), 0, stream>>>(tmp, state());
        index_type out = 0;
        (void)hipMemcpyAsync(&out, tmp, sizeof(index_type), hipMemcpyDeviceToHost, stream);
        (void)hipStreamSynchronize(stream);
        return out;
    }

    WC_H float key_load_factor(hipStream_t stream = 0) const noexcept { return hash_table_.load_factor(stream); }
    WC_H float value_load_factor(hipStream_t stream = 0) const noexcept { return value_store_.load_factor(stream); }
    WC_H index_type bytes_total() const noexcept { return hash_table_.bytes_total() + value_store_.bytes_total(); }
    WC_H index_type bytes_keys(hipStream_t stream = 0) const noexcept { return num_keys(stream) * sizeof(key_type); }
    WC_H index_type bytes_values(hipStream_t stream = 0) const noexcept {
        return num_values(stream) * sizeof(value_type);
    }
    WC_H index_type bytes_payload(hipStream_t stream = 0) const noexcept {
        return bytes_keys(stream) + bytes_values(stream);
    }
    WC_H float storage_density(hipStream_t stream = 0) const noexcept {
        return float(bytes_payload(stream)) / float(bytes_total());
    }
    WC_H float relative_storage_density(hipStream_t stream = 0) const noexcept {
        const float bytes_hash_table = float(hash_table_.capacity() * (sizeof(key_type) + sizeof(handle_type)));
        const float bytes_value_store = float(value_store_.bytes_occupied(stream));
        return float(bytes_payload(stream)) / (bytes_value_store + bytes_hash_table);
    }
    WC_HD bool is_initialized() const noexcept { return hash_table_.is_initialized(); }
    WC_H status_type peek_status(hipStream_t stream = 0) const noexcept { return hash_table_.peek_status(stream); }
    WC_H status_type pop_status(hipStream_t stream = 0) noexcept { return hash_table_.pop_status(stream); }
    WC_HD index_type key_capacity() const noexcept { return hash_table_.capacity(); }
    WC_HD index_type value_capacity() const noexcept { return value_store_.capacity(); }
    WC_H index_type num_keys(hipStream_t stream = 0) const noexcept { return hash_table_.size(stream); }
    WC_H index_type value_cells_used(hipStream_t stream = 0) const noexcept { return value_store_.next_free(stream); }
    WC_HD index_type max_values_per_key() const noexcept { return max_values_per_key_; }
    WC_HD bool is_copy() const noexcept { return is_copy_; }

    // device state for a caller's kernels, which may modify the table at any time
    WC_HD view_type view() const noexcept {
        return view_type{hash_table_.view(), value_store_.view(), max_values_per_key_};
    }

private:
    WC_H void join_status(status_type status, hipStream_t stream = 0) const noexcept {
        hash_table_.join_status(status, stream);
    }
    hash_table_type hash_table_;
    value_store_type value_store_;
    index_type max_values_per_key_;
    bool is_copy_;
    index_type* scan_parts_;   // scratch of the two-pass retrieve's prefix sum
    // scratch of the two-pass insert (per pair of a chunk: its key's slot and
    // its key status), grown on demand; copies of the table do not own it
    std::uint32_t* scratch_ = nullptr;
    index_type scratch_cap_ = 0;
    WC_H bool reserve_scratch(index_type n) noexcept {
        if (n <= scratch_cap_) return true;
        if (is_copy_) return false;
        if (scratch_ != nullptr) (void)hipFree(scratch_);
        scratch_ = nullptr;
        scratch_cap_ = 0;
        if (warpcore::detail::device_malloc(&scratch_, 2 * sizeof(std::uint32_t) * n) != hipSuccess) {
            scratch_ = nullptr;
            return false;
        }
        scratch_cap_ = n;
        return true;
    }
};

}  // namespace warpcore
