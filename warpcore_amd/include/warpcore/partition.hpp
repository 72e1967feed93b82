// Partitioned bulk inserts.
//
// A bulk insert that touches most windows of a table pays, per key, a random
// window read, a memory-side compare-and-swap and a value store: about 3.6
// memory requests of the 50 G/s the memory system serves at random (2^28 u64
// keys at load 0.9: 18 ms). Here the batch is first sorted by region of the
// table (a run of windows whose slots fit in LDS), and one workgroup per
// region then inserts the region's keys in LDS and writes its slots back, so
// the table and the batch are streamed instead.
//
// Passes (on the caller's stream, no host round trip):
//  scatter   reads the batch tile by tile, sorts each tile in LDS by region
//            (or by bucket of regions) and appends each run to the bucket's
//            segment. Every XCD has segments of its own: the lines being
//            filled (one per bucket, 128 B x 1024 buckets) then live in one
//            L2, which merges the runs into whole lines. Measured for 2^28
//            records of 16 B: 1.8-1.95 ms with up to 1024 buckets and eight
//            segments each, 3.4 ms with one shared segment; a plain copy of
//            the same bytes takes 1.8 ms.
//  refine    (tables of more than 1024 regions) sorts each bucket
//            by region the same way. All tiles of a bucket run on one XCD, so
//            one segment per region is enough.
//  leftover  records a refine segment had no room for (general insert).
//  build     one workgroup per region: slots to LDS, keys inserted there by
//            LDS compare-and-swap into their first window, slots back. A key
//            whose first window is full marks the overflow filter and is
//            appended to the overflow list.
//  tail      the overflow lists from their second window on, and the records
//            scatter had no room for (or the whole batch, see below), by the
//            lane-owner kernel.
//
// Segments are sized for a uniformly hashed batch (mean + 6 standard
// deviations); what does not fit (many copies of a key) takes the general
// insert. A batch whose keys repeat much takes it whole, without the sorting:
// copies of a hot key find its window in the L2 there, while here they would
// fill one region's segment (power-law keys, 2^26 slots of 16 B: 1.3 ms
// general, 36 ms sorted). The first launch, which clears the counters, looks
// at 4096 keys of the batch and decides.
//
// Per key the protocol is the general one's: a key is stored in a window
// only when every earlier window of its probe sequence was full, a window
// that holds the key makes it a duplicate, and slots never become EMPTY
// again, so lookups and later inserts of any kind see an ordinary table
// (slot order inside a window is placement only).
//
// The build kernel writes whole regions back without atomics, so it runs
// only while nothing else can modify the table (mutation.hpp).
#pragma once

#include "base.hpp"
#include "batched_probing.hpp"
#include "engine.hpp"
#include "mutation.hpp"
#include "owner_probing.hpp"
#include "refill_probing.hpp"
#include "status.hpp"
#include "storage.hpp"
#include "workspace.hpp"

#include <cmath>

namespace warpcore {
namespace detail {

// What a region's workgroup does with a key it finds or claims: assign the
// value (single-value tables), add it (counters), nothing (sets).
enum class RegionOp { assign, add, none };

constexpr unsigned kPartThreads = 1024;      // threads of every block here
constexpr unsigned kPartXcds = 8;            // XCDs of the device; block b runs on XCD b % 8
constexpr unsigned kOnePassRegions = 1024;   // most buckets of one scatter pass
constexpr index_t kRegionBytes = 64 * 1024;  // keys and values of a region: two blocks per CU
constexpr index_t kPartChunk = index_t(1) << 28;   // most keys of one run of the passes
constexpr unsigned kPartGroups = 64;               // most overflow lists
constexpr unsigned kPartSample = 4096, kPartRepeat = 4;   // part_begin
// bytes of refined records in flight (one group's second segments): three
// launches a group (2^28 records of 16 B: 192 MB 22.59 ms for the whole join,
// 512 MB 22.30, 1 GB 22.20)
constexpr index_t kRefineBytes = index_t(512) << 20;

template<class Rec, bool Idx>
constexpr unsigned part_items() noexcept {   // records per thread of a tile
    return sizeof(Rec) >= 16 ? 4 : sizeof(Rec) >= 8 || Idx ? 8 : 16;
}

// Wavefronts per SIMD of the sorting kernels: their tiles leave LDS for two
// blocks per CU with 16-byte records (8 wavefronts per SIMD, 64 VGPRs), else
// for one.
template<class Rec, bool Idx>
constexpr unsigned part_waves() noexcept { return sizeof(Rec) >= 16 && !Idx ? 8 : 4; }

// Windows per region: a power of two whose keys and values fill kRegionBytes.
template<class Core>
constexpr unsigned region_windows() noexcept {
    using K = typename Core::key_type;
    constexpr std::size_t per = sizeof(K) + (Core::region_op == RegionOp::none ? 0 : sizeof(typename Core::value_type));
    unsigned w = 1;
    while (2 * w * Core::cg_size() * per <= kRegionBytes) w *= 2;
    return w;
}

// Records a region's segment holds beyond a uniformly hashed batch's share.
// Counters: the entries of one combining pass repeat keys that are frequent
// but not frequent enough for its block maps, up to some 10^4 times (2^28
// occurrences, Zipf 1.1: without the room those entries took the general
// insert, 5.6 of 13.6 ms).
template<class Core>
constexpr unsigned region_slack() noexcept { return Core::region_op == RegionOp::add ? 32768 : 0; }

// Shape of one run of the passes over at most n keys.
struct PartPlan {
    index_t n = 0;
    unsigned shift = 0;        // log2(windows per region)
    unsigned regions = 0;
    unsigned p2log = 0;        // log2(regions per bucket); 0: one pass
    unsigned buckets = 0;
    unsigned cap1 = 0;         // records per (bucket, XCD) segment
    unsigned cap2 = 0;         // records per region segment
    unsigned tiles = 0;        // refine tiles per segment
    unsigned group_buckets = 0, groups = 1;
    unsigned tile = 0;         // records per tile
    // byte offsets into the workspace
    index_t a = 0, a_idx = 0, b = 0, b_idx = 0, spill = 0, c1 = 0, c2 = 0, left = 0, lists = 0, skewed = 0, bytes = 0;
    index_t counter_words = 0;

    WC_HD bool two_pass() const noexcept { return p2log != 0; }
};

// mean of a Poisson-like count to a segment size: `sigmas` standard deviations
WC_H unsigned part_capacity(double mean, double sigmas = 6.0) noexcept {
    const double c = mean + sigmas * std::sqrt(mean) + 32.0;
    return unsigned((index_t(c) + 31) / 32 * 32);
}

template<class Core, class Rec, bool Idx>
WC_H PartPlan make_part_plan(index_t n, const probing_schemes::Geometry& geo, unsigned rw = region_windows<Core>(),
                             double sigmas = 6.0) noexcept {
    PartPlan p;
    p.n = n;
    while ((1u << p.shift) < rw) ++p.shift;
    const index_t regions = SDIV(geo.windows, index_t(rw));
    if (regions > index_t(kOnePassRegions) * 256) return PartPlan{};
    p.regions = unsigned(regions);
    p.tile = kPartThreads * part_items<Rec, Idx>();
    if (regions > kOnePassRegions) {
        while ((index_t(1) << (2 * p.p2log)) < regions) ++p.p2log;
        if (p.p2log > 8) p.p2log = 8;
    }
    p.buckets = unsigned(SDIV(regions, index_t(1) << p.p2log));
    const double share = double(SDIV(SDIV(n, index_t(p.tile)), kPartXcds) * p.tile);   // records of one XCD
    const double per_region = double(rw) / double(geo.windows);
    const double f1 = std::min(1.0, per_region * double(index_t(1) << p.p2log));
    p.cap1 = part_capacity(std::min(share, double(n)) * f1, sigmas);
    const index_t rec = sizeof(Rec) + (Idx ? 4 : 0);
    auto place = [&](index_t& at, index_t bytes) {
        at = p.bytes;
        p.bytes += (bytes + 255) / 256 * 256;
    };
    const index_t a_records = index_t(p.buckets) * kPartXcds * p.cap1;
    index_t b_records;
    if (p.two_pass()) {
        p.cap2 = part_capacity(double(n) * std::min(1.0, per_region), sigmas) + region_slack<Core>();
        p.tiles = unsigned(SDIV(index_t(p.cap1), index_t(p.tile)));
        const index_t bucket_bytes = (index_t(1) << p.p2log) * p.cap2 * rec;
        index_t gb = kRefineBytes / bucket_bytes / kPartXcds * kPartXcds;   // every XCD gets as many buckets
        if (gb < kPartXcds) gb = kPartXcds;
        const index_t least = SDIV(SDIV(index_t(p.buckets), index_t(kPartGroups)), index_t(kPartXcds)) * kPartXcds;
        if (gb < least) gb = least;
        if (gb > p.buckets) gb = p.buckets;
        p.group_buckets = unsigned(gb);
        p.groups = unsigned(SDIV(index_t(p.buckets), gb));
        b_records = gb * (index_t(1) << p.p2log) * p.cap2;
    } else {
        p.group_buckets = p.buckets;
        b_records = n;   // the overflow list
    }
    place(p.a, a_records * sizeof(Rec));
    if (Idx) place(p.a_idx, a_records * 4);
    place(p.b, b_records * sizeof(Rec));
    if (Idx) place(p.b_idx, b_records * 4);
    place(p.spill, n * 4);
    // counters, cleared together: one contiguous run of words
    const index_t first = p.bytes;
    place(p.c1, index_t(p.buckets) * kPartXcds * 4);
    if (p.two_pass()) {
        place(p.c2, index_t(p.regions) * 4);
        place(p.left, index_t(p.buckets) * kPartXcds * p.tiles * 4);
    }
    place(p.lists, (1 + kPartGroups) * sizeof(index_t));   // spill count, overflow counts
    p.counter_words = (p.bytes - first) / 4;
    place(p.skewed, 4);
    return p;
}

// Key and value of a record: a slot, or a bare key.
template<class Rec>
WC_D auto rec_key(const Rec& r) noexcept {
    if constexpr (std::is_integral<Rec>::value) return r;
    else return r.key;
}

// Input of the general inserts here, the same for the whole wavefront: the
// batch, a list of its positions, or records, as keys and values at equal
// distances.
template<class K, class V, class Rec, bool HasValues>
struct PartInput {
    const unsigned char* keys;
    const unsigned char* values;
    std::uint32_t key_step, value_step;
    const std::uint32_t* list;      // positions of the batch, or null
    const std::uint32_t* where;     // positions of the records, or null
    bool skip_first;
    WC_D static PartInput records(const Rec* rec, const std::uint32_t* idx, bool skip) noexcept {
        PartInput in;
        in.keys = reinterpret_cast<const unsigned char*>(rec);
        in.values = in.keys;
        if constexpr (HasValues) in.values = reinterpret_cast<const unsigned char*>(&rec->value);
        in.key_step = in.value_step = sizeof(Rec);
        in.list = nullptr;
        in.where = idx;
        in.skip_first = skip;
        return in;
    }
    WC_D static PartInput batch(const K* keys, const V* values, const std::uint32_t* list) noexcept {
        PartInput in;
        in.keys = reinterpret_cast<const unsigned char*>(keys);
        in.values = reinterpret_cast<const unsigned char*>(values);
        in.key_step = sizeof(K);
        in.value_step = sizeof(V);
        in.list = list;
        in.where = list;
        in.skip_first = false;
        return in;
    }
    WC_D index_t at(index_t i) const noexcept { return list != nullptr ? index_t(list[i]) : i; }
    WC_D K key(index_t i) const noexcept { return *reinterpret_cast<const K*>(keys + at(i) * key_step); }
    WC_D V value(index_t i) const noexcept {
        if constexpr (HasValues) return *reinterpret_cast<const V*>(values + at(i) * value_step);
        else return V{};
    }
    WC_D index_t position(index_t i) const noexcept { return where != nullptr ? index_t(where[i]) : i; }
};

// Slots per lane of the general inserts here (as the lane-owner launches choose).
template<class Core>
constexpr unsigned part_spl() noexcept { return owner_pairs_capable<Core>() ? 2 : 1; }

template<class Core>
WC_D std::uint32_t first_window(const Core& core, typename Core::key_type key) noexcept {
    WindowCursor<typename Core::probing_scheme_type> c;
    c.begin(key, core.hash_seed(), core.geometry());
    return std::uint32_t(c.w);
}

// One tile of up to kPartThreads * I records, sorted by digit in LDS and
// appended run by run to the digits' segments. counts[d]: records appended
// to digit d's segment so far (by every tile); segment(d): its first record
// in `out`. Records that do not fit are counted; one thread calls
// reserve(count), and each is handed to left(j, at) (item j of the calling
// thread) with its place from there.
template<class Rec, unsigned I, unsigned MaxDigits, bool Idx>
struct TileSort {
    static constexpr unsigned T = kPartThreads * I;
    Rec buf[T];
    std::uint32_t bidx[Idx ? T : 1];
    std::uint16_t dig[T];
    std::uint32_t base[MaxDigits];    // count of a digit, then (segment position of its run) - (its run's place)
    std::uint16_t run[MaxDigits];     // place of the digit's run in the tile (T = 16384 at most)
    std::uint32_t wave[kPartThreads / 64];
    std::uint32_t total;
    std::uint32_t over;               // some digit's segment was too short
    std::uint32_t num_left;           // records of the tile without room
    index_t left_base;

    WC_D void clear(unsigned digits) noexcept {
        for (unsigned d = threadIdx.x; d < digits; d += kPartThreads) base[d] = 0;
        if (threadIdx.x == 0) {
            over = 0;
            num_left = 0;
        }
    }
    // digit[j] == ~0u: no record. Starts after a barrier behind clear(); the
    // caller puts a barrier before the next clear().
    template<class Segment, class Reserve, class Left>
    WC_D void append(const Rec (&rec)[I], const std::uint32_t (&idx)[Idx ? I : 1], const std::uint32_t (&digit)[I],
                     unsigned digits, std::uint32_t* __restrict__ counts, unsigned cap, const Segment& segment,
                     Rec* __restrict__ out, std::uint32_t* __restrict__ out_idx, const Reserve& reserve,
                     const Left& left) noexcept {
        std::uint32_t rank[I];
#pragma unroll
        for (unsigned j = 0; j < I; ++j) {
            rank[j] = 0;
            if (digit[j] != ~0u) rank[j] = atomicAdd(base + digit[j], 1u);
        }
        __syncthreads();
        // exclusive scan of the digits' counts; one atomic per digit present
        // reserves its run in the digit's segment
        const unsigned per = (digits + kPartThreads - 1) / kPartThreads;
        std::uint32_t mine = 0;
        for (unsigned q = 0; q < per; ++q) {
            const unsigned d = threadIdx.x * per + q;
            if (d < digits) mine += base[d];
        }
        std::uint32_t incl = mine;
#pragma unroll
        for (unsigned s = 1; s < 64; s <<= 1) {
            const std::uint32_t o = __shfl_up(incl, s, 64);
            if (lane_id() >= s) incl += o;
        }
        if (lane_id() == 63) wave[threadIdx.x / 64] = incl;
        __syncthreads();
        std::uint32_t at = incl - mine;
        for (unsigned w = 0; w < threadIdx.x / 64; ++w) at += wave[w];
        if (threadIdx.x == kPartThreads - 1) total = at + mine;
        bool full = false;
        for (unsigned q = 0; q < per; ++q) {
            const unsigned d = threadIdx.x * per + q;
            if (d >= digits) break;
            const std::uint32_t c = base[d];
            const std::uint32_t b = c != 0 ? atomic_add(counts + d, c) : 0;
            full = full || b + c > cap;
            run[d] = std::uint16_t(at);
            base[d] = b - at;
            at += c;
        }
        if (full) over = 1;
        __syncthreads();
#pragma unroll
        for (unsigned j = 0; j < I; ++j) {
            if (digit[j] == ~0u) continue;
            const std::uint32_t to = run[digit[j]] + rank[j];
            buf[to] = rec[j];
            if constexpr (Idx) bidx[to] = idx[j];
            dig[to] = std::uint16_t(digit[j]);
        }
        __syncthreads();
        const std::uint32_t m = total;
        for (std::uint32_t i = threadIdx.x; i < m; i += kPartThreads) {
            const std::uint32_t d = dig[i];
            const std::uint32_t pos = base[d] + i;
            if (pos < cap) {
                const index_t o = segment(d) + pos;
                out[o] = buf[i];
                if constexpr (Idx) out_idx[o] = bidx[i];
            }
        }
        if (over != 0) {   // uniform: written before the last barriers
            std::uint32_t place[I];
#pragma unroll
            for (unsigned j = 0; j < I; ++j) {
                const bool l = digit[j] != ~0u && base[digit[j]] + run[digit[j]] + rank[j] >= cap;
                const std::uint64_t all = __builtin_amdgcn_ballot_w64(l);
                std::uint32_t first = 0;
                if (all != 0) {
                    if (lane_id() == 0) first = atomicAdd(&num_left, unsigned(__builtin_popcountll(all)));
                    first = unsigned(__builtin_amdgcn_readfirstlane(int(first)));
                }
                place[j] = l ? first + lanes_below(all) : ~0u;
            }
            __syncthreads();
            if (threadIdx.x == 0) left_base = reserve(num_left);
            __syncthreads();
#pragma unroll
            for (unsigned j = 0; j < I; ++j)
                if (place[j] != ~0u) left(j, left_base + place[j]);
        }
    }
};

}  // namespace detail

namespace kernels {

// Clears the counters; the last block samples the batch: kPartSample keys at
// equal distances, counted per key in LDS. *skewed = 1 when one of them came
// kPartRepeat times (about one key in a thousand of the batch); without
// `sample` it is 0.
template<class Core>
__global__ __launch_bounds__(1024) void part_begin(std::uint32_t* __restrict__ counters, index_t num_counters,
                                                   const typename Core::key_type* __restrict__ keys_in, index_t num_in,
                                                   bool sample, std::uint32_t* __restrict__ skewed) {
    using K = typename Core::key_type;
    if (blockIdx.x + 1 < gridDim.x) {
        const index_t stride = index_t(gridDim.x - 1) * blockDim.x;
        for (index_t i = index_t(blockIdx.x) * blockDim.x + threadIdx.x; i < num_counters; i += stride) counters[i] = 0;
        return;
    }
    constexpr unsigned S = 2 * detail::kPartSample;
    __shared__ K skey[S];
    __shared__ std::uint32_t scount[S];
    __shared__ std::uint32_t most;
    const K none = Core::probe_key(Core::empty_probe());
    for (unsigned s = threadIdx.x; s < S; s += detail::kPartThreads) {
        skey[s] = none;
        scount[s] = 0;
    }
    if (threadIdx.x == 0) most = 0;
    if (!sample) num_in = 0;
    const index_t step = num_in / detail::kPartSample;
    constexpr unsigned P = detail::kPartSample / detail::kPartThreads;
    K key[P];
#pragma unroll
    for (unsigned j = 0; j < P; ++j)
        key[j] = step != 0 ? keys_in[(j * detail::kPartThreads + threadIdx.x) * step] : none;
    __syncthreads();
#pragma unroll
    for (unsigned j = 0; j < P; ++j) {
        if (key[j] == none) continue;
        unsigned s = unsigned(hashers::MurmurHash<K>::hash(key[j])) & (S - 1);
        while (true) {
            const K prev = detail::atomic_cas(skey + s, none, key[j]);
            if (prev == none || prev == key[j]) break;
            s = (s + 1) & (S - 1);
        }
        if (atomicAdd(scount + s, 1u) + 1 >= detail::kPartRepeat) most = 1;
    }
    __syncthreads();
    if (threadIdx.x == 0) *skewed = most;
}

// First pass over the batch: records of bucket d, appended by XCD x, go to
// out[(d * 8 + x) * cap1 ..], counted in counts[x * buckets + d]. Positions
// of the batch without room go to spill_list. With statuses every key's
// status starts as none (or invalid_key); later passes write the others.
// 80 KB of LDS (16-byte records): two blocks per CU.
template<class Core, class StatusHandler, class Rec, bool HasValues, bool Idx>
__global__ __launch_bounds__(1024, (detail::part_waves<Rec, Idx>())) void part_scatter(const typename Core::key_type* __restrict__ keys_in,
                                                     const typename Core::value_type* __restrict__ values_in,
                                                     index_t num_in, const index_t* __restrict__ num_dev,
                                                     const std::uint32_t* __restrict__ skewed, Core core,
                                                     detail::PartPlan plan, Rec* __restrict__ out,
                                                     std::uint32_t* __restrict__ out_idx,
                                                     std::uint32_t* __restrict__ counts,
                                                     std::uint32_t* __restrict__ spill_list,
                                                     index_t* __restrict__ spill_count,
                                                     typename StatusHandler::base_type* __restrict__ status_out) {
    using K = typename Core::key_type;
    constexpr unsigned I = detail::part_items<Rec, Idx>();
    __shared__ detail::TileSort<Rec, I, detail::kOnePassRegions, Idx> ts;
    if (*skewed != 0) return;   // the tail takes the whole batch
    detail::DeferredJoin join;
    if (num_dev != nullptr && *num_dev < num_in) num_in = *num_dev;
    const unsigned x = blockIdx.x % detail::kPartXcds;
    const unsigned shift = plan.shift + plan.p2log;
    const index_t T = index_t(detail::kPartThreads) * I;
    for (index_t tile = index_t(blockIdx.x) * T; tile < num_in; tile += index_t(gridDim.x) * T) {
        ts.clear(plan.buckets);
        Rec rec[I];
        std::uint32_t idx[Idx ? I : 1], digit[I];
        K key[I];
#pragma unroll
        for (unsigned j = 0; j < I; ++j) {
            const index_t i = tile + j * detail::kPartThreads + threadIdx.x;
            key[j] = K{};
            if (i < num_in) {
                key[j] = keys_in[i];
                if constexpr (std::is_integral<Rec>::value) rec[j] = key[j];
                else {
                    rec[j].key = key[j];
                    if constexpr (HasValues) rec[j].value = values_in[i];
                }
            }
        }
#pragma unroll
        for (unsigned j = 0; j < I; ++j) {
            const index_t i = tile + j * detail::kPartThreads + threadIdx.x;
            digit[j] = ~0u;
            if constexpr (Idx) idx[j] = std::uint32_t(i);
            if (i >= num_in) continue;
            if (core.is_valid_key(key[j])) {
                digit[j] = detail::first_window(core, key[j]) >> shift;
                StatusHandler::handle(Status::none(), status_out, i);
            } else {
                join(Status::invalid_key());
                StatusHandler::handle(Status::invalid_key(), status_out, i);
            }
        }
        __syncthreads();
        const index_t cap = plan.cap1;
        ts.append(
            rec, idx, digit, plan.buckets, counts + x * plan.buckets, plan.cap1,
            [=](std::uint32_t d) { return (index_t(d) * detail::kPartXcds + x) * cap; }, out, out_idx,
            [&](std::uint32_t m) { return m != 0 ? detail::atomic_add(spill_count, index_t(m)) : index_t(0); },
            [&](unsigned j, index_t at) {
                spill_list[at] = std::uint32_t(tile + j * detail::kPartThreads + threadIdx.x);
            });
        __syncthreads();
    }
    join.flush(core.status_word());
}

// Second pass over buckets [first_bucket, last_bucket): bucket q runs on XCD
// q % 8 alone, its records of region d go to out[((q - first) * R + d) *
// cap2 ..] (R regions per bucket). A tile's records without room are left at
// the tile's start, their number in left[].
template<class Core, class Rec, bool Idx>
__global__ __launch_bounds__(1024, (detail::part_waves<Rec, Idx>())) void part_refine(Rec* __restrict__ in, std::uint32_t* __restrict__ in_idx,
                                                    const std::uint32_t* __restrict__ counts_in, Core core,
                                                    detail::PartPlan plan, unsigned first_bucket, unsigned last_bucket,
                                                    Rec* __restrict__ out, std::uint32_t* __restrict__ out_idx,
                                                    std::uint32_t* __restrict__ counts,
                                                    std::uint32_t* __restrict__ left) {
    constexpr unsigned I = detail::part_items<Rec, Idx>();
    constexpr unsigned T = detail::kPartThreads * I;
    __shared__ detail::TileSort<Rec, I, 256, Idx> ts;
    const unsigned R = 1u << plan.p2log;
    const unsigned x = blockIdx.x % detail::kPartXcds;
    const unsigned units = detail::kPartXcds * plan.tiles;   // tiles of a bucket
    const unsigned rows = (last_bucket - first_bucket + detail::kPartXcds - 1) / detail::kPartXcds;
    for (unsigned v = blockIdx.x / detail::kPartXcds; v < rows * units; v += gridDim.x / detail::kPartXcds) {
        const unsigned q = first_bucket + (v / units) * detail::kPartXcds + x;
        if (q >= last_bucket) continue;
        const unsigned seg = (v % units) / plan.tiles, t = (v % units) % plan.tiles;
        const std::uint32_t have = counts_in[seg * plan.buckets + q];
        const std::uint32_t c = have < plan.cap1 ? have : plan.cap1;
        const std::uint32_t lo = t * T;
        if (lo >= c) continue;   // uniform over the block
        const index_t base = (index_t(q) * detail::kPartXcds + seg) * plan.cap1 + lo;
        const std::uint32_t m = c - lo < T ? c - lo : T;
        ts.clear(R);
        Rec rec[I];
        std::uint32_t idx[Idx ? I : 1], digit[I];
#pragma unroll
        for (unsigned j = 0; j < I; ++j) {
            const std::uint32_t i = j * detail::kPartThreads + threadIdx.x;
            if (i < m) {
                rec[j] = in[base + i];
                if constexpr (Idx) idx[j] = in_idx[base + i];
            }
        }
#pragma unroll
        for (unsigned j = 0; j < I; ++j) {
            const std::uint32_t i = j * detail::kPartThreads + threadIdx.x;
            digit[j] = i < m ? (detail::first_window(core, detail::rec_key(rec[j])) >> plan.shift) & (R - 1) : ~0u;
        }
        __syncthreads();
        const index_t cap = plan.cap2;
        const index_t row = index_t(q - first_bucket) << plan.p2log;
        ts.append(
            rec, idx, digit, R, counts + (index_t(q) << plan.p2log), plan.cap2,
            [=](std::uint32_t d) { return (row + d) * cap; }, out, out_idx,
            [&](std::uint32_t m) {
                left[(index_t(q) * detail::kPartXcds + seg) * plan.tiles + t] = m;
                return base;
            },
            [&](unsigned j, index_t at) {
                in[at] = rec[j];
                if constexpr (Idx) in_idx[at] = idx[j];
            });
        __syncthreads();
    }
}

// General insert of what part_refine left of buckets [first, last).
template<class Core, class StatusHandler, class Rec, bool HasValues, bool Idx>
__global__ __launch_bounds__(256) void part_leftover(const Rec* __restrict__ rec,
                                                     const std::uint32_t* __restrict__ rec_idx,
                                                     const std::uint32_t* __restrict__ left, Core core,
                                                     detail::PartPlan plan, unsigned first_bucket,
                                                     unsigned last_bucket, index_t probing_length,
                                                     typename StatusHandler::base_type* __restrict__ status_out) {
    using K = typename Core::key_type;
    using V = typename Core::value_type;
    using Input = detail::PartInput<K, V, Rec, HasValues>;
    __shared__ detail::OwnerEntry<K, std::uint32_t> lds[256];
    detail::DeferredJoin join;
    const index_t budget = probing_schemes::detail::window_budget(probing_length, Core::cg_size(),
                                                                  core.geometry().windows);
    const index_t wave = (index_t(blockIdx.x) * blockDim.x + threadIdx.x) / 64;
    const index_t waves = (index_t(gridDim.x) * blockDim.x) / 64;
    const index_t begin = index_t(first_bucket) * detail::kPartXcds * plan.tiles;
    const index_t end = index_t(last_bucket) * detail::kPartXcds * plan.tiles;
    for (index_t u = begin + wave * 64; u < end; u += waves * 64) {
        const std::uint32_t l = u + lane_id() < end ? left[u + lane_id()] : 0u;
        for (std::uint64_t some = __builtin_amdgcn_ballot_w64(l != 0); some != 0; some &= some - 1) {
            const unsigned at = unsigned(__builtin_ctzll(some));
            const index_t unit = u + at;
            const index_t n = unsigned(__builtin_amdgcn_readlane(int(l), int(at)));
            const index_t base = unit / plan.tiles * plan.cap1 + unit % plan.tiles * plan.tile;
            const Input in = Input::records(rec + base, Idx ? rec_idx + base : nullptr, false);
            detail::insert_owner_from<Core, StatusHandler, std::uint32_t, HasValues, detail::part_spl<Core>()>(
                in, 0, n, core, budget, status_out, lds + (threadIdx.x & ~63u), join);
        }
    }
    join.flush(core.status_word());
}

// One region per block: its slots in LDS (keys and values apart, so that the
// lanes' window scans spread over the banks; each window is scanned from a
// part that depends on the window, for the same reason), the region's
// records inserted there, its slots written back whole. Bound by the stream:
// the region's records and slots in, the slots out. 64 KB and 1024 threads,
// two blocks per CU, so that one block's loads run beside the other's
// probing.
template<class Core, class StatusHandler, class Rec, unsigned Segments, bool HasValues, bool Idx>
__global__ __launch_bounds__(1024, 8) void part_build(const Rec* __restrict__ in, const std::uint32_t* __restrict__ in_idx,
                                                   const std::uint32_t* __restrict__ counts, unsigned count_stride,
                                                   unsigned cap, unsigned first_region, unsigned last_region,
                                                   Core core, Rec* __restrict__ over_out,
                                                   std::uint32_t* __restrict__ over_idx,
                                                   index_t* __restrict__ over_count,
                                                   typename StatusHandler::base_type* __restrict__ status_out) {
    using K = typename Core::key_type;
    using V = typename Core::value_type;
    using Cursor = detail::WindowCursor<typename Core::probing_scheme_type>;
    using detail::RegionOp;
    constexpr unsigned CG = unsigned(Core::cg_size());
    constexpr unsigned RW = detail::region_windows<Core>();
    constexpr unsigned S = RW * CG;
    constexpr unsigned PER = 16 / sizeof(K), CH = CG / PER;   // keys per 16 bytes; 16-byte parts of a window's keys
    static_assert(CH >= 1, "windows of at least 16 bytes of keys");
    constexpr RegionOp op = Core::region_op;
    constexpr bool values = op != RegionOp::none;
    constexpr bool filtered = detail::has_overflow_filter<Core>::value;
    constexpr unsigned I = sizeof(K) >= 8 || Idx ? 4 : 8;   // records per thread and round
    __shared__ alignas(16) K lkey[S];
    __shared__ V lval[values ? S : 1];
    __shared__ std::uint32_t lfilter[filtered ? RW / 4 : 1];
    __shared__ std::uint32_t num_over;
    __shared__ index_t over_base;
    detail::DeferredJoin join;
    const probing_schemes::Geometry& geo = core.geometry();
    for (unsigned r = first_region + blockIdx.x; r < last_region; r += gridDim.x) {
        // records of the region: `Segments` runs, one after another
        std::uint32_t upto[Segments];
        std::uint32_t total = 0;
#pragma unroll
        for (unsigned s = 0; s < Segments; ++s) {
            const std::uint32_t c = counts[s * count_stride + r];
            total += c < cap ? c : cap;
            upto[s] = total;
        }
        if (total == 0) continue;   // uniform over the block
        const index_t w0 = index_t(r) * RW;
        const unsigned nw = geo.windows - w0 < RW ? unsigned(geo.windows - w0) : RW;
        const unsigned ns = nw * CG;
        auto* g = core.slot_ptr() + w0 * CG;
        if constexpr (values) {
            for (unsigned i = threadIdx.x; i < ns; i += detail::kPartThreads) {
                const auto s = detail::load_slot(g + i);
                lkey[i] = s.key;
                lval[i] = s.value;
            }
        } else {   // bare keys, 16 bytes per access (a window is a multiple of 16 bytes)
            constexpr unsigned per = 16 / sizeof(K);
            const uint4* g4 = reinterpret_cast<const uint4*>(g);
            uint4* l4 = reinterpret_cast<uint4*>(lkey);
            for (unsigned i = threadIdx.x; i < ns / per; i += detail::kPartThreads) l4[i] = g4[i];
        }
        if constexpr (filtered)
            for (unsigned i = threadIdx.x; i < RW / 4; i += detail::kPartThreads) lfilter[i] = 0;
        const index_t seg0 = index_t(r - (Segments == 1 ? first_region : 0)) * Segments * cap;
        for (std::uint32_t lo = 0; lo < total; lo += detail::kPartThreads * I) {
            Rec rec[I];
            std::uint32_t idx[Idx ? I : 1];
            if (threadIdx.x == 0) num_over = 0;
#pragma unroll
            for (unsigned j = 0; j < I; ++j) {
                const std::uint32_t i = lo + j * detail::kPartThreads + threadIdx.x;
                if (i >= total) continue;
                index_t at = i;
                if constexpr (Segments > 1) {
#pragma unroll
                    for (unsigned s = 0; s + 1 < Segments; ++s)
                        if (i >= upto[s]) at = index_t(s + 1) * cap + (i - upto[s]);
                }
                rec[j] = in[seg0 + at];
                if constexpr (Idx) idx[j] = in_idx[seg0 + at];
            }
            __syncthreads();
            std::uint32_t place[I];   // position among the block's overflowing records, or ~0
#pragma unroll
            for (unsigned j = 0; j < I; ++j) {
                const std::uint32_t i = lo + j * detail::kPartThreads + threadIdx.x;
                bool over = false;
                if (i < total) {
                    const K key = detail::rec_key(rec[j]);
                    Cursor c;
                    c.begin(key, core.hash_seed(), geo);
                    const unsigned wl = unsigned(c.w - w0);
                    // the whole window is read for the key (other paths fill
                    // windows in other slot orders), 16 bytes per access
                    const unsigned turn = wl >> 2;
                    auto slot = [=](unsigned o) {   // o-th slot in the window's order
                        return wl * CG + ((turn + o / PER) & (CH - 1)) * PER + o % PER;
                    };
                    unsigned hit = CG, empty = CG;
#pragma unroll
                    for (unsigned t = 0; t < CH; ++t) {
                        const uint4 v = reinterpret_cast<const uint4*>(lkey)[wl * CH + ((turn + t) & (CH - 1))];
                        K k[PER];
                        __builtin_memcpy(k, &v, 16);
#pragma unroll
                        for (unsigned e = 0; e < PER; ++e) {
                            if (k[e] == key) hit = t * PER + e;
                            if (empty == CG && Core::is_empty_key(k[e])) empty = t * PER + e;
                        }
                    }
                    // claims go through the EMPTY slots in that order, so a
                    // copy of the key claimed meanwhile is met on the way
                    bool claimed = false;
                    if (hit == CG) {
                        for (unsigned o = empty; o < CG; ++o) {
                            K k = lkey[slot(o)];
                            if (Core::is_empty_key(k)) {
                                k = detail::atomic_cas(lkey + slot(o), k, key);
                                claimed = Core::is_empty_key(k);
                            }
                            if (claimed || k == key) {
                                hit = o;
                                break;
                            }
                        }
                    }
                    over = hit == CG;
                    if (!over) {
                        if constexpr (op == RegionOp::assign) lval[slot(hit)] = rec[j].value;
                        else if constexpr (op == RegionOp::add) (void)detail::atomic_add(lval + slot(hit), rec[j].value);
                        if constexpr (op == RegionOp::add)   // several occurrences at once: all but one are duplicates
                            if (rec[j].value > V(1)) join(Status::duplicate_key());
                        if (!claimed) {
                            join(Status::duplicate_key());
                            if constexpr (Idx) StatusHandler::handle(Status::duplicate_key(), status_out, idx[j]);
                        }
                    }
                    if constexpr (filtered)
                        if (over) atomicOr(lfilter + (wl >> 2), detail::overflow_bit(wl, c.step));
                }
                const std::uint64_t all = __builtin_amdgcn_ballot_w64(over);
                std::uint32_t first = 0;
                if (all != 0) {
                    if (lane_id() == 0) first = atomicAdd(&num_over, unsigned(__builtin_popcountll(all)));
                    first = unsigned(__builtin_amdgcn_readfirstlane(int(first)));
                }
                place[j] = over ? first + detail::lanes_below(all) : ~0u;
            }
            __syncthreads();
            if (threadIdx.x == 0) over_base = num_over != 0 ? detail::atomic_add(over_count, index_t(num_over)) : 0;
            if (lo + detail::kPartThreads * I >= total) {   // the last round: the slots go back meanwhile
                if constexpr (values) {
                    for (unsigned i = threadIdx.x; i < ns; i += detail::kPartThreads) {
                        auto s = typename Core::slot_type{};
                        s.key = lkey[i];
                        s.value = lval[i];
                        g[i] = s;
                    }
                } else {
                    constexpr unsigned per = 16 / sizeof(K);
                    uint4* g4 = reinterpret_cast<uint4*>(g);
                    const uint4* l4 = reinterpret_cast<const uint4*>(lkey);
                    for (unsigned i = threadIdx.x; i < ns / per; i += detail::kPartThreads) g4[i] = l4[i];
                }
                if constexpr (filtered)
                    if (core.filter != nullptr)
                        for (unsigned i = threadIdx.x; i < RW / 4; i += detail::kPartThreads)
                            if (lfilter[i] != 0)
                                (void)__hip_atomic_fetch_or(core.filter + w0 / 4 + i, lfilter[i], __ATOMIC_RELAXED,
                                                            __HIP_MEMORY_SCOPE_AGENT);
            }
            __syncthreads();
#pragma unroll
            for (unsigned j = 0; j < I; ++j) {
                if (place[j] == ~0u) continue;
                over_out[over_base + place[j]] = rec[j];
                if constexpr (Idx) over_idx[over_base + place[j]] = idx[j];
            }
            __syncthreads();
        }
    }
    join.flush(core.status_word());
}

// The overflow lists (group g's at over + g * stride, counted in
// over_counts[g]) from the second window on, in equal shares per wavefront
// of their concatenation, then the listed positions of the batch.
template<class Core, class StatusHandler, class Rec, bool HasValues, bool Idx>
__global__ __launch_bounds__(256) void part_tail(const Rec* __restrict__ over, const std::uint32_t* __restrict__ over_idx,
                                                 index_t stride, unsigned groups,
                                                 const index_t* __restrict__ over_counts,
                                                 const std::uint32_t* __restrict__ spill_list,
                                                 const index_t* __restrict__ spill_count,
                                                 const std::uint32_t* __restrict__ skewed,
                                                 const typename Core::key_type* __restrict__ keys_in,
                                                 const typename Core::value_type* __restrict__ values_in,
                                                 index_t num_in, const index_t* __restrict__ num_dev, Core core,
                                                 index_t probing_length,
                                                 typename StatusHandler::base_type* __restrict__ status_out) {
    using K = typename Core::key_type;
    using V = typename Core::value_type;
    using Input = detail::PartInput<K, V, Rec, HasValues>;
    __shared__ detail::OwnerEntry<K, std::uint32_t> lds[256];
    auto* my = lds + (threadIdx.x & ~63u);
    detail::DeferredJoin join;
    const index_t budget = probing_schemes::detail::window_budget(probing_length, Core::cg_size(),
                                                                  core.geometry().windows);
    const index_t wave = (index_t(blockIdx.x) * blockDim.x + threadIdx.x) / 64;
    const index_t waves = (index_t(gridDim.x) * blockDim.x) / 64;
    if (num_dev != nullptr && *num_dev < num_in) num_in = *num_dev;
    const bool whole = *skewed != 0;
    // part 0: the overflow lists, one after another; part 1: the listed
    // positions of the batch, or (skewed) all of it. One call for both keeps
    // the kernel to one copy of the insert.
    const index_t listed = whole ? num_in : *spill_count;
    index_t overflowed = 0;
    if (!whole)
        for (unsigned g = 0; g < groups; ++g) overflowed += over_counts[g];
    for (unsigned part = 0; part < 2; ++part) {
        // equal shares of at least one key per lane
        const index_t total = part == 0 ? overflowed : listed;
        index_t per = SDIV(total, waves);
        per = per < 64 ? 64 : per;
        const index_t first = wave * per;
        const index_t end = first + per < total ? first + per : total;
        const unsigned lists = part == 0 ? groups : 1;
        index_t base = 0;
        for (unsigned g = 0; g < lists; ++g) {
            const index_t n = part == 0 ? over_counts[g] : total;
            const index_t lo = first > base ? first - base : 0;
            const index_t hi = end > base ? (end - base < n ? end - base : n) : 0;
            Input in = Input::batch(keys_in, values_in, whole ? nullptr : spill_list);
            if (part == 0)
                in = Input::records(over + g * stride, Idx ? over_idx + g * stride : nullptr, true);
            if (first < end && lo < hi)
                detail::insert_owner_from<Core, StatusHandler, std::uint32_t, HasValues, detail::part_spl<Core>()>(
                    in, lo, hi, core, budget, status_out, my, join);
            base += n;
        }
    }
    join.flush(core.status_word());
}

}  // namespace kernels

namespace detail {

template<class Core, class = void>
struct has_region_op : std::false_type {};
template<class Core>
struct has_region_op<Core, std::void_t<decltype(Core::region_op)>> : std::true_type {};

// Records that the sorting tiles hold in LDS: up to 16 bytes (a tile of them
// takes 80 KB, two blocks per CU; of 24 bytes 112 KB, half the wavefronts, of
// 32 bytes 176 KB, more than a CU has), and plain enough for shared memory.
template<class Rec>
constexpr bool part_record() noexcept {
    return sizeof(Rec) <= 16 && std::is_trivially_default_constructible<Rec>::value;
}

// Windows of 4..16 slots with a fixed step, at most 64 KB a region; handlers
// that may run twice per key.
template<class Core, class Rec, class StatusHandler>
constexpr bool partition_capable() noexcept {
    return has_region_op<Core>::value && fixed_step_scheme<typename Core::probing_scheme_type>::value &&
           Core::cg_size() >= 4 && Core::cg_size() <= 16 && part_record<Rec>() &&
           status_handlers::overwrites<StatusHandler>::value;
}

// Grid of a launch whose blocks are dealt to the XCDs in turn: a multiple of 8
// (part_refine strides by eighths of it), at most the resident blocks where
// there are as many.
constexpr unsigned part_blocks(index_t wanted, unsigned resident) noexcept {
    const index_t up = SDIV(wanted < 1 ? 1 : wanted, index_t(kPartXcds)) * kPartXcds;
    const unsigned most = resident < kPartXcds ? kPartXcds : resident / kPartXcds * kPartXcds;
    return unsigned(up < most ? up : most);
}
template<auto Kernel>
WC_H unsigned part_grid(index_t wanted) noexcept {
    static const unsigned resident = [] {
        int blocks = 0;
        if (hipOccupancyMaxActiveBlocksPerMultiprocessor(&blocks, Kernel, int(kPartThreads), 0) != hipSuccess ||
            blocks < 1)
            blocks = 1;
        return unsigned(num_compute_units()) * unsigned(blocks);
    }();
    return part_blocks(wanted, resident);
}

// Whether a batch of n keys is partitioned. Below 2^20 keys the passes'
// launches cost more than the random requests they save. The build streams
// the whole table, so the batch must be large against it: 8-byte slots from a
// quarter of the slots on (2^26 slots, empty table: 530 us against 737 general;
// 60 % full: 716 against 929; an eighth of the slots: no gain), 16-byte
// slots, twice the stream per key, from three eighths on (a quarter, 60 %
// full: 1272 us against 1169). A batch of more than twice the table's slots is
// mostly duplicates.
template<class Core>
WC_H bool partition_pays(index_t n, const probing_schemes::Geometry& geo) noexcept {
    constexpr index_t least = index_t(1) << 20;
    constexpr index_t eighths = sizeof(*std::declval<const Core&>().slot_ptr()) > 8 ? 3 : 2;
    return n >= least && n >= geo.capacity / 8 * eighths && n <= 2 * geo.capacity && geo.windows < (index_t(1) << 31);
}

// Runs the passes over one chunk, `end` behind them; false (nothing launched)
// without a workspace for it. With num_dev the chunk holds min(n, *num_dev) keys (a
// count made on the device), none of them frequent, so none are sampled.
template<class Core, class StatusHandler, bool HasValues, class Rec>
WC_H bool insert_partitioned_chunk(const typename Core::key_type* keys_in, const typename Core::value_type* values_in,
                                   index_t n, const index_t* num_dev, const Core& core, index_t probing_length,
                                   typename StatusHandler::base_type* status_out, hipStream_t stream,
                                   CompletionMark& end) noexcept {
    using V = typename Core::value_type;
    constexpr bool Idx = !std::is_same<StatusHandler, status_handlers::ReturnNothing>::value;
    const PartPlan p = make_part_plan<Core, Rec, Idx>(n, core.geometry());
    if (p.regions == 0) return false;
    WorkspaceLease ws(p.bytes, stream, &end);
    if (!ws) return false;
    auto* at = static_cast<unsigned char*>(ws.get());
    auto* A = reinterpret_cast<Rec*>(at + p.a);
    auto* B = reinterpret_cast<Rec*>(at + p.b);
    auto word = [&](index_t off) { return reinterpret_cast<std::uint32_t*>(at + off); };
    std::uint32_t* a_idx = Idx ? word(p.a_idx) : nullptr;
    std::uint32_t* b_idx = Idx ? word(p.b_idx) : nullptr;
    auto* lists = reinterpret_cast<index_t*>(at + p.lists);   // [0] spilled, [1 + g] overflow of group g
    const std::uint32_t* skewed = word(p.skewed);
    const index_t clear = SDIV(p.counter_words, index_t(4 * kPartThreads));
    kernels::part_begin<Core><<<unsigned(clear < 256 ? clear : 256) + 1, kPartThreads, 0, stream>>>(
        word(p.c1), p.counter_words, keys_in, n, num_dev == nullptr, word(p.skewed));
    const index_t tiles = SDIV(n, index_t(p.tile));
    constexpr auto scatter = kernels::part_scatter<Core, StatusHandler, Rec, HasValues, Idx>;
    scatter<<<part_grid<scatter>(tiles), kPartThreads, 0, stream>>>(
        keys_in, values_in, n, num_dev, skewed, core, p, A, a_idx, word(p.c1), word(p.spill), lists, status_out);
    const index_t stride = index_t(p.group_buckets) * kPartXcds * p.cap1;   // records of a group's buckets
    if (p.two_pass()) {
        for (unsigned g = 0; g < p.groups; ++g) {
            const unsigned q0 = g * p.group_buckets;
            const unsigned q1 = q0 + p.group_buckets < p.buckets ? q0 + p.group_buckets : p.buckets;
            constexpr auto refine = kernels::part_refine<Core, Rec, Idx>;
            refine<<<part_grid<refine>(index_t(q1 - q0) * kPartXcds * p.tiles), kPartThreads, 0, stream>>>(
                A, a_idx, word(p.c1), core, p, q0, q1, B, b_idx, word(p.c2), word(p.left));
            constexpr auto leftover = kernels::part_leftover<Core, StatusHandler, Rec, HasValues, Idx>;
            leftover<<<owner_grid<leftover>(index_t(q1 - q0) * kPartXcds * p.tiles), block_size(), 0, stream>>>(
                A, a_idx, word(p.left), core, p, q0, q1, probing_length, status_out);
            const unsigned r0 = q0 << p.p2log;
            const unsigned r1 = (q1 << p.p2log) < p.regions ? q1 << p.p2log : p.regions;
            constexpr auto build = kernels::part_build<Core, StatusHandler, Rec, 1, HasValues, Idx>;
            build<<<part_grid<build>(r1 - r0), kPartThreads, 0, stream>>>(
                B, b_idx, word(p.c2), 0u, p.cap2, r0, r1, core, A + g * stride, Idx ? a_idx + g * stride : nullptr,
                lists + 1 + g, status_out);
        }
    } else {
        constexpr auto build = kernels::part_build<Core, StatusHandler, Rec, kPartXcds, HasValues, Idx>;
        build<<<part_grid<build>(p.regions), kPartThreads, 0, stream>>>(A, a_idx, word(p.c1), p.buckets, p.cap1, 0u,
                                                                        p.regions, core, B, b_idx, lists + 1,
                                                                        status_out);
    }
    constexpr auto tail = kernels::part_tail<Core, StatusHandler, Rec, HasValues, Idx>;
    tail<<<refill_grid<tail>(), block_size(), 0, stream>>>(
        p.two_pass() ? A : B, p.two_pass() ? a_idx : b_idx, stride, p.groups, lists + 1, word(p.spill), lists, skewed,
        keys_in, HasValues ? values_in : static_cast<const V*>(nullptr), n, num_dev, core, probing_length, status_out);
    return true;
}

// Partitioned insert of the batch, chunk by chunk; returns the keys handled
// (fewer than n when a workspace was refused: the caller inserts the rest).
template<class Core, class StatusHandler, bool HasValues, class Rec>
WC_H index_t insert_partitioned(const typename Core::key_type* keys_in, const typename Core::value_type* values_in,
                                index_t n, const Core& core, index_t probing_length,
                                typename StatusHandler::base_type* status_out, hipStream_t stream,
                                CompletionMark& end) noexcept {
    index_t done = 0;
    while (done < n) {
        const index_t m = n - done < kPartChunk ? n - done : kPartChunk;
        if (!partition_pays<Core>(m, core.geometry())) break;
        typename StatusHandler::base_type* st = nullptr;
        if constexpr (!std::is_same<StatusHandler, status_handlers::ReturnNothing>::value)
            if (status_out != nullptr) st = status_out + done;
        if (!insert_partitioned_chunk<Core, StatusHandler, HasValues, Rec>(
                keys_in + done, HasValues ? values_in + done : nullptr, m, nullptr, core, probing_length, st, stream, end))
            break;
        done += m;
    }
    return done;
}

// The partitioned insert of a batch that fills much of the table, where
// nothing else can modify the table meanwhile (else the call is noted with
// the tracker for the kernels that follow); advances the arguments past the
// keys it took, true if that is all. Tables whose inserts a process-wide
// setting sends to another kernel family are left to it.
template<class Core, class StatusHandler, bool HasValues, class Rec>
WC_H bool insert_partitioned_first(const MutationTracker& mutations, const typename Core::key_type*& keys_in,
                                   const typename Core::value_type*& values_in, index_t& num_in, const Core& core,
                                   index_t probing_length, typename StatusHandler::base_type*& status_out,
                                   hipStream_t stream, index_t table_bytes) noexcept {
    if (!refill_inserts() || !owner_inserts() || table_bytes <= lane_insert_table_bytes() ||
        !partition_pays<Core>(num_in, core.geometry())) {
        mutations.note(stream);
        return false;
    }
    MutationTracker::Exclusive exclusive(mutations, stream);
    if (!exclusive.granted()) return false;
    CompletionMark end;
    const index_t done = insert_partitioned<Core, StatusHandler, HasValues, Rec>(
        keys_in, values_in, num_in, core, probing_length, status_out, stream, end);
    if (done == 0) return false;
    exclusive.use(end);
    keys_in += done;
    if constexpr (HasValues) values_in += done;
    num_in -= done;
    if constexpr (!std::is_same<StatusHandler, status_handlers::ReturnNothing>::value)
        if (status_out != nullptr) status_out += done;
    return num_in == 0;
}

}  // namespace detail
}  // namespace warpcore
