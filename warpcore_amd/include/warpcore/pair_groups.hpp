// Inserts of (key, value) pairs into tables whose keys own lists of values: a
// large batch is sorted by table region (partition.hpp's passes) until a
// region holds a few thousand pairs, and one workgroup per region brings the
// pairs of each key together in LDS, so that the table is walked, and a key's
// bookkeeping updated, once per key of the region instead of once per pair.
// Slots are claimed by compare-and-swap on the table, as the pair-by-pair
// inserts do.
//
// Passes (all on the caller's stream, no host round trip):
//   begin, scatter, refine   as in partition.hpp, over finer regions
//   groups                   part_groups: the region's keys, each once
//   rest                     the records and positions of the batch for which
//                            a segment had no room, pair by pair
// A batch with very frequent keys (part_begin's sample) is left to the
// table's general insert, which reads on the device that it is wanted.
#pragma once

#include "partition.hpp"

namespace warpcore {
namespace detail {

template<class K, class V>
struct PairRecord {
    K key;
    V value;
};

// The view under which the sorting passes see a table: its keys' windows, and
// values of the pairs' type.
template<class View, class V>
struct PairSortCore : View {
    using value_type = V;
    static constexpr RegionOp region_op = RegionOp::assign;
};

// Pairs per thread and round of part_groups: with the digits, the list of
// keys and the table's scratch at most 80 KB of LDS, two blocks per CU.
template<class Rec>
constexpr unsigned group_items() noexcept { return sizeof(Rec) >= 16 ? 2 : 4; }
constexpr unsigned kGroupDigits = 1024;   // one per thread
// standard deviations of a segment's size: pairs of one key go together, so
// counts spread by the square root of the pairs per key more than keys do
constexpr double kGroupSigmas = 24.0;
// least pairs of a grouped batch, and of one of 16-byte pairs that may hold
// few pairs per key (groups_pay)
constexpr index_t kGroupLeast = index_t(1) << 20, kGroupLeastWide = index_t(1) << 23;

// The pairs of a round, sorted by digit of the key: those of digit d are
// buf[base[d] .. base[d + 1]). list[g] is the first pair of the g-th key.
template<class Rec>
struct PairGroups {
    static constexpr unsigned I = group_items<Rec>(), R = kPartThreads * I;
    using K = decltype(Rec::key);
    alignas(16) Rec buf[R];
    std::uint32_t base[kGroupDigits + 1];
    std::uint16_t list[R];
    std::uint32_t wave[kPartThreads / 64];
    std::uint32_t groups;

    // a hash of its own: the keys of a region share the table's
    WC_D static unsigned digit(K k) noexcept {
        return unsigned(hashers::MurmurHash<K>::hash(K(k ^ K(0x5bd1e995u)))) & (kGroupDigits - 1);
    }
    WC_D K key(index_t g) const noexcept { return buf[list[g]].key; }
    WC_D unsigned end(index_t g) const noexcept { return base[digit(key(g)) + 1]; }

    // all threads; m <= R pairs, item j of the thread is pair j * 1024 + thread
    WC_D void group(const Rec (&rec)[I], std::uint32_t m) noexcept {
        base[threadIdx.x] = 0;
        if (threadIdx.x == 0) groups = 0;
        __syncthreads();
        std::uint32_t d[I], rank[I];
#pragma unroll
        for (unsigned j = 0; j < I; ++j) {
            if (j * kPartThreads + threadIdx.x >= m) continue;
            d[j] = digit(rec[j].key);
            rank[j] = atomicAdd(base + d[j], 1u);
        }
        __syncthreads();
        const std::uint32_t mine = base[threadIdx.x];
        std::uint32_t incl = mine;
#pragma unroll
        for (unsigned s = 1; s < 64; s <<= 1) {
            const std::uint32_t o = __shfl_up(incl, s, 64);
            if (lane_id() >= s) incl += o;
        }
        if (lane_id() == 63) wave[threadIdx.x / 64] = incl;
        __syncthreads();
        for (unsigned w = 0; w < threadIdx.x / 64; ++w) incl += wave[w];
        base[threadIdx.x + 1] = incl;   // the digit's end: the next one's begin
        if (threadIdx.x == 0) base[0] = 0;
        __syncthreads();
#pragma unroll
        for (unsigned j = 0; j < I; ++j)
            if (j * kPartThreads + threadIdx.x < m) buf[base[d[j]] + rank[j]] = rec[j];
        __syncthreads();
#pragma unroll
        for (unsigned j = 0; j < I; ++j) {
            const std::uint32_t i = j * kPartThreads + threadIdx.x;
            bool first = i < m;
            if (first) {
                const K k = buf[i].key;
                for (std::uint32_t q = base[digit(k)]; q < i; ++q)
                    if (buf[q].key == k) {
                        first = false;
                        break;
                    }
            }
            const std::uint64_t all = __builtin_amdgcn_ballot_w64(first);
            if (all == 0) continue;
            std::uint32_t at = 0;
            if (lane_id() == 0) at = atomicAdd(&groups, unsigned(__builtin_popcountll(all)));
            at = unsigned(__builtin_amdgcn_readfirstlane(int(at))) + lanes_below(all);
            if (first) list[at] = std::uint16_t(i);
        }
        __syncthreads();
    }
};

}  // namespace detail

namespace kernels {

// One region per block, in rounds of R pairs: the pairs of each key brought
// together (PairGroups) and handed to core.insert_groups, which every thread
// of the block calls after core.begin_region. Two blocks per CU, so that one block's table walks run
// beside the other's sorting.
template<class Core, class Rec, unsigned Segments>
__global__ __launch_bounds__(1024, 8) void part_groups(const Rec* __restrict__ in,
                                                       const std::uint32_t* __restrict__ counts, unsigned count_stride,
                                                       unsigned cap, unsigned first_region, unsigned last_region,
                                                       unsigned shift, Core core, index_t probing_length) {
    using Groups = detail::PairGroups<Rec>;
    constexpr unsigned I = Groups::I;
    __shared__ Groups groups;
    __shared__ typename Core::group_scratch scratch;
    detail::DeferredJoin join;
    for (unsigned r = first_region + blockIdx.x; r < last_region; r += gridDim.x) {
        std::uint32_t upto[Segments];
        std::uint32_t total = 0;
#pragma unroll
        for (unsigned s = 0; s < Segments; ++s) {
            const std::uint32_t c = counts[s * count_stride + r];
            total += c < cap ? c : cap;
            upto[s] = total;
        }
        if (total == 0) continue;   // uniform over the block
        const index_t w0 = index_t(r) << shift;
        core.begin_region(scratch, w0, 1u << shift);
        const index_t seg0 = index_t(r - (Segments == 1 ? first_region : 0)) * Segments * cap;
        for (std::uint32_t lo = 0; lo < total; lo += Groups::R) {
            Rec rec[I];
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
            }
            groups.group(rec, total - lo < Groups::R ? total - lo : Groups::R);
            core.insert_groups(groups, scratch, w0, probing_length, join);
            __syncthreads();
        }
    }
    join.flush(core.status_word());
}

// The pairs without room, one by one: the listed positions of the batch,
// then what part_refine left. *general = the pairs that the table's general
// insert is to take: all of a batch with very frequent keys, else none.
template<class Core, class Rec>
__global__ __launch_bounds__(256) void part_rest(const Rec* __restrict__ rec, const std::uint32_t* __restrict__ left,
                                                 detail::PartPlan plan, const std::uint32_t* __restrict__ spill_list,
                                                 const index_t* __restrict__ spill_count,
                                                 const std::uint32_t* __restrict__ skewed,
                                                 const typename Core::key_type* __restrict__ keys_in,
                                                 const typename Core::pair_value_type* __restrict__ values_in,
                                                 Core core, index_t probing_length, index_t* __restrict__ general) {
    using K = typename Core::key_type;
    using V = typename Core::pair_value_type;
    using Input = detail::PartInput<K, V, Rec, true>;
    __shared__ typename Core::rest_scratch scratch;
    detail::DeferredJoin join;
    if (blockIdx.x == 0 && threadIdx.x == 0) *general = *skewed != 0 ? plan.n : 0;
    const index_t wave = (index_t(blockIdx.x) * blockDim.x + threadIdx.x) / 64;
    const index_t waves = (index_t(gridDim.x) * blockDim.x) / 64;
    const index_t listed = *spill_count;
    const index_t units = plan.two_pass() ? index_t(plan.buckets) * detail::kPartXcds * plan.tiles : 0;
    // unit 0 ..: 64 listed positions each; then 64 counts of left records each
    const index_t lists = SDIV(listed, index_t(64)), parts = lists + SDIV(units, index_t(64));
    for (index_t u = wave; u < parts; u += waves) {
        const bool list = u < lists;
        const index_t first = (list ? u : u - lists) * 64;
        const std::uint32_t l = list ? 0 : first + lane_id() < units ? left[first + lane_id()] : 0u;
        std::uint64_t some = list ? 1 : __builtin_amdgcn_ballot_w64(l != 0);
        for (; some != 0; some &= some - 1) {
            const unsigned at = unsigned(__builtin_ctzll(some));
            Input in = Input::batch(keys_in, values_in, spill_list);
            index_t lo = first, hi = first + 64 < listed ? first + 64 : listed;
            if (!list) {
                const index_t unit = first + at;
                const index_t base = unit / plan.tiles * plan.cap1 + unit % plan.tiles * plan.tile;
                in = Input::records(rec + base, nullptr, false);
                lo = 0;
                hi = unsigned(__builtin_amdgcn_readlane(int(l), int(at)));
            }
            core.insert_pairs(in, lo, hi, scratch, probing_length, join);
        }
    }
    join.flush(core.status_word());
}

}  // namespace kernels

namespace detail {

// Windows per region of a grouped insert: the largest power of two whose
// share of the batch leaves room in a round for the spread of key counts, and
// whose slots the core takes (Core::most_region_slots).
template<class Core, class Rec>
WC_H unsigned group_windows(index_t n, const probing_schemes::Geometry& geo) noexcept {
    const double per_window = double(n) / double(geo.windows);
    const double most = double(PairGroups<Rec>::R) * 0.92;
    unsigned w = 1;
    while (2.0 * w * per_window <= most && 2 * w * Core::cg_size() <= Core::most_region_slots) w *= 2;
    return w;
}

// Whether the pairs of a batch are grouped: not in a stream capture (the
// workspace is the call's own), and where the passes cost less than they
// save, bucket lists into an empty table of load 0.9, grouped and pair by pair:
//   8-byte pairs   2^20 1.5 per key 175 / 181 us, 8 per key 174 / 337;
//                  2^24 1179 / 1783, 972 / 1854
//   16-byte pairs  2^20 191 / 183 us, 205 / 336; 2^22 447 / 432, 519 / 539;
//                  2^24 1497 / 1815, 1590 / 1920
// (below 2^20 the passes' launches cost more). A batch of fewer pairs than the
// table has slots fills the regions too thinly; one of three per slot or more
// has several pairs per key for certain.
template<class Rec>
WC_H bool groups_pay(index_t n, const probing_schemes::Geometry& geo, hipStream_t stream) noexcept {
    if (n < kGroupLeast || n < geo.capacity || geo.windows >= (index_t(1) << 31) || !refill_inserts() || !owner_inserts())
        return false;
    if (sizeof(Rec) >= 16 && n < kGroupLeastWide && n / 3 < geo.capacity) return false;
    hipStreamCaptureStatus capture = hipStreamCaptureStatusNone;
    if (hipStreamIsCapturing(stream, &capture) != hipSuccess || capture != hipStreamCaptureStatusNone) {
        (void)hipGetLastError();
        return false;
    }
    return true;
}

// Grouped insert of n <= kPartChunk pairs, then general(count) where *count
// (on the device) is n or 0; false (nothing launched) without a workspace.
template<class Core, class SortView, class General>
WC_H bool insert_grouped(const typename Core::key_type* keys_in, const typename Core::pair_value_type* values_in,
                         index_t n, const Core& core, const SortView& view, index_t probing_length, hipStream_t stream,
                         CompletionMark& end, const General& general) noexcept {
    using K = typename Core::key_type;
    using V = typename Core::pair_value_type;
    using Rec = PairRecord<K, V>;
    using Sort = PairSortCore<SortView, V>;
    const Sort sort{view};
    const PartPlan p = make_part_plan<Sort, Rec, false>(n, core.geometry(), group_windows<Core, Rec>(n, core.geometry()),
                                                        kGroupSigmas);
    if (p.regions == 0) return false;
    WorkspaceLease ws(p.bytes + sizeof(index_t), stream, &end);   // and the general insert's count
    if (!ws) return false;
    auto* at = static_cast<unsigned char*>(ws.get());
    auto* A = reinterpret_cast<Rec*>(at + p.a);
    auto* B = reinterpret_cast<Rec*>(at + p.b);
    auto word = [&](index_t off) { return reinterpret_cast<std::uint32_t*>(at + off); };
    auto* spilled = reinterpret_cast<index_t*>(at + p.lists);
    auto* count = reinterpret_cast<index_t*>(at + p.bytes);
    const index_t clear = SDIV(p.counter_words, index_t(4 * kPartThreads));
    kernels::part_begin<Sort><<<unsigned(clear < 256 ? clear : 256) + 1, kPartThreads, 0, stream>>>(
        word(p.c1), p.counter_words, keys_in, n, true, word(p.skewed));
    constexpr auto scatter = kernels::part_scatter<Sort, status_handlers::ReturnNothing, Rec, true, false>;
    scatter<<<part_grid<scatter>(SDIV(n, index_t(p.tile))), kPartThreads, 0, stream>>>(
        keys_in, values_in, n, nullptr, word(p.skewed), sort, p, A, nullptr, word(p.c1), word(p.spill), spilled,
        nullptr);
    if (p.two_pass()) {
        for (unsigned g = 0; g < p.groups; ++g) {
            const unsigned q0 = g * p.group_buckets;
            const unsigned q1 = q0 + p.group_buckets < p.buckets ? q0 + p.group_buckets : p.buckets;
            constexpr auto refine = kernels::part_refine<Sort, Rec, false>;
            refine<<<part_grid<refine>(index_t(q1 - q0) * kPartXcds * p.tiles), kPartThreads, 0, stream>>>(
                A, nullptr, word(p.c1), sort, p, q0, q1, B, nullptr, word(p.c2), word(p.left));
            const unsigned r0 = q0 << p.p2log;
            const unsigned r1 = (q1 << p.p2log) < p.regions ? q1 << p.p2log : p.regions;
            constexpr auto groups = kernels::part_groups<Core, Rec, 1>;
            groups<<<part_grid<groups>(r1 - r0), kPartThreads, 0, stream>>>(B, word(p.c2), 0u, p.cap2, r0, r1,
                                                                           p.shift, core, probing_length);
        }
    } else {
        constexpr auto groups = kernels::part_groups<Core, Rec, kPartXcds>;
        groups<<<part_grid<groups>(p.regions), kPartThreads, 0, stream>>>(A, word(p.c1), p.buckets, p.cap1, 0u,
                                                                         p.regions, p.shift, core, probing_length);
    }
    constexpr auto rest = kernels::part_rest<Core, Rec>;
    rest<<<owner_grid<rest>(SDIV(n, index_t(64))), block_size(), 0, stream>>>(
        A, word(p.left), p, word(p.spill), spilled, word(p.skewed), keys_in, values_in, core, probing_length, count);
    general(count);
    return true;
}

}  // namespace detail
}  // namespace warpcore
