// Tables of value types other than one machine word: bulk inserts large
// enough for the region passes, whose records are bounded. Test
// infrastructure.
#include <warpcore/warpcore.hpp>

using namespace warpcore;

namespace {

struct V12 {   // 16-byte slots with 32-bit keys
    std::uint32_t w[3];
};
struct V16 {
    std::uint64_t w[2];
};
struct V32 {
    std::uint64_t w[4];
};
struct Defaulted {   // trivially copyable, with a default constructor that does something
    std::uint32_t w[2] = {1, 2};
};

template<class K, class V>
WC_HD V value_for(K key, index_t i) {
    V v{};
    constexpr unsigned words = sizeof(v.w) / sizeof(v.w[0]);
    for (unsigned j = 0; j < words; ++j)
        v.w[j] = decltype(+v.w[0])(std::uint64_t(key) * (2 * j + 3) + i * (j + 1));
    return v;
}

template<class K, class V>
__global__ void make_values(const K* keys, index_t n, V* values) {
    const index_t i = index_t(blockIdx.x) * blockDim.x + threadIdx.x;
    if (i < n) values[i] = value_for<K, V>(keys[i], 0);
}
// values[at(i)] against the value of key i
template<class K, class V>
__global__ void count_wrong(const K* keys, index_t n, const V* values, const index_t* begin, const index_t* end,
                            unsigned long long* wrong) {
    const index_t i = index_t(blockIdx.x) * blockDim.x + threadIdx.x;
    if (i >= n) return;
    const V want = value_for<K, V>(keys[i], 0);
    const index_t lo = begin != nullptr ? begin[i] : i, hi = end != nullptr ? end[i] : i + 1;
    bool bad = lo >= hi;
    for (index_t q = lo; q < hi; ++q)
        for (unsigned j = 0; j < sizeof(want.w) / sizeof(want.w[0]); ++j) bad = bad || values[q].w[j] != want.w[j];
    if (bad) atomicAdd(wrong, 1ull);
}

unsigned blocks_for(index_t n) { return unsigned((n + 255) / 256); }

template<class T>
struct Buffer {
    T* p = nullptr;
    explicit Buffer(index_t n) {
        if (hipMalloc(&p, n * sizeof(T)) != hipSuccess) p = nullptr;
    }
    ~Buffer() { (void)hipFree(p); }
};

// keys without their value after an insert and a retrieve of all n; -1: an error
template<class K, class V>
std::int64_t single(const K* keys, index_t n, index_t min_capacity) {
    SingleValueHashTable<K, V> table(min_capacity);
    Buffer<V> in(n), out(n);
    Buffer<unsigned long long> wrong(1);
    unsigned long long bad = 0;
    if (in.p == nullptr || out.p == nullptr || wrong.p == nullptr) return -1;
    if (hipMemcpy(wrong.p, &bad, sizeof(bad), hipMemcpyHostToDevice) != hipSuccess) return -1;
    make_values<<<blocks_for(n), 256>>>(keys, n, in.p);
    table.insert(keys, in.p, n);
    table.retrieve(keys, n, out.p);
    count_wrong<<<blocks_for(n), 256>>>(keys, n, out.p, nullptr, nullptr, wrong.p);
    if (hipMemcpy(&bad, wrong.p, sizeof(bad), hipMemcpyDeviceToHost) != hipSuccess) return -1;
    return table.size() == n && !table.peek_status().has_any() ? std::int64_t(bad) : -2;
}

// the same for bucket lists, one call with every key `copies` times
template<class K, class V>
std::int64_t lists(const K* keys, index_t n, index_t key_capacity, unsigned copies) {
    BucketListHashTable<K, V> table(key_capacity, copies * 4 * n);
    Buffer<K> all(copies * n);
    Buffer<V> in(copies * n), out(copies * n);
    Buffer<index_t> begin(n), end(n);
    Buffer<unsigned long long> wrong(1);
    unsigned long long bad = 0;
    if (all.p == nullptr || in.p == nullptr || out.p == nullptr || begin.p == nullptr || end.p == nullptr || wrong.p == nullptr) return -1;
    if (hipMemcpy(wrong.p, &bad, sizeof(bad), hipMemcpyHostToDevice) != hipSuccess) return -1;
    for (unsigned c = 0; c < copies; ++c)
        if (hipMemcpy(all.p + c * n, keys, n * sizeof(K), hipMemcpyDeviceToDevice) != hipSuccess) return -1;
    make_values<<<blocks_for(copies * n), 256>>>(all.p, copies * n, in.p);
    table.insert(all.p, in.p, copies * n);
    index_t total = 0;
    table.retrieve(keys, n, begin.p, end.p, out.p, total);
    if (total != copies * n) return -3;
    count_wrong<<<blocks_for(n), 256>>>(keys, n, out.p, begin.p, end.p, wrong.p);
    if (hipMemcpy(&bad, wrong.p, sizeof(bad), hipMemcpyDeviceToHost) != hipSuccess) return -1;
    return std::int64_t(bad);
}

// Pairs stored by one call with buckets of 2^26 + 2^14 values in a pool of
// 2^27 - 2 cells, none of whose arenas holds one: the values are the keys' positions.
// The table's status word goes to *status.
std::int64_t large_buckets(const std::uint32_t* keys, index_t n, bool statuses, std::uint32_t* status) {
    using store = storage::multi_value::BucketListStore<std::uint32_t, 27, 8, 27>;
    BucketListHashTable<std::uint32_t, std::uint32_t, defaults::empty_key<std::uint32_t>(),
                        defaults::tombstone_key<std::uint32_t>(), store>
        table(n / 2, (index_t(1) << 27) - 2, defaults::seed<std::uint32_t>(), 1.1f, (1u << 26) + (1u << 14));
    Buffer<Status> out(n);
    if (out.p == nullptr) return -1;
    if (statuses)
        table.insert<status_handlers::ReturnStatus>(keys, keys, n, 0, defaults::probing_length(), out.p);
    else
        table.insert(keys, keys, n);
    *status = table.peek_status().base();
    const std::int64_t stored = std::int64_t(table.num_values());
    return hipDeviceSynchronize() == hipSuccess ? stored : -1;
}

}  // namespace

extern "C" {

std::int64_t wcv_large_buckets(const std::uint32_t* keys, std::uint64_t n, int statuses, std::uint32_t* status) {
    return large_buckets(keys, n, statuses != 0, status);
}

// kind 0 <u64, 32 bytes>, 1 <u64, 16 bytes>, 2 <u32, 12 bytes>; lists: 3 <u32, defaulted>
std::int64_t wcv_single(int kind, const void* keys, std::uint64_t n, std::uint64_t min_capacity) {
    const auto* k64 = static_cast<const std::uint64_t*>(keys);
    const auto* k32 = static_cast<const std::uint32_t*>(keys);
    switch (kind) {
    case 0: return single<std::uint64_t, V32>(k64, n, min_capacity);
    case 1: return single<std::uint64_t, V16>(k64, n, min_capacity);
    case 2: return single<std::uint32_t, V12>(k32, n, min_capacity);
    default: return -1;
    }
}

std::int64_t wcv_lists(int kind, const void* keys, std::uint64_t n, std::uint64_t key_capacity) {
    const auto* k64 = static_cast<const std::uint64_t*>(keys);
    const auto* k32 = static_cast<const std::uint32_t*>(keys);
    switch (kind) {
    case 0: return lists<std::uint64_t, V32>(k64, n, key_capacity, 4);
    case 1: return lists<std::uint64_t, V16>(k64, n, key_capacity, 4);
    case 2: return lists<std::uint32_t, V12>(k32, n, key_capacity, 4);
    case 3: return lists<std::uint32_t, Defaulted>(k32, n, key_capacity, 4);
    default: return -1;
    }
}

}  // extern "C"
