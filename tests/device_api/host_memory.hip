// Bulk inserts while the host has no memory left for C++ allocations: this
// library's operator new throws on demand. Test infrastructure.
#include <warpcore/warpcore.hpp>

#include <cstdlib>
#include <new>

namespace {
bool refuse = false;
}

void* operator new(std::size_t bytes) {
    void* p = refuse ? nullptr : std::malloc(bytes);
    if (p == nullptr) throw std::bad_alloc();
    return p;
}
void operator delete(void* p) noexcept { std::free(p); }
void operator delete(void* p, std::size_t) noexcept { std::free(p); }

using namespace warpcore;

// keys stored by an insert during which operator new throws
extern "C" std::uint64_t wch_insert(const std::uint64_t* keys, std::uint64_t n, std::uint64_t min_capacity,
                                    std::uint64_t* values_out) {
    SingleValueHashTable<std::uint64_t, std::uint64_t> table(min_capacity);
    refuse = true;
    table.insert(keys, keys, n);
    refuse = false;
    table.retrieve(keys, n, values_out);
    const std::uint64_t stored = table.size();
    return hipDeviceSynchronize() == hipSuccess ? stored : 0;
}
