// Host memory of the bulk inserts: this library's operator new throws on demand,
// and its operator delete counts. Test infrastructure.
#include <warpcore/warpcore.hpp>

#include <cstdlib>
#include <new>

namespace {
bool refuse = false;
unsigned deletes = 0;
}  // namespace

void* operator new(std::size_t bytes) {
    void* p = refuse ? nullptr : std::malloc(bytes);
    if (p == nullptr) throw std::bad_alloc();
    return p;
}
void operator delete(void* p) noexcept {
    ++deletes;
    std::free(p);
}
void operator delete(void* p, std::size_t) noexcept { operator delete(p); }

using namespace warpcore;

// Deletions of a tracker's state after its table's tracker, a copy of it, and a
// copy of the copy made in between are gone, one decimal digit each (no device
// call).
extern "C" int wch_tracker_lifetime() {
    using tracker = detail::MutationTracker;
    auto* place = static_cast<tracker*>(std::malloc(3 * sizeof(tracker)));
    new (place) tracker();
    new (place + 1) tracker(place[0]);
    deletes = 0;
    int seen = 0;
    place[0].~tracker();
    seen = seen * 10 + int(deletes);
    new (place + 2) tracker(place[1]);
    place[1].~tracker();
    seen = seen * 10 + int(deletes);
    place[2].~tracker();
    seen = seen * 10 + int(deletes);
    std::free(place);
    return seen;
}

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
