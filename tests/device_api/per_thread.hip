// A table modified from several host threads on the null stream, in a
// translation unit whose null stream is the calling thread's own
// (-fgpu-default-stream=per-thread). Test infrastructure.
#include <warpcore/warpcore.hpp>

#include <atomic>
#include <thread>
#include <vector>

using namespace warpcore;

extern "C" {

// what this translation unit takes the null, the per-thread and another
// handle for (no device call)
int wcp_per_thread_stream(int which) {
    int other = 0;
    hipStream_t s[3] = {nullptr, hipStreamPerThread, reinterpret_cast<hipStream_t>(&other)};
    return detail::per_thread_stream(s[which]) ? 1 : 0;
}

// grid of the region passes' launches (no device call)
unsigned wcp_part_blocks(std::uint64_t wanted, unsigned resident) { return detail::part_blocks(wanted, resident); }

// `parts` equal shares of the keys, each inserted by a host thread of its own,
// one call after another, none waited for; returns the keys stored. The
// values are the keys.
std::uint64_t wcp_insert_from_threads(const std::uint64_t* keys, std::uint64_t n, std::uint64_t parts,
                                      std::uint64_t min_capacity, std::uint64_t* values_out) {
    SingleValueHashTable<std::uint64_t, std::uint64_t> table(min_capacity);
    if (hipDeviceSynchronize() != hipSuccess) return 0;
    std::atomic<std::uint64_t> turn{0};   // the thread that inserts; parts + 1: all may end (and their streams)
    std::vector<std::thread> threads;
    for (std::uint64_t p = 0; p < parts; ++p)
        threads.emplace_back([&, p] {
            while (turn.load() != p) std::this_thread::yield();
            const std::uint64_t lo = n / parts * p, hi = p + 1 == parts ? n : lo + n / parts;
            table.insert(keys + lo, keys + lo, hi - lo);
            turn.store(p + 1);
            while (turn.load() <= parts) std::this_thread::yield();
        });
    while (turn.load() != parts) std::this_thread::yield();
    const bool ok = hipDeviceSynchronize() == hipSuccess;
    turn.store(parts + 1);
    for (auto& t : threads) t.join();
    if (!ok) return 0;
    table.retrieve(keys, n, values_out);
    const std::uint64_t stored = table.size();
    return hipDeviceSynchronize() == hipSuccess ? stored : 0;
}

}  // extern "C"
