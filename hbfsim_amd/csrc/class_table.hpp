// class_table.hpp -- how large the class table of a batch is (hybrid.hip).
//
// Open addressing with linear probing; lookups end at the class or at an empty
// slot, so a table whose probes have no limit must never be full.
#pragma once

#include <algorithm>
#include <cstddef>
#include <cstdint>

namespace hbfamd {

// A batch of n requests on top of `seen` classes: at least two slots per class
// they can hold, in a power of two.  `limit`: the slots the caller can number
// (the calibrator, whose slot numbers are 32-bit: n is below 2^32 there, so a
// slot stays empty).
inline std::uint64_t most_slots(std::size_t n, std::size_t seen,
                                std::uint64_t limit = std::uint64_t{1} << 63)
{
    std::uint64_t cap = 1ull << 10;
    while (cap < 2 * (static_cast<std::uint64_t>(n) + seen)) {
        cap <<= 1;
    }
    return std::min(cap, limit);
}

// The first table: 2^16 slots, or four per seen class, at most `most`.
inline std::uint64_t first_slots(std::size_t seen, std::uint64_t most)
{
    std::uint64_t cap = 1ull << 16;
    while (cap < 4 * static_cast<std::uint64_t>(seen)) {
        cap <<= 1;
    }
    return std::min(cap, most);
}

// The next table after one that proved too small.
inline std::uint64_t next_slots(std::uint64_t cap, std::uint64_t most)
{
    return std::min(cap * 16, most);
}

// Workgroups of 256 threads for kernels that walk a table (or a list) of
// `count` entries, each a run of them: one atomic per workgroup stays cheap,
// and the launch stays below 2^32 threads whatever the table's size.
inline unsigned walk_blocks(std::uint64_t count)
{
    return static_cast<unsigned>(
        std::min<std::uint64_t>(2048, std::max<std::uint64_t>(1, (count + 255) / 256)));
}

}  // namespace hbfamd
