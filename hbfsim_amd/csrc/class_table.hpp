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

// Batches of at least four times the sample look 16,384 requests up first.
// More than kSampleLimit classes among them (of some 30,000 equally frequent
// ones, whose longest probe in 2^16 slots is near the limit of 64) and the
// batch does not try that table: 4M requests of 50,000 classes 1,291 us ->
// 440, of 1M 7,837 -> 557.  Up to kSampleMany (340,000) 2^20 slots hold the
// classes, beyond it 2^24 or `most`.
constexpr std::size_t kSample = 16384;
constexpr std::uint32_t kSampleLimit = 12600;
constexpr std::uint32_t kSampleMany = 16000;

// The most classes among the sample for a table of `cap` slots to be tried.
inline std::uint32_t sample_limit(std::uint64_t cap, std::uint64_t most)
{
    return cap < most && cap <= 1ull << 16 ? kSampleLimit : 0xffffffffu;
}

// The next table after one that proved too small; `sampled`: the classes of
// the sample.
inline std::uint64_t next_slots(std::uint64_t cap, std::uint64_t most, std::uint32_t sampled)
{
    return std::min(cap * (sampled > kSampleMany ? 256 : 16), most);
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
