// hybrid.hip -- the hybrid model's request sampler and calibrator
// (src/hybrid/calibrator.cpp:67-138) on the GPU.
//
// HybridSampler::reference(sequence, access) (calibrator.cpp:83-96) sends a
// request to the detailed model when its sequence is a warm-up one, when its
// access class was never seen before, or when a SplitMix64 hash of
// (sequence, seed, class) falls at or below the rate's threshold.  Over a
// batch the "never seen" requests are the first occurrence of each class in
// the batch whose class is also absent from the classes earlier batches saw.
//
// Calibrator (calibrator.cpp:98-136) keeps every latency per class and
// reports count, mean, p50/p95/p99 and the mean and deviation of the logs.
//
// Neither sorts requests by class.  A batch's classes go into an open-addressed
// hash table whose slots name a representative (a request of the batch or a
// class an earlier batch saw), so one pass over the 16-byte classes gives
// every request its class: 4M requests of 2,000 classes take 55-61 us,
// against 1.5 ms for two 64-bit radix sorts with payload.  The sampler's
// first occurrences are atomic minima per slot.  The calibrator numbers the
// classes in class order (the order of the reference's std::map), sorts one
// combined key (class number above latency) and reads rank statistics from
// each class's segment.
#include <hip/hip_runtime.h>

#include <cstring>  // rocPRIM's host code uses memset
#include <rocprim/device/device_radix_sort.hpp>

#include "class_table.hpp"
#include "engine.hpp"
#include "scratch.hpp"

#include <algorithm>
#include <cmath>
#include <cstdint>
#include <limits>

namespace hbfamd {
namespace {

constexpr int kThreads = 256;

__device__ __forceinline__ std::uint64_t class_hi(const hbfsim_amd_access_class& c)
{
    return (static_cast<std::uint64_t>(c.operation) << 32) | c.bytes;
}

__device__ __forceinline__ std::uint64_t class_lo(const hbfsim_amd_access_class& c)
{
    return (static_cast<std::uint64_t>(c.queue_bucket) << 32) | c.locality_bucket;
}

// SplitMix64 finaliser (calibrator.cpp:12-18).
__device__ __forceinline__ std::uint64_t mix(std::uint64_t v)
{
    v += 0x9e3779b97f4a7c15ull;
    v = (v ^ (v >> 30)) * 0xbf58476d1ce4e5b9ull;
    v = (v ^ (v >> 27)) * 0x94d049bb133111ebull;
    return v ^ (v >> 31);
}

unsigned blocks_for(std::size_t n)
{
    return static_cast<unsigned>((n + kThreads - 1) / kThreads);
}

// Grid-stride launches: eight 256-thread blocks per CU fill the chip, and one
// atomic per block keeps the totals' contention down.
constexpr std::size_t kMaxBlocks = 2048;

unsigned stride_blocks(std::size_t n)
{
    return static_cast<unsigned>(
        std::min(kMaxBlocks, std::max<std::size_t>((n + kThreads - 1) / kThreads, 1)));
}

__device__ __forceinline__ bool same_class(const hbfsim_amd_access_class& a,
                                           const hbfsim_amd_access_class& b)
{
    return a.operation == b.operation && a.bytes == b.bytes &&
           a.queue_bucket == b.queue_bucket && a.locality_bucket == b.locality_bucket;
}

// One 16-byte load (hipMalloc and torch align further; the ABI asks for 4).
__device__ __forceinline__ hbfsim_amd_access_class load_class(const hbfsim_amd_access_class* p,
                                                              std::size_t i, bool aligned)
{
    hbfsim_amd_access_class c;
    if (aligned) {
        const uint4 v = reinterpret_cast<const uint4*>(p)[i];
        c.operation = v.x;
        c.bytes = v.y;
        c.queue_bucket = v.z;
        c.locality_bucket = v.w;
    } else {
        c = p[i];
    }
    return c;
}

bool aligned16(const void* p) { return (reinterpret_cast<std::uintptr_t>(p) & 15u) == 0; }

// ---- the class table ------------------------------------------------------
// slot: kEmpty, a request index, or kSeen | index into the seen classes.  A
// slot is set once (compare-and-swap from empty) and never changes, and what
// it names is read-only, so readers need no lock: a stale "empty" only leads
// to a compare-and-swap that returns the slot's value.
constexpr std::uint64_t kEmpty = ~0ull;
constexpr std::uint64_t kSeen = 1ull << 63;
constexpr std::uint32_t kNone = 0xffffffffu;
constexpr std::uint32_t kProbes = 64;  // then the table counts as too small
constexpr std::uint32_t kProbesFree = 16;  // from here on also where another lookup said so

struct ClassTable {
    unsigned long long* slot;            // [mask + 1]
    std::uint32_t* first;                // [mask + 1], the caller's use
    std::uint64_t mask;
    std::uint32_t probes;                // probe limit; 0: none (the largest table, class_table.hpp)
    const hbfsim_amd_access_class* access;
    const hbfsim_amd_access_class* seen;
    std::uint32_t* overflow;             // set when the table is too small; then the classes sampled
    std::uint32_t sample_limit;          // the most of those (class_table.hpp)
    bool aligned;                        // access lies on 16 bytes (seen always does)
};

__device__ __forceinline__ std::uint64_t class_hash(const hbfsim_amd_access_class& c)
{
    std::uint64_t h = class_hi(c) * 0x9e3779b97f4a7c15ull ^ class_lo(c);
    h = (h ^ (h >> 32)) * 0xd6e8feb86659fd93ull;
    h = (h ^ (h >> 29)) * 0xd6e8feb86659fd93ull;
    return h ^ (h >> 32);
}

// The slot of class c, taken for `name` if the class has none yet.  Returns
// kEmpty when the probe limit is reached.
__device__ __forceinline__ std::uint64_t class_slot(const ClassTable& t,
                                                    const hbfsim_amd_access_class& c,
                                                    std::uint64_t name, std::uint64_t& found)
{
    std::uint64_t s = class_hash(c) & t.mask;
    for (std::uint32_t k = 0;; ++k) {
        unsigned long long v = t.slot[s];
        if (v == kEmpty) {
            v = atomicCAS(&t.slot[s], static_cast<unsigned long long>(kEmpty),
                          static_cast<unsigned long long>(name));
            if (v == kEmpty) {
                found = name;
                return s;
            }
        }
        const hbfsim_amd_access_class o = (v & kSeen) != 0
                                              ? load_class(t.seen, v & ~kSeen, true)
                                              : load_class(t.access, v, t.aligned);
        if (same_class(o, c)) {
            found = v;
            return s;
        }
        if (t.probes != 0 && k >= kProbesFree) {
            // (asked for only here: the one word is slow to read from everywhere,
            // 170 us for a pass over 4M requests)
            if (k >= t.probes || __hip_atomic_load(t.overflow, __ATOMIC_RELAXED,
                                                   __HIP_MEMORY_SCOPE_AGENT) != 0) {
                return kEmpty;
            }
        }
        s = (s + 1) & t.mask;
    }
}

// The slots of four requests at once (i, i + step, ...; those below n): their
// classes, first-probe slots and representatives are each loaded together, so
// the three dependent loads of a lookup overlap over four requests.  Requests
// whose first probe is not their class go through class_slot.
constexpr int kAtOnce = 4;

__device__ __forceinline__ void class_slots(const ClassTable& t, std::size_t i, std::size_t step,
                                            std::size_t n, hbfsim_amd_access_class c[kAtOnce],
                                            std::uint64_t at[kAtOnce],
                                            std::uint64_t found[kAtOnce])
{
    hbfsim_amd_access_class o[kAtOnce];
#pragma unroll
    for (int k = 0; k < kAtOnce; ++k) {
        const std::size_t j = i + k * step;
        c[k] = load_class(t.access, j < n ? j : i, t.aligned);
    }
#pragma unroll
    for (int k = 0; k < kAtOnce; ++k) {
        at[k] = class_hash(c[k]) & t.mask;
        found[k] = t.slot[at[k]];
    }
#pragma unroll
    for (int k = 0; k < kAtOnce; ++k) {
        const bool old = (found[k] & kSeen) != 0 && found[k] != kEmpty;
        const hbfsim_amd_access_class* from = old ? t.seen : t.access;
        const std::uint64_t where = found[k] == kEmpty ? i : found[k] & ~kSeen;
        o[k] = load_class(from, where, old || t.aligned);
    }
#pragma unroll
    for (int k = 0; k < kAtOnce; ++k) {
        if (i + k * step < n && (found[k] == kEmpty || !same_class(o[k], c[k]))) {
            at[k] = class_slot(t, c[k], i + k * step, found[k]);
        }
    }
}

// An empty table would meet every thread of a full launch with a
// compare-and-swap at once (203 us instead of 61 at 4M requests): a sample of
// the batch, spread evenly over it, takes its classes' slots first.  The
// classes among it say whether the table is worth trying.
__global__ __launch_bounds__(kThreads) void k_class_sample(ClassTable t, std::size_t n)
{
    const std::size_t k = static_cast<std::size_t>(blockIdx.x) * kThreads + threadIdx.x;
    const std::size_t i = k * (n / kSample);
    bool fresh = false;
    if (k < kSample && i < n) {
        std::uint64_t found = kEmpty;
        // (a probe limit reached here is reached again by the full pass)
        const std::uint64_t at =
            class_slot(t, load_class(t.access, i, t.aligned), i, found);
        fresh = at == kEmpty || found == i;
    }
    const std::uint64_t m = __ballot(fresh);
    if ((threadIdx.x & 63) == 0 && m != 0) {
        atomicAdd(&t.overflow[1], static_cast<std::uint32_t>(__popcll(m)));
    }
}

// Whether the sample says that the table is too small: a full pass over it
// would be thrown away (1M classes in 2^16 slots: 64 probes for each of 4M
// requests).
__device__ __forceinline__ bool too_small(const ClassTable& t)
{
    return t.overflow[1] > t.sample_limit;
}

// The classes earlier batches saw (all different) take their slots first.
__global__ __launch_bounds__(kThreads) void k_seen_insert(ClassTable t, std::size_t seen)
{
    const std::size_t stride = static_cast<std::size_t>(gridDim.x) * kThreads;
    for (std::size_t k = static_cast<std::size_t>(blockIdx.x) * kThreads + threadIdx.x; k < seen;
         k += stride) {
        std::uint64_t found;
        if (class_slot(t, load_class(t.seen, k, true), kSeen | k, found) == kEmpty) {
            *t.overflow = 1;
            return;
        }
    }
}

__device__ __forceinline__ std::uint64_t wave_sum(std::uint64_t v)
{
    for (int off = 32; off > 0; off >>= 1) {
        v += __shfl_down(v, off);
    }
    return v;
}

// Sum of v over the workgroup, in thread 0.
__device__ __forceinline__ std::uint64_t block_sum(std::uint64_t v)
{
    __shared__ std::uint64_t part[kThreads / 64];
    v = wave_sum(v);
    __syncthreads();  // (a sum before this one has been read)
    if ((threadIdx.x & 63) == 0) {
        part[threadIdx.x / 64] = v;
    }
    __syncthreads();
    v = 0;
    for (int w = 0; w < kThreads / 64; ++w) {
        v += part[w];
    }
    return v;
}

// This workgroup's run of `slots` table slots.
struct SlotRun {
    std::uint64_t begin, end;
};

__device__ __forceinline__ SlotRun slot_run(std::uint64_t slots)
{
    const std::uint64_t per =
        (slots + static_cast<std::uint64_t>(gridDim.x) * kThreads - 1) /
        (static_cast<std::uint64_t>(gridDim.x) * kThreads) * kThreads;
    const std::uint64_t b = blockIdx.x * per;
    return SlotRun{b < slots ? b : slots, b + per < slots ? b + per : slots};
}

// Numbers the slots that `take` accepts, from *count on, and hands each to
// `emit`: counted first, so that a workgroup asks for its numbers with one
// atomic (one per wave took 0.6 ms over 2^23 slots, one per slot 1.6).
template <typename Take, typename Emit>
__device__ __forceinline__ void compact_slots(std::uint64_t slots, unsigned long long* count,
                                              Take take, Emit emit)
{
    __shared__ unsigned long long start;
    __shared__ std::uint32_t w_count[kThreads / 64];
    const SlotRun run = slot_run(slots);
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    std::uint64_t own = 0;
    for (std::uint64_t s = run.begin + threadIdx.x; s < run.end; s += kThreads) {
        own += take(s) ? 1u : 0u;
    }
    const std::uint64_t total = block_sum(own);
    if (total == 0) {
        return;  // (the same in every thread)
    }
    if (threadIdx.x == 0) {
        start = atomicAdd(count, static_cast<unsigned long long>(total));
    }
    __syncthreads();
    std::uint64_t at = start;
    for (std::uint64_t b = run.begin; b < run.end; b += kThreads) {
        const std::uint64_t s = b + threadIdx.x;
        const bool taken = s < run.end && take(s);
        const std::uint64_t m = __ballot(taken);
        if (lane == 0) {
            w_count[wave] = static_cast<std::uint32_t>(__popcll(m));
        }
        __syncthreads();
        std::uint64_t mine = at + __popcll(m & ((1ull << lane) - 1));
        for (int w = 0; w < kThreads / 64; ++w) {
            mine += w < wave ? w_count[w] : 0u;
            at += w_count[w];
        }
        if (taken) {
            emit(s, mine);
        }
        __syncthreads();
    }
}

// flags[i] = warm-up or hash decision (calibrator.cpp:86-95), counted in
// totals[0]; each unseen class's first request goes to first[slot].
// Reads 16 B and writes 1 B per request (55 us at 4M); the table (768 KiB) stays
// in the caches.
__global__ __launch_bounds__(kThreads) void k_sampler_pass(
    ClassTable t, const std::uint64_t* sequence, std::uint64_t first_sequence, std::size_t n,
    std::uint32_t warmup, std::uint64_t threshold, std::uint64_t seed, std::uint8_t* flags,
    unsigned long long* totals)
{
    __shared__ unsigned long long part[kThreads / 64];
    const std::size_t stride = static_cast<std::size_t>(gridDim.x) * kThreads;
    std::uint64_t count = 0;
    bool full = too_small(t);  // then the host tries again with a larger table
    if (full) {
        *t.overflow = 1;
    }
    for (std::size_t b = static_cast<std::size_t>(blockIdx.x) * kThreads + threadIdx.x;
         b < n && !full; b += stride * kAtOnce) {
        hbfsim_amd_access_class cs[kAtOnce];
        std::uint64_t at[kAtOnce], found[kAtOnce];
        class_slots(t, b, stride, n, cs, at, found);
#pragma unroll
        for (int k = 0; k < kAtOnce; ++k) {
            const std::size_t i = b + k * stride;
            if (i >= n) {
                continue;
            }
            const hbfsim_amd_access_class c = cs[k];
            const std::uint64_t s = sequence != nullptr ? sequence[i] : first_sequence + i;
            std::uint64_t v = s ^ seed;
            v ^= static_cast<std::uint64_t>(c.bytes) << 17;
            v ^= static_cast<std::uint64_t>(c.queue_bucket) << 33;
            v ^= static_cast<std::uint64_t>(c.locality_bucket) << 49;
            v ^= static_cast<std::uint64_t>(c.operation) << 61;
            const bool hit = s < warmup || mix(v) <= threshold;
            flags[i] = hit ? 1 : 0;
            count += hit ? 1u : 0u;
            if (at[k] == kEmpty) {
                *t.overflow = 1;
                full = true;
            } else if ((found[k] & kSeen) == 0 && i < t.first[at[k]]) {
                atomicMin(&t.first[at[k]], static_cast<std::uint32_t>(i));
            }
        }
    }
    count = wave_sum(count);
    if ((threadIdx.x & 63) == 0) {
        part[threadIdx.x / 64] = count;
    }
    __syncthreads();
    if (threadIdx.x == 0) {
        std::uint64_t sum = 0;
        for (int w = 0; w < kThreads / 64; ++w) {
            sum += part[w];
        }
        if (sum != 0) {
            atomicAdd(&totals[0], static_cast<unsigned long long>(sum));
        }
    }
}

// The first request of every class new to the sampler is a reference request.
// totals[0] counts those not flagged already, totals[1] the new classes.
__global__ __launch_bounds__(kThreads) void k_sampler_first(ClassTable t, std::uint8_t* flags,
                                                            unsigned long long* totals)
{
    if (*t.overflow != 0) {
        return;
    }
    const SlotRun run = slot_run(t.mask + 1);
    std::uint64_t fresh = 0, raised = 0;
    for (std::uint64_t s = run.begin + threadIdx.x; s < run.end; s += kThreads) {
        const std::uint32_t i = t.first[s];
        if (i != kNone) {
            ++fresh;
            if (flags[i] == 0) {
                flags[i] = 1;
                ++raised;
            }
        }
    }
    fresh = block_sum(fresh);
    if (fresh == 0) {
        return;  // (the same in every thread)
    }
    raised = block_sum(raised);
    if (threadIdx.x == 0) {
        if (raised != 0) {
            atomicAdd(&totals[0], static_cast<unsigned long long>(raised));
        }
        atomicAdd(&totals[1], static_cast<unsigned long long>(fresh));
    }
}

// The new classes join the seen ones, in no particular order.
__global__ __launch_bounds__(kThreads) void k_sampler_grow(ClassTable t,
                                                           hbfsim_amd_access_class* out,
                                                           unsigned long long* at)
{
    compact_slots(
        t.mask + 1, at, [&](std::uint64_t s) { return t.first[s] != kNone; },
        [&](std::uint64_t s, std::uint64_t k) {
            out[k] = load_class(t.access, t.first[s], t.aligned);
        });
}

// Calibrator: slot_of[i] = the slot of request i's class; the latencies'
// maximum and whether one is 0.
__global__ __launch_bounds__(kThreads) void k_calib_classes(ClassTable t,
                                                            const std::uint64_t* latency,
                                                            std::size_t n, std::uint32_t* slot_of,
                                                            unsigned long long* max_latency,
                                                            std::uint32_t* bad)
{
    __shared__ unsigned long long part[kThreads / 64];
    const std::size_t stride = static_cast<std::size_t>(gridDim.x) * kThreads;
    unsigned long long most = 0;
    bool full = too_small(t);  // (the next table's pass then checks every latency)
    if (full) {
        *t.overflow = 1;
    }
    for (std::size_t b = static_cast<std::size_t>(blockIdx.x) * kThreads + threadIdx.x;
         b < n && !full; b += stride * kAtOnce) {
        hbfsim_amd_access_class cs[kAtOnce];
        std::uint64_t at[kAtOnce], found[kAtOnce], v[kAtOnce];
#pragma unroll
        for (int k = 0; k < kAtOnce; ++k) {
            v[k] = b + k * stride < n ? latency[b + k * stride] : 1;
        }
        class_slots(t, b, stride, n, cs, at, found);
#pragma unroll
        for (int k = 0; k < kAtOnce; ++k) {
            if (b + k * stride >= n) {
                continue;
            }
            if (v[k] == 0) {
                *bad = 1;
            }
            most = v[k] > most ? v[k] : most;
            if (at[k] == kEmpty) {
                *t.overflow = 1;
                full = true;
            } else {
                slot_of[b + k * stride] = static_cast<std::uint32_t>(at[k]);
            }
        }
    }
    for (int off = 32; off > 0; off >>= 1) {
        const unsigned long long o = __shfl_down(most, off);
        most = o > most ? o : most;
    }
    if ((threadIdx.x & 63) == 0) {
        part[threadIdx.x / 64] = most;
    }
    __syncthreads();
    if (threadIdx.x == 0) {
        for (int w = 1; w < kThreads / 64; ++w) {
            most = part[w] > most ? part[w] : most;
        }
        atomicMax(max_latency, most);
    }
}

// The table's classes as a list (in no particular order): their slots and
// keys (high, low).
__global__ __launch_bounds__(kThreads) void k_calib_list(ClassTable t, std::uint32_t* list,
                                                         ulonglong2* keys,
                                                         unsigned long long* count)
{
    if (*t.overflow != 0) {
        return;
    }
    compact_slots(
        t.mask + 1, count, [&](std::uint64_t s) { return t.slot[s] != kEmpty; },
        [&](std::uint64_t s, std::uint64_t k) {
            list[k] = static_cast<std::uint32_t>(s);
            const hbfsim_amd_access_class c = load_class(t.access, t.slot[s], t.aligned);
            keys[k] = make_ulonglong2(class_hi(c), class_lo(c));
        });
}

// Up to this many classes are numbered by counting, for each, the classes
// below it (k^2 compares, one wave per class reading the 16-byte keys from L2:
// 2,000 classes take 15 us, 8,192 read 1 GiB); more are sorted (two radix sorts,
// about 0.2 ms of launches).
constexpr std::size_t kCountedClasses = 8192;

// number[slot] = how many classes are below that slot's class.
__global__ __launch_bounds__(kThreads) void k_calib_number(const ulonglong2* keys,
                                                           const std::uint32_t* list,
                                                           std::uint32_t classes,
                                                           std::uint32_t* number)
{
    const std::uint32_t j = blockIdx.x * (kThreads / 64) + (threadIdx.x >> 6);
    if (j >= classes) {
        return;
    }
    const ulonglong2 own = keys[j];
    std::uint32_t below = 0;
#pragma unroll 4
    for (std::uint32_t m = threadIdx.x & 63; m < classes; m += 64) {
        const ulonglong2 k = keys[m];
        below += k.x < own.x || (k.x == own.x && k.y < own.y) ? 1u : 0u;
    }
    for (int off = 32; off > 0; off >>= 1) {
        below += __shfl_down(below, off);
    }
    if ((threadIdx.x & 63) == 0) {
        number[list[j]] = below;
    }
}

// The same by sorting: key[j] = the low or high class key of list entry
// idx[j] (j itself when idx is null); then number[list[idx[j]]] = j.
template <bool kHi>
__global__ __launch_bounds__(kThreads) void k_calib_class_keys(const ulonglong2* keys,
                                                               const std::uint32_t* idx,
                                                               std::size_t classes,
                                                               std::uint64_t* key,
                                                               std::uint32_t* iota)
{
    const std::size_t j = static_cast<std::size_t>(blockIdx.x) * kThreads + threadIdx.x;
    if (j < classes) {
        const std::uint32_t m = idx != nullptr ? idx[j] : static_cast<std::uint32_t>(j);
        key[j] = kHi ? keys[m].x : keys[m].y;
        if (iota != nullptr) {
            iota[j] = m;
        }
    }
}

__global__ __launch_bounds__(kThreads) void k_calib_renumber(const std::uint32_t* list,
                                                             const std::uint32_t* idx,
                                                             std::size_t classes,
                                                             std::uint32_t* number)
{
    const std::size_t j = static_cast<std::size_t>(blockIdx.x) * kThreads + threadIdx.x;
    if (j < classes) {
        number[list[idx[j]]] = static_cast<std::uint32_t>(j);
    }
}

// Sort keys: the class number above `shift` bits of latency (K 32 or 64 bits
// wide, whichever holds both).
template <typename K>
__global__ __launch_bounds__(kThreads) void k_calib_keys(const std::uint32_t* slot_of,
                                                         const std::uint32_t* number,
                                                         const std::uint64_t* latency,
                                                         std::size_t n, unsigned shift, K* key)
{
    const std::size_t stride = static_cast<std::size_t>(gridDim.x) * kThreads;
    for (std::size_t i = static_cast<std::size_t>(blockIdx.x) * kThreads + threadIdx.x; i < n;
         i += stride) {
        key[i] = (static_cast<K>(number[slot_of[i]]) << shift) | static_cast<K>(latency[i]);
    }
}

// Where the two do not fit 64 bits: the class numbers as payload.
__global__ __launch_bounds__(kThreads) void k_calib_numbers(const std::uint32_t* slot_of,
                                                            const std::uint32_t* number,
                                                            std::size_t n, std::uint32_t* out)
{
    const std::size_t stride = static_cast<std::size_t>(gridDim.x) * kThreads;
    for (std::size_t i = static_cast<std::size_t>(blockIdx.x) * kThreads + threadIdx.x; i < n;
         i += stride) {
        out[i] = number[slot_of[i]];
    }
}

// starts[c] = the first sorted sample of class c (every class has one).
template <typename K>
__global__ __launch_bounds__(kThreads) void k_calib_starts(const K* key, std::size_t n,
                                                           unsigned shift, std::uint32_t* starts)
{
    const std::size_t stride = static_cast<std::size_t>(gridDim.x) * kThreads;
    for (std::size_t j = static_cast<std::size_t>(blockIdx.x) * kThreads + threadIdx.x; j < n;
         j += stride) {
        const K c = key[j] >> shift;
        if (j == 0 || (key[j - 1] >> shift) != c) {
            starts[c] = static_cast<std::uint32_t>(j);
        }
    }
}

// 128-bit sum as two 64-bit words.
struct U128 {
    std::uint64_t lo, hi;
};

__device__ __forceinline__ U128 add128(U128 a, U128 b)
{
    U128 r;
    r.lo = a.lo + b.lo;
    r.hi = a.hi + b.hi + (r.lo < a.lo ? 1ull : 0ull);
    return r;
}

// floor(s / d) for d < 2^32 and a quotient below 2^64, in 32-bit digits.
__device__ __forceinline__ std::uint64_t div128(U128 s, std::uint64_t d)
{
    const std::uint64_t digit[4] = {s.hi >> 32, s.hi & 0xffffffffull, s.lo >> 32,
                                    s.lo & 0xffffffffull};
    std::uint64_t r = 0, q = 0;
    for (int k = 0; k < 4; ++k) {
        const std::uint64_t cur = (r << 32) | digit[k];
        q = (q << 32) | (cur / d);
        r = cur % d;
    }
    return q;
}

// calibrator.cpp:20-30: the sample of rank ceil(size * num / den), 1-based,
// clamped to the segment.
__device__ __forceinline__ std::uint64_t rank_index(std::uint64_t size, std::uint32_t num,
                                                    std::uint32_t den)
{
    const std::uint64_t rank = (size * num + den - 1) / den;
    const std::uint64_t index = rank == 0 ? 0 : rank - 1;
    return index < size - 1 ? index : size - 1;
}

// A sum of doubles as an unevaluated pair, each addition exact to the pair's
// precision (Knuth's two-sum), so that the order of a split sum does not show
// in the result.
struct Pair {
    double hi, lo;
};

__device__ __forceinline__ Pair pair_add(Pair a, double b)
{
    const double s = a.hi + b;
    const double t = s - a.hi;
    const double e = (a.hi - (s - t)) + (b - t);
    return Pair{s, a.lo + e};
}

__device__ __forceinline__ Pair pair_join(Pair a, Pair b)
{
    Pair r = pair_add(a, b.hi);
    r.lo += b.lo;
    return r;
}

// Sums over samples of one class: the latencies in 128 bits, and the first two
// moments of their logarithms about the logarithm of the class's median.  The
// median lies within one deviation of the mean, so that taking the mean's
// square off the second moment costs at most one bit, and one pass over the
// samples gives both statistics.
struct ClassSum {
    std::uint64_t lo, hi;
    Pair m1, m2;
};

__device__ __forceinline__ ClassSum sum_join(const ClassSum& a, const ClassSum& b)
{
    const U128 s = add128(U128{a.lo, a.hi}, U128{b.lo, b.hi});
    return ClassSum{s.lo, s.hi, pair_join(a.m1, b.m1), pair_join(a.m2, b.m2)};
}

// The sum over kLanes neighbouring lanes, in the first of them.
template <int kLanes>
__device__ __forceinline__ ClassSum lanes_sum(ClassSum v)
{
    for (int off = kLanes / 2; off > 0; off >>= 1) {
        ClassSum o;
        o.lo = __shfl_down(static_cast<unsigned long long>(v.lo), off);
        o.hi = __shfl_down(static_cast<unsigned long long>(v.hi), off);
        o.m1 = Pair{__shfl_down(v.m1.hi, off), __shfl_down(v.m1.lo, off)};
        o.m2 = Pair{__shfl_down(v.m2.hi, off), __shfl_down(v.m2.lo, off)};
        v = sum_join(v, o);
    }
    return v;
}

// The sorted samples: `key` holds the latency below `shift` bits and the class
// number above them; with `cls` it is the latency alone and cls the number.
template <typename K>
struct Samples {
    const K* key;
    const std::uint32_t* cls;
    unsigned shift;
    std::uint64_t mask;
    const std::uint32_t* starts;  // [classes]
    std::size_t classes, n;
    __device__ std::uint64_t latency(std::size_t j) const
    {
        return static_cast<std::uint64_t>(key[j]) & mask;
    }
    __device__ std::size_t number(std::size_t j) const
    {
        return cls != nullptr ? cls[j] : static_cast<std::size_t>(key[j] >> shift);
    }
    __device__ std::size_t end(std::size_t c) const { return c + 1 < classes ? starts[c + 1] : n; }
};

// This lane's share of samples [b, e): every kLanes-th, kAhead loads at once.
template <int kLanes, int kAhead, typename K>
__device__ __forceinline__ void add_samples(ClassSum& a, const Samples<K>& in, std::size_t b,
                                            std::size_t e, double centre, int lane)
{
    for (std::size_t j0 = b + lane; j0 < e; j0 += kLanes * kAhead) {
        K v[kAhead];
#pragma unroll
        for (int k = 0; k < kAhead; ++k) {
            const std::size_t j = j0 + static_cast<std::size_t>(k) * kLanes;
            v[k] = in.key[j < e ? j : j0];
        }
#pragma unroll
        for (int k = 0; k < kAhead; ++k) {
            if (j0 + static_cast<std::size_t>(k) * kLanes < e) {
                const std::uint64_t x = static_cast<std::uint64_t>(v[k]) & in.mask;
                const U128 s = add128(U128{a.lo, a.hi}, U128{x, 0});
                const double d = log(static_cast<double>(x)) - centre;
                a = ClassSum{s.lo, s.hi, pair_add(a.m1, d), pair_add(a.m2, d * d)};
            }
        }
    }
}

template <typename K>
__device__ __forceinline__ double median_log(const Samples<K>& in, std::size_t c)
{
    const std::size_t s = in.starts[c];
    return log(static_cast<double>(in.latency(s + rank_index(in.end(c) - s, 50, 100))));
}

// Whole runs of kPart sorted samples that lie within one class are summed by a
// wave each, so that one large class does not hold up the rest (one 256-thread
// block per class took 248 us at 4M samples of 2,000 classes, its largest
// holding 90,000).
constexpr std::uint32_t kPart = 512;

template <typename K>
__global__ __launch_bounds__(kThreads) void k_calib_part(Samples<K> in, ClassSum* parts)
{
    const std::size_t part =
        static_cast<std::size_t>(blockIdx.x) * (kThreads / 64) + (threadIdx.x >> 6);
    const int lane = threadIdx.x & 63;
    const std::size_t b = part * kPart, e = b + kPart;
    if (e > in.n) {
        return;
    }
    const std::size_t c = in.number(b);
    if (in.number(e - 1) != c) {
        return;
    }
    ClassSum v{0, 0, {0.0, 0.0}, {0.0, 0.0}};
    add_samples<64, kPart / 64>(v, in, b, e, median_log(in, c), lane);
    v = lanes_sum<64>(v);
    if (lane == 0) {
        parts[part] = v;
    }
}

// kLanes lanes per class: its whole parts and the samples on either side of
// them, in a fixed order (the result depends only on the samples), and the
// estimate of calibrator.cpp:107-136.
template <typename K, int kLanes>
__global__ __launch_bounds__(kThreads) void k_calib_rows(ClassTable t, const std::uint32_t* list,
                                                         const std::uint32_t* number, Samples<K> in,
                                                         const ClassSum* parts,
                                                         hbfsim_amd_calibration* rows)
{
    const int lane = threadIdx.x % kLanes;
    const std::size_t stride = static_cast<std::size_t>(gridDim.x) * (kThreads / kLanes);
    for (std::size_t j = static_cast<std::size_t>(blockIdx.x) * (kThreads / kLanes) +
                         threadIdx.x / kLanes;
         j < in.classes; j += stride) {
        const std::uint32_t slot = list[j];
        const std::size_t c = number[slot];
        const std::size_t s = in.starts[c], e = in.end(c);
        const std::uint64_t size = e - s;
        const double centre = median_log(in, c);
        const std::size_t p0 = (s + kPart - 1) / kPart, p1 = e / kPart;
        ClassSum v{0, 0, {0.0, 0.0}, {0.0, 0.0}};
        constexpr int kAhead = kLanes == 64 ? 8 : 2;
        if (p0 < p1) {
            for (std::size_t p = p0 + lane; p < p1; p += kLanes) {
                v = sum_join(v, parts[p]);
            }
            add_samples<kLanes, kAhead>(v, in, s, p0 * kPart, centre, lane);
            add_samples<kLanes, kAhead>(v, in, p1 * kPart, e, centre, lane);
        } else {
            add_samples<kLanes, kAhead>(v, in, s, e, centre, lane);
        }
        v = lanes_sum<kLanes>(v);
        if (lane == 0) {
            const double m1 = (v.m1.hi + v.m1.lo) / static_cast<double>(size);
            const double m2 = (v.m2.hi + v.m2.lo) / static_cast<double>(size);
            const double variance = m2 - m1 * m1;
            hbfsim_amd_calibration r;
            r.access = load_class(t.access, t.slot[slot], t.aligned);
            r.count = size;
            r.mean_ns = div128(U128{v.lo, v.hi}, size);
            r.p50_ns = in.latency(s + rank_index(size, 50, 100));
            r.p95_ns = in.latency(s + rank_index(size, 95, 100));
            r.p99_ns = in.latency(s + rank_index(size, 99, 100));
            r.log_mean = centre + m1;
            r.log_sigma = sqrt(variance > 0.0 ? variance : 0.0);
            rows[c] = r;
        }
    }
}

// The buffers of the table and whatever else the call adds to `plan`.
struct TablePlan {
    ScratchPlan plan;
    std::size_t o_slot, o_first, o_words;
    std::uint64_t cap;
    explicit TablePlan(std::uint64_t slots) : cap(slots)
    {
        o_slot = plan.add<unsigned long long>(slots);
        o_first = plan.add<std::uint32_t>(slots);
        o_words = plan.add<unsigned long long>(4);
    }
};

}  // namespace

struct sampler_state {
    std::uint32_t warmup;
    std::uint64_t threshold;
    std::uint64_t seed;
    hbfsim_amd_access_class* seen_class = nullptr;  // classes seen, in no order
    std::size_t seen = 0;
    std::size_t seen_cap = 0;
};

int sampler_create(std::uint32_t warmup, double sample_rate, std::uint64_t seed,
                   sampler_state** out)
{
    if (out == nullptr) {
        return HBFSIM_INVALID_ARGUMENT;
    }
    *out = nullptr;
    // calibrator.cpp:67-81
    if (!std::isfinite(sample_rate) || sample_rate < 0.0 || sample_rate > 1.0) {
        return HBFSIM_INVALID_ARGUMENT;
    }
    auto* s = new (std::nothrow) sampler_state;
    if (s == nullptr) {
        return HBFSIM_INVALID_ARGUMENT;
    }
    scratch_hold();
    s->warmup = warmup;
    s->seed = seed;
    s->threshold = sample_rate >= 1.0
                       ? std::numeric_limits<std::uint64_t>::max()
                       : static_cast<std::uint64_t>(
                             sample_rate * static_cast<long double>(
                                               std::numeric_limits<std::uint64_t>::max()));
    *out = s;
    return HBFSIM_OK;
}

void sampler_destroy(sampler_state* s)
{
    if (s != nullptr) {
        (void)hipFree(s->seen_class);
        delete s;
        scratch_drop();
    }
}

int sampler_reference(sampler_state* s, const hbfsim_amd_access_class* d_access,
                      const std::uint64_t* d_sequence, std::uint64_t first_sequence,
                      std::size_t n, std::uint8_t* d_flags, std::uint64_t* references,
                      void* stream_ptr)
{
    if (s == nullptr || (n != 0 && (d_access == nullptr || d_flags == nullptr))) {
        return HBFSIM_INVALID_ARGUMENT;
    }
    if (references != nullptr) {
        *references = 0;
    }
    if (n == 0) {
        return HBFSIM_OK;
    }
    if (n > 0xffffffffull) {
        return HBFSIM_UNSUPPORTED;
    }
    hipStream_t stream = static_cast<hipStream_t>(stream_ptr);
    const std::uint64_t most = most_slots(n, s->seen);
    std::uint64_t cap = first_slots(s->seen, most);
    // references, new classes, overflow | classes sampled << 32, -
    unsigned long long host[4] = {0, 0, 0, 0};
    for (;; cap = next_slots(cap, most, static_cast<std::uint32_t>(host[2] >> 32))) {
        TablePlan p(cap);
        ScratchLease lease(p.plan.bytes, stream);
        if (!lease.ok()) {
            return HBFSIM_CUDA_ERROR;
        }
        auto* words = lease.at<unsigned long long>(p.o_words);
        ClassTable t{lease.at<unsigned long long>(p.o_slot), lease.at<std::uint32_t>(p.o_first),
                     cap - 1, cap < most ? kProbes : 0u, d_access, s->seen_class,
                     reinterpret_cast<std::uint32_t*>(words + 2), sample_limit(cap, most),
                     aligned16(d_access)};
        hipError_t err = hipMemsetAsync(t.slot, 0xff, p.o_words - p.o_slot, stream);
        if (err == hipSuccess) err = hipMemsetAsync(words, 0, sizeof(host), stream);
        if (err != hipSuccess) {
            return HBFSIM_CUDA_ERROR;
        }
        if (s->seen != 0) {
            hipLaunchKernelGGL(k_seen_insert, dim3(stride_blocks(s->seen)), dim3(kThreads), 0, stream,
                               t, s->seen);
        }
        if (s->seen == 0 && n >= 4 * kSample) {
            hipLaunchKernelGGL(k_class_sample, dim3(blocks_for(kSample)), dim3(kThreads), 0,
                               stream, t, n);
        }
        hipLaunchKernelGGL(k_sampler_pass, dim3(stride_blocks(n)), dim3(kThreads), 0, stream, t,
                           d_sequence, first_sequence, n, s->warmup, s->threshold, s->seed,
                           d_flags, words);
        hipLaunchKernelGGL(k_sampler_first, dim3(walk_blocks(cap)), dim3(kThreads), 0, stream, t,
                           d_flags, words);
        err = hipGetLastError();
        if (err == hipSuccess) err = hipMemcpyAsync(host, words, sizeof(host),
                                                    hipMemcpyDeviceToHost, stream);
        if (err == hipSuccess) err = hipStreamSynchronize(stream);
        if (err != hipSuccess) {
            return HBFSIM_CUDA_ERROR;
        }
        if (static_cast<std::uint32_t>(host[2]) != 0) {
            continue;  // the table was too small; the largest never is
        }
        if (host[1] != 0) {
            const std::size_t total = s->seen + host[1];
            hbfsim_amd_access_class* grown = s->seen_class;
            if (total > s->seen_cap) {
                const std::size_t room = total + total / 2 + 64;
                if (hipMalloc(reinterpret_cast<void**>(&grown),
                              room * sizeof(hbfsim_amd_access_class)) != hipSuccess) {
                    (void)hipGetLastError();
                    return HBFSIM_CUDA_ERROR;
                }
                if (s->seen != 0) {
                    err = hipMemcpyAsync(grown, s->seen_class,
                                         s->seen * sizeof(hbfsim_amd_access_class),
                                         hipMemcpyDeviceToDevice, stream);
                }
                if (err == hipSuccess) err = hipStreamSynchronize(stream);
                if (err != hipSuccess) {
                    (void)hipFree(grown);
                    return HBFSIM_CUDA_ERROR;
                }
                (void)hipFree(s->seen_class);
                s->seen_class = grown;
                s->seen_cap = room;
            }
            // words[3] counts the classes written from here on
            hipLaunchKernelGGL(k_sampler_grow, dim3(walk_blocks(cap)), dim3(kThreads), 0, stream, t,
                               s->seen_class + s->seen, words + 3);
            err = hipGetLastError();
            if (err == hipSuccess) err = hipStreamSynchronize(stream);
            if (err != hipSuccess) {
                return HBFSIM_CUDA_ERROR;
            }
            s->seen = total;
        }
        lease.synced(err);
        break;
    }
    if (references != nullptr) {
        *references = host[0];
    }
    return HBFSIM_OK;
}

namespace {

// The rest of a calibration once the classes are known: `classes` of them,
// latencies below 2^shift.  K: the width of the combined sort key; with kWide
// class and latency do not fit 64 bits together, the latencies are sorted with
// the class numbers as payload and then stably by class.
template <typename K, bool kWide>
int calibrate_rows(const ClassTable& t, const std::uint64_t* d_latency, std::size_t n,
                   const std::uint32_t* slot_of, const std::uint32_t* list,
                   const ulonglong2* keys, std::size_t classes, unsigned shift,
                   hbfsim_amd_calibration* d_rows, hipStream_t stream)
{
    const unsigned number_bits = [&] {
        unsigned b = 1;
        while ((std::uint64_t{1} << b) < classes) {
            ++b;
        }
        return b;
    }();
    const bool counted = classes <= kCountedClasses;
    const std::size_t parts = n / kPart;
    std::size_t tb_class = 0, tb_main = 0, tb_second = 0;
    hipError_t err = hipSuccess;
    if (!counted) {
        err = rocprim::radix_sort_pairs(nullptr, tb_class, static_cast<std::uint64_t*>(nullptr),
                                        static_cast<std::uint64_t*>(nullptr),
                                        static_cast<std::uint32_t*>(nullptr),
                                        static_cast<std::uint32_t*>(nullptr), classes, 0, 64,
                                        stream);
    }
    if (err == hipSuccess) {
        if constexpr (kWide) {
            err = rocprim::radix_sort_pairs(nullptr, tb_main, static_cast<std::uint64_t*>(nullptr),
                                            static_cast<std::uint64_t*>(nullptr),
                                            static_cast<std::uint32_t*>(nullptr),
                                            static_cast<std::uint32_t*>(nullptr), n, 0, shift,
                                            stream);
            if (err == hipSuccess) {
                err = rocprim::radix_sort_pairs(nullptr, tb_second,
                                                static_cast<std::uint32_t*>(nullptr),
                                                static_cast<std::uint32_t*>(nullptr),
                                                static_cast<std::uint64_t*>(nullptr),
                                                static_cast<std::uint64_t*>(nullptr), n, 0,
                                                number_bits, stream);
            }
        } else {
            err = rocprim::radix_sort_keys(nullptr, tb_main, static_cast<K*>(nullptr),
                                           static_cast<K*>(nullptr), n, 0, shift + number_bits,
                                           stream);
        }
    }
    if (err != hipSuccess) {
        return HBFSIM_CUDA_ERROR;
    }
    ScratchPlan p;
    const std::size_t o_starts = p.add<std::uint32_t>(classes);
    const std::size_t o_parts = p.add<ClassSum>(parts);
    const std::size_t o_a = p.add<K>(n), o_b = p.add<K>(n);
    const std::size_t o_na = p.add<std::uint32_t>(kWide ? n : 0);
    const std::size_t o_nb = p.add<std::uint32_t>(kWide ? n : 0);
    const std::size_t kc = counted ? 0 : classes;
    const std::size_t o_ka = p.add<std::uint64_t>(kc), o_kb = p.add<std::uint64_t>(kc);
    const std::size_t o_ia = p.add<std::uint32_t>(kc), o_ib = p.add<std::uint32_t>(kc);
    const std::size_t o_temp =
        p.add<unsigned char>(std::max(tb_class, std::max(tb_main, tb_second)));
    ScratchLease lease(p.bytes, stream);
    if (!lease.ok()) {
        return HBFSIM_CUDA_ERROR;
    }
    // Sorted class numbers are indices to what follows: nothing is launched after
    // a sort that failed (the lease then waits for what was).
    void* temp = lease.at<unsigned char>(o_temp);
    std::uint32_t* number = t.first;  // [slots]
    const dim3 block(kThreads);
    if (counted) {
        hipLaunchKernelGGL(k_calib_number, dim3(blocks_for(classes * 64)), block, 0, stream, keys,
                           list, static_cast<std::uint32_t>(classes), number);
    } else {
        auto* ka = lease.at<std::uint64_t>(o_ka);
        auto* kb = lease.at<std::uint64_t>(o_kb);
        auto* ia = lease.at<std::uint32_t>(o_ia);
        auto* ib = lease.at<std::uint32_t>(o_ib);
        hipLaunchKernelGGL((k_calib_class_keys<false>), dim3(blocks_for(classes)), block, 0,
                           stream, keys, static_cast<const std::uint32_t*>(nullptr), classes, ka,
                           ia);
        err = rocprim::radix_sort_pairs(temp, tb_class, ka, kb, ia, ib, classes, 0, 64, stream);
        if (err != hipSuccess) {
            return HBFSIM_CUDA_ERROR;
        }
        hipLaunchKernelGGL((k_calib_class_keys<true>), dim3(blocks_for(classes)), block, 0, stream,
                           keys, static_cast<const std::uint32_t*>(ib), classes, ka,
                           static_cast<std::uint32_t*>(nullptr));
        err = rocprim::radix_sort_pairs(temp, tb_class, ka, kb, ib, ia, classes, 0, 64, stream);
        if (err != hipSuccess) {
            return HBFSIM_CUDA_ERROR;
        }
        hipLaunchKernelGGL(k_calib_renumber, dim3(blocks_for(classes)), block, 0, stream, list,
                           static_cast<const std::uint32_t*>(ia), classes, number);
    }
    K* a = lease.at<K>(o_a);
    K* b = lease.at<K>(o_b);
    const K* sorted = b;
    auto* starts = lease.at<std::uint32_t>(o_starts);
    auto* psum = lease.at<ClassSum>(o_parts);
    const std::uint32_t* cls = nullptr;
    const dim3 wide(stride_blocks(n));
    if constexpr (kWide) {
        auto* na = lease.at<std::uint32_t>(o_na);
        auto* nb = lease.at<std::uint32_t>(o_nb);
        hipLaunchKernelGGL(k_calib_numbers, wide, block, 0, stream, slot_of, number, n, na);
        err = rocprim::radix_sort_pairs(temp, tb_main, d_latency, b, na, nb, n, 0, shift, stream);
        if (err == hipSuccess) {
            err = rocprim::radix_sort_pairs(temp, tb_second, nb, na, b, a, n, 0, number_bits,
                                            stream);
        }
        if (err != hipSuccess) {
            return HBFSIM_CUDA_ERROR;
        }
        sorted = a;
        cls = na;
        hipLaunchKernelGGL((k_calib_starts<std::uint32_t>), wide, block, 0, stream,
                           static_cast<const std::uint32_t*>(na), n, 0u, starts);
    } else {
        hipLaunchKernelGGL((k_calib_keys<K>), wide, block, 0, stream, slot_of, number, d_latency,
                           n, shift, a);
        err = rocprim::radix_sort_keys(temp, tb_main, a, b, n, 0, shift + number_bits, stream);
        if (err != hipSuccess) {
            return HBFSIM_CUDA_ERROR;
        }
        hipLaunchKernelGGL((k_calib_starts<K>), wide, block, 0, stream, sorted, n, shift, starts);
    }
    const std::uint64_t low_mask = kWide || shift >= 64 ? ~0ull : (1ull << shift) - 1;
    const Samples<K> in{sorted, cls, shift, low_mask, starts, classes, n};
    if (parts != 0) {
        hipLaunchKernelGGL((k_calib_part<K>), dim3(blocks_for(parts * 64)), block, 0, stream, in,
                           psum);
    }
    // a wave per class, or eight lanes where classes hold fewer than 32 samples
    // on average (4M samples of 4M classes: the whole call 19.5 ms with a wave
    // per class and a scan over the classes' parts, 2.2 ms now; 1M classes 10.0
    // and 1.4, 2,000 classes 438 and 429 us)
    const bool few = n / 32 < classes;
    const dim3 groups(static_cast<unsigned>(std::min<std::size_t>(
        std::size_t{1} << 20, blocks_for(classes * (few ? 8 : 64)))));
    hipLaunchKernelGGL((few ? k_calib_rows<K, 8> : k_calib_rows<K, 64>), groups, block, 0, stream,
                       t, list, number, in, psum, d_rows);
    err = hipGetLastError();
    if (err == hipSuccess) err = hipStreamSynchronize(stream);
    if (err != hipSuccess) {
        return HBFSIM_CUDA_ERROR;
    }
    lease.synced(err);
    return HBFSIM_OK;
}

}  // namespace

int calibrate(const hbfsim_amd_access_class* d_access, const std::uint64_t* d_latency,
              std::size_t n, hbfsim_amd_calibration* d_rows, std::size_t max_rows,
              std::size_t* rows_out, void* stream_ptr)
{
    if (rows_out == nullptr || (n != 0 && (d_access == nullptr || d_latency == nullptr))) {
        return HBFSIM_INVALID_ARGUMENT;
    }
    *rows_out = 0;
    if (n == 0) {
        return HBFSIM_OK;
    }
    if (n > 0xffffffffull) {
        return HBFSIM_UNSUPPORTED;
    }
    const ScratchHold hold;  // outlives every lease of the call
    hipStream_t stream = static_cast<hipStream_t>(stream_ptr);
    const std::uint64_t most = most_slots(n, 0, std::uint64_t{1} << 32);
    std::uint64_t cap = first_slots(0, most);
    // classes, largest latency, overflow | classes sampled << 32, zero latency
    unsigned long long host[4] = {0, 0, 0, 0};
    for (;; cap = next_slots(cap, most, static_cast<std::uint32_t>(host[2] >> 32))) {
        TablePlan p(cap);
        const std::size_t o_slot_of = p.plan.add<std::uint32_t>(n);
        const std::size_t o_list = p.plan.add<std::uint32_t>(std::min<std::uint64_t>(cap, n));
        const std::size_t o_keys = p.plan.add<ulonglong2>(std::min<std::uint64_t>(cap, n));
        ScratchLease lease(p.plan.bytes, stream);
        if (!lease.ok()) {
            return HBFSIM_CUDA_ERROR;
        }
        auto* words = lease.at<unsigned long long>(p.o_words);
        ClassTable t{lease.at<unsigned long long>(p.o_slot), lease.at<std::uint32_t>(p.o_first),
                     cap - 1, cap < most ? kProbes : 0u, d_access, nullptr,
                     reinterpret_cast<std::uint32_t*>(words + 2), sample_limit(cap, most),
                     aligned16(d_access)};
        auto* slot_of = lease.at<std::uint32_t>(o_slot_of);
        auto* list = lease.at<std::uint32_t>(o_list);
        auto* keys = lease.at<ulonglong2>(o_keys);
        hipError_t err = hipMemsetAsync(t.slot, 0xff, p.o_first - p.o_slot, stream);
        if (err == hipSuccess) err = hipMemsetAsync(words, 0, sizeof(host), stream);
        if (err != hipSuccess) {
            return HBFSIM_CUDA_ERROR;
        }
        if (n >= 4 * kSample) {
            hipLaunchKernelGGL(k_class_sample, dim3(blocks_for(kSample)), dim3(kThreads), 0,
                               stream, t, n);
        }
        hipLaunchKernelGGL(k_calib_classes, dim3(stride_blocks(n)), dim3(kThreads), 0, stream, t,
                           d_latency, n, slot_of, words + 1,
                           reinterpret_cast<std::uint32_t*>(words + 3));
        hipLaunchKernelGGL(k_calib_list, dim3(walk_blocks(cap)), dim3(kThreads), 0, stream, t, list,
                           keys, words);
        err = hipGetLastError();
        if (err == hipSuccess) err = hipMemcpyAsync(host, words, sizeof(host),
                                                    hipMemcpyDeviceToHost, stream);
        if (err == hipSuccess) err = hipStreamSynchronize(stream);
        if (err != hipSuccess) {
            return HBFSIM_CUDA_ERROR;
        }
        if (host[3] != 0) {
            return HBFSIM_INVALID_ARGUMENT;  // Calibrator::observe: latency_ns must be positive
        }
        if (static_cast<std::uint32_t>(host[2]) != 0) {
            continue;  // the table was too small; the largest never is
        }
        const std::size_t classes = host[0];
        *rows_out = classes;
        if (classes > max_rows || d_rows == nullptr) {
            return HBFSIM_INVALID_ARGUMENT;
        }
        unsigned shift = 1, number_bits = 1;
        while (shift < 64 && (host[1] >> shift) != 0) {
            ++shift;
        }
        while ((std::uint64_t{1} << number_bits) < classes) {
            ++number_bits;
        }
        const int st =
            shift + number_bits <= 32
                ? calibrate_rows<std::uint32_t, false>(t, d_latency, n, slot_of, list, keys, classes,
                                                       shift, d_rows, stream)
            : shift + number_bits <= 64
                ? calibrate_rows<std::uint64_t, false>(t, d_latency, n, slot_of, list, keys, classes,
                                                       shift, d_rows, stream)
                : calibrate_rows<std::uint64_t, true>(t, d_latency, n, slot_of, list, keys, classes,
                                                      shift, d_rows, stream);
        return st;
    }
}

}  // namespace hbfamd
