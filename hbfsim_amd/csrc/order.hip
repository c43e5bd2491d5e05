// order.hip -- issue-time order of a record stream (gfx950).
//
// The engine serves every resource in (issue time, stream position) order,
// the order in which the reference's MQSim adapter serves staged arrivals:
// sorted by (arrival, sequence) (src/mqsim_adapter/mqsim_online.cpp:
// 269-289).  Streams that are already issue-ordered (every workload
// generator's) are timed as they lie; the main pipeline notices any record
// whose issue time goes back while it summarises its tiles, and the engine
// then times the stream once more from a copy sorted here by (issue time,
// position), and scatters completion times and status bytes back to the
// records' stream positions.
//
// Issue times are spread over the span of the stream, so one partition by
// their top bits leaves buckets that a workgroup sorts in LDS: 8 bytes per
// record (issue time within the bucket, position) are written and read once.
//   k_issue_range     the least and greatest issue time;
//   k_bucket_count    records per bucket, by LDS histograms;
//   k_bucket_scan     bucket offsets;
//   k_bucket_scatter  keys into their buckets, in any order;
//   k_bucket_sort     each bucket by key, and its records gathered in order.
// 8.4M merged records: 32 + 27 + 15 + 60 + 125 us; rocPRIM's radix sort of
// 64-bit keys with positions (seven passes over 56 bits), its keys and the
// gather of the records took 810 us.  It
// still serves streams whose buckets overflow LDS (most records within a small
// part of the span), spans of more than 32 bits within a bucket, and more than
// kMaxBucketed records.
#include <hip/hip_runtime.h>

#include <cstring>  // rocPRIM's host code uses memset
#include <rocprim/device/device_radix_sort.hpp>

#include "engine.hpp"
#include "scratch.hpp"

#include <algorithm>
#include <cstdint>

namespace hbfamd {
namespace {

constexpr int kThreads = 256;
constexpr unsigned kMaxBlocks = 65536;

// Issue time of record i: 32-byte records hold it in word 2; packed records
// in bits 0-55 of their second word.
template <bool kPacked>
__device__ __forceinline__ std::uint64_t issue_of(const void* rec, std::size_t i)
{
    if (kPacked) {
        const std::uint64_t w = static_cast<const hbf_record16*>(rec)[i].issue_op;
        return w & ((1ull << 56) - 1);
    }
    return static_cast<const hbf_record32*>(rec)[i].issue_ps;
}

unsigned blocks_for(std::size_t n)
{
    const std::size_t b = (n + kThreads - 1) / kThreads;
    return static_cast<unsigned>(b < kMaxBlocks ? (b == 0 ? 1 : b) : kMaxBlocks);
}

// *flag = 1 when some record's issue time is below its predecessor's.
template <bool kPacked>
__global__ __launch_bounds__(kThreads) void k_order_check(const void* rec, std::size_t n,
                                                          std::uint32_t* flag)
{
    const std::size_t stride = static_cast<std::size_t>(gridDim.x) * kThreads;
    bool bad = false;
    for (std::size_t i = static_cast<std::size_t>(blockIdx.x) * kThreads + threadIdx.x + 1; i < n;
         i += stride) {
        bad = bad || issue_of<kPacked>(rec, i) < issue_of<kPacked>(rec, i - 1);
    }
    if (bad) {
        *flag = 1u;
    }
}

template <bool kPacked>
__global__ __launch_bounds__(kThreads) void k_issue_keys(const void* rec, std::size_t n,
                                                         std::uint64_t* keys, std::uint32_t* pos)
{
    const std::size_t stride = static_cast<std::size_t>(gridDim.x) * kThreads;
    for (std::size_t i = static_cast<std::size_t>(blockIdx.x) * kThreads + threadIdx.x; i < n;
         i += stride) {
        keys[i] = issue_of<kPacked>(rec, i);
        pos[i] = static_cast<std::uint32_t>(i);
    }
}

// out[j] = rec[pos[j]] (T: hbf_record32 or hbf_record16).
template <typename T>
__global__ __launch_bounds__(kThreads) void k_gather_records(const T* rec,
                                                             const std::uint32_t* pos,
                                                             std::size_t n, T* out)
{
    const std::size_t stride = static_cast<std::size_t>(gridDim.x) * kThreads;
    for (std::size_t j = static_cast<std::size_t>(blockIdx.x) * kThreads + threadIdx.x; j < n;
         j += stride) {
        out[j] = rec[pos[j]];
    }
}

// comp[pos[j]] = scomp[p], status[pos[j]] = sstatus[p] with p = place[j], or j
// when place is null (status optional).  After the bucket sort j is the order
// the records came into their buckets, in which an issuer's records lie next
// to each other in the stream: the stores then come in runs, and the loads
// stay within a bucket's 8 KiB.  Each XCD takes one contiguous eighth
// (workgroups go round the eight XCDs), so that stores to one line meet in one
// L2.  8.4M merged records: 60 us, against 99 storing in sorted order one
// record at a time.
__global__ __launch_bounds__(kThreads) void k_scatter(const std::uint32_t* pos,
                                                      const std::uint32_t* place, std::size_t n,
                                                      const std::uint64_t* scomp,
                                                      const std::uint8_t* sstatus,
                                                      std::uint64_t* comp, std::uint8_t* status)
{
    const unsigned per = gridDim.x / 8;  // workgroups per XCD (the grid is a multiple of 8)
    const std::size_t part = (n + 8ull * per - 1) / (8ull * per);
    const std::size_t b = (static_cast<std::size_t>(blockIdx.x % 8) * per + blockIdx.x / 8) * part;
    const std::size_t e = b + part < n ? b + part : n;
    // four records at once: their loads depend on each other in pairs
    for (std::size_t j = b + threadIdx.x; j < e; j += 4 * kThreads) {
        std::uint32_t i[4], p[4];
        std::uint64_t done[4];
        std::uint8_t st[4];
#pragma unroll
        for (int k = 0; k < 4; ++k) {
            const std::size_t at = j + static_cast<std::size_t>(k) * kThreads;
            const std::size_t from = at < e ? at : j;
            i[k] = pos[from];
            p[k] = place != nullptr ? place[from] : static_cast<std::uint32_t>(from);
        }
#pragma unroll
        for (int k = 0; k < 4; ++k) {
            done[k] = scomp[p[k]];
            st[k] = status != nullptr ? sstatus[p[k]] : std::uint8_t{0};
        }
#pragma unroll
        for (int k = 0; k < 4; ++k) {
            if (j + static_cast<std::size_t>(k) * kThreads < e) {
                comp[i[k]] = done[k];
                if (status != nullptr) {
                    status[i[k]] = st[k];
                }
            }
        }
    }
}

// ---- bucket sort ----------------------------------------------------------

constexpr std::size_t kBucketMean = 1024;    // records per bucket aimed at
constexpr std::size_t kMaxBuckets = 16384;   // their LDS histogram: 64 KiB
constexpr std::size_t kMaxBucketed = kMaxBuckets * 2048;
constexpr std::uint32_t kBucketCap = 4096;   // records of a bucket in LDS (32 KiB)
constexpr int kCapPer = kBucketCap / kThreads;
constexpr std::uint32_t kSubs = 1024;        // sub-buckets within a bucket
constexpr std::uint32_t kCrowd = 96;         // records of a sub-bucket told apart by comparing
constexpr std::size_t kChunk = 8192;         // records per workgroup of the partition
constexpr unsigned kRangeParts = 2048;       // workgroups of k_issue_range

struct Buckets {
    unsigned long long* range;   // least, greatest issue time
    std::uint32_t* count;        // [buckets] records, then the next free place
    std::uint32_t* first;        // [buckets + 1]
    std::uint32_t* overflow;     // set when a bucket or its keys do not fit
    std::uint32_t log2;          // buckets = 1 << log2
};

// A record's bucket is (issue - least) >> shift.
__device__ __forceinline__ std::uint32_t bucket_shift(std::uint64_t least, std::uint64_t most,
                                                      std::uint32_t log2)
{
    const std::uint64_t span = most - least;
    const std::uint32_t bits = span == 0 ? 0u : 64u - static_cast<std::uint32_t>(__clzll(span));
    return bits > log2 ? bits - log2 : 0u;
}

__device__ __forceinline__ std::uint32_t bucket_shift(const Buckets& k)
{
    return bucket_shift(k.range[0], k.range[1], k.log2);
}

__device__ __forceinline__ void block_range(std::uint64_t& lo, std::uint64_t& hi)
{
    __shared__ std::uint64_t w_lo[kThreads / 64], w_hi[kThreads / 64];
    for (int o = 32; o > 0; o >>= 1) {
        const std::uint64_t l = __shfl_xor(static_cast<unsigned long long>(lo), o);
        const std::uint64_t h = __shfl_xor(static_cast<unsigned long long>(hi), o);
        lo = l < lo ? l : lo;
        hi = h > hi ? h : hi;
    }
    if ((threadIdx.x & 63) == 0) {
        w_lo[threadIdx.x / 64] = lo;
        w_hi[threadIdx.x / 64] = hi;
    }
    __syncthreads();
    for (int w = 0; w < kThreads / 64; ++w) {
        lo = w_lo[w] < lo ? w_lo[w] : lo;
        hi = w_hi[w] > hi ? w_hi[w] : hi;
    }
}

// Per workgroup its least and greatest issue time (atomics on two words took
// 170 us with one pair per wave, 20 with one per workgroup).
template <bool kPacked>
__global__ __launch_bounds__(kThreads) void k_issue_range(const void* rec, std::size_t n,
                                                          ulonglong2* part)
{
    const std::size_t stride = static_cast<std::size_t>(gridDim.x) * kThreads;
    std::uint64_t lo = ~0ull, hi = 0;
    for (std::size_t i = static_cast<std::size_t>(blockIdx.x) * kThreads + threadIdx.x; i < n;
         i += 8 * stride) {
        std::uint64_t t[8];
#pragma unroll
        for (int k = 0; k < 8; ++k) {
            t[k] = issue_of<kPacked>(rec, i + k * stride < n ? i + k * stride : i);
        }
#pragma unroll
        for (int k = 0; k < 8; ++k) {
            lo = t[k] < lo ? t[k] : lo;
            hi = t[k] > hi ? t[k] : hi;
        }
    }
    block_range(lo, hi);
    if (threadIdx.x == 0) {
        part[blockIdx.x] = make_ulonglong2(lo, hi);
    }
}

template <bool kPacked>
__global__ __launch_bounds__(kThreads) void k_bucket_count(const void* rec, std::size_t n,
                                                           Buckets bk, const ulonglong2* part,
                                                           std::uint32_t parts)
{
    extern __shared__ std::uint32_t hist[];
    const std::uint32_t buckets = 1u << bk.log2;
    for (std::uint32_t b = threadIdx.x; b < buckets; b += kThreads) {
        hist[b] = 0;
    }
    std::uint64_t least = ~0ull, most = 0;
    for (std::uint32_t k = threadIdx.x; k < parts; k += kThreads) {
        const ulonglong2 p = part[k];
        least = p.x < least ? p.x : least;
        most = p.y > most ? p.y : most;
    }
    block_range(least, most);  // (also a barrier for the histogram)
    if (blockIdx.x == 0 && threadIdx.x == 0) {
        bk.range[0] = least;
        bk.range[1] = most;
    }
    const std::uint32_t shift = bucket_shift(least, most, bk.log2);
    const std::size_t begin = static_cast<std::size_t>(blockIdx.x) * kChunk;
    const std::size_t end = begin + kChunk < n ? begin + kChunk : n;
#pragma unroll 8
    for (std::size_t i = begin + threadIdx.x; i < end; i += kThreads) {
        atomicAdd(&hist[(issue_of<kPacked>(rec, i) - least) >> shift], 1u);
    }
    __syncthreads();
    for (std::uint32_t b = threadIdx.x; b < buckets; b += kThreads) {
        if (hist[b] != 0) {
            atomicAdd(&bk.count[b], hist[b]);
        }
    }
}

// One block: bucket offsets; count[] becomes the next free place of each.
__global__ __launch_bounds__(1024) void k_bucket_scan(Buckets bk, std::size_t n)
{
    __shared__ std::uint32_t w_sum[1024 / 64];
    const std::uint32_t buckets = 1u << bk.log2;
    const std::uint32_t per = (buckets + 1023) / 1024;
    const std::uint32_t b = threadIdx.x * per;
    const std::uint32_t e = b + per < buckets ? b + per : buckets;
    std::uint32_t own = 0, most = 0;
    for (std::uint32_t k = b; k < e; ++k) {
        const std::uint32_t c = bk.count[k];
        own += c;
        most = c > most ? c : most;
    }
    if (most > kBucketCap || (threadIdx.x == 0 && bucket_shift(bk) > 32)) {
        *bk.overflow = 1;
    }
    std::uint32_t incl = own;
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    for (int o = 1; o < 64; o <<= 1) {
        const std::uint32_t v = __shfl_up(incl, o);
        incl += lane >= o ? v : 0u;
    }
    if (lane == 63) {
        w_sum[wave] = incl;
    }
    __syncthreads();
    std::uint32_t at = incl - own;
    for (int w = 0; w < wave; ++w) {
        at += w_sum[w];
    }
    for (std::uint32_t k = b; k < e; ++k) {
        const std::uint32_t c = bk.count[k];
        bk.first[k] = at;
        bk.count[k] = at;
        at += c;
    }
    if (threadIdx.x == 0) {
        bk.first[buckets] = static_cast<std::uint32_t>(n);
    }
}

// key = issue time within the bucket << 32 | stream position.
template <bool kPacked>
__global__ __launch_bounds__(kThreads) void k_bucket_scatter(const void* rec, std::size_t n,
                                                             Buckets bk, std::uint64_t* key)
{
    extern __shared__ std::uint32_t hist[];
    const std::uint32_t buckets = 1u << bk.log2;
    for (std::uint32_t b = threadIdx.x; b < buckets; b += kThreads) {
        hist[b] = 0;
    }
    const std::uint32_t shift = bucket_shift(bk);
    const std::uint64_t least = bk.range[0];
    const std::size_t begin = static_cast<std::size_t>(blockIdx.x) * kChunk;
    std::uint64_t t[kChunk / kThreads];
#pragma unroll
    for (std::size_t k = 0; k < kChunk / kThreads; ++k) {
        const std::size_t i = begin + k * kThreads + threadIdx.x;
        t[k] = i < n ? issue_of<kPacked>(rec, i) - least : 0;
    }
    __syncthreads();
#pragma unroll
    for (std::size_t k = 0; k < kChunk / kThreads; ++k) {
        if (begin + k * kThreads + threadIdx.x < n) {
            atomicAdd(&hist[t[k] >> shift], 1u);
        }
    }
    __syncthreads();
    for (std::uint32_t b = threadIdx.x; b < buckets; b += kThreads) {
        if (hist[b] != 0) {
            hist[b] = atomicAdd(&bk.count[b], hist[b]);  // the chunk's place in it
        }
    }
    __syncthreads();
    const std::uint64_t low = (1ull << shift) - 1;
#pragma unroll
    for (std::size_t k = 0; k < kChunk / kThreads; ++k) {
        const std::size_t i = begin + k * kThreads + threadIdx.x;
        if (i < n) {
            key[atomicAdd(&hist[t[k] >> shift], 1u)] = ((t[k] & low) << 32) | i;
        }
    }
}

// Orders keys[0, 2^m), m >= 6, ascending: a bitonic network over the workgroup.
__device__ __forceinline__ void sort_keys(std::uint64_t* keys, std::uint32_t size)
{
    for (std::uint32_t run = 2; run <= size; run *= 2) {
        for (std::uint32_t gap = run / 2; gap != 0; gap /= 2) {
            for (std::uint32_t p = threadIdx.x; p < size / 2; p += kThreads) {
                const std::uint32_t i = 2 * p - (p & (gap - 1));
                const std::uint64_t a = keys[i], b = keys[i + gap];
                if ((a > b) == ((i & run) == 0)) {
                    keys[i] = b;
                    keys[i + gap] = a;
                }
            }
            __syncthreads();
        }
    }
}

// One workgroup per bucket.  Keys are unique, so a record's place is the
// number of smaller keys: all of the sub-buckets below its own, and those it
// finds by comparing within its own (one or two records unless many share an
// issue time).  A bucket with more than kCrowd records in one sub-bucket is
// sorted whole by a network instead, and a place found by bisection: comparing
// is quadratic in the records that share a time (4M packed records, whole run:
// 512 at a time 1,393 -> 838 us, 2,000 3,182 -> 878, about 4,000 7,231 ->
// 1,337; the radix sort alone 3,480, whatever the times).  The line lies
// above steps of one issue time: 4M lines in steps of 64 take 450 us by
// comparing and 523 by the network, records at random times of 64 each 781 and
// 842; at 128 each 909 and 792.
// pos and place (stream position, sorted position) are written in
// the order the records came into the bucket, for k_scatter.
template <typename T>
__global__ __launch_bounds__(kThreads) void k_bucket_sort(Buckets bk, const std::uint64_t* key,
                                                          const T* rec, std::uint32_t* pos,
                                                          std::uint32_t* place, T* out)
{
    __shared__ std::uint64_t keys[kBucketCap];
    __shared__ std::uint32_t sub[kSubs + 1];
    __shared__ std::uint32_t w_sum[kThreads / 64];
    const std::uint32_t s = bk.first[blockIdx.x];
    const std::uint32_t count = bk.first[blockIdx.x + 1] - s;
    if (count == 0 || count > kBucketCap) {
        return;
    }
    const std::uint32_t shift = bucket_shift(bk);
    if (shift > 32) {
        return;  // the keys do not hold it (k_bucket_scan says so)
    }
    const std::uint32_t down = 32 + (shift > 10 ? shift - 10 : 0);  // key -> sub-bucket
    for (std::uint32_t k = threadIdx.x; k <= kSubs; k += kThreads) {
        sub[k] = 0;
    }
    std::uint64_t mine[kCapPer];
    std::uint32_t rank[kCapPer];
#pragma unroll
    for (int k = 0; k < kCapPer; ++k) {
        const std::uint32_t j = k * kThreads + threadIdx.x;
        mine[k] = j < count ? key[s + j] : ~0ull;
    }
    __syncthreads();
#pragma unroll
    for (int k = 0; k < kCapPer; ++k) {
        if (k * kThreads + threadIdx.x < count) {
            rank[k] = atomicAdd(&sub[mine[k] >> down], 1u);
        }
    }
    __syncthreads();
    // exclusive scan of the sub-bucket counts, four per thread
    std::uint32_t c[4], own = 0;
    bool crowd = false;
#pragma unroll
    for (int k = 0; k < 4; ++k) {
        c[k] = sub[threadIdx.x * 4 + k];
        own += c[k];
        crowd = crowd || c[k] > kCrowd;
    }
    std::uint32_t incl = own;
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    for (int o = 1; o < 64; o <<= 1) {
        const std::uint32_t v = __shfl_up(incl, o);
        incl += lane >= o ? v : 0u;
    }
    if (lane == 63) {
        w_sum[wave] = incl;
    }
    __syncthreads();
    std::uint32_t at = incl - own;
    for (int w = 0; w < wave; ++w) {
        at += w_sum[w];
    }
#pragma unroll
    for (int k = 0; k < 4; ++k) {
        sub[threadIdx.x * 4 + k] = at;
        at += c[k];
    }
    if (threadIdx.x == kThreads - 1) {
        sub[kSubs] = count;
    }
    __syncthreads();
#pragma unroll
    for (int k = 0; k < kCapPer; ++k) {
        if (k * kThreads + threadIdx.x < count) {
            keys[sub[mine[k] >> down] + rank[k]] = mine[k];
        }
    }
    const bool crowded = __syncthreads_or(crowd ? 1 : 0) != 0;
    if (crowded) {
        std::uint32_t size = 64;
        while (size < count) {
            size *= 2;
        }
        for (std::uint32_t j = count + threadIdx.x; j < size; j += kThreads) {
            keys[j] = ~0ull;
        }
        __syncthreads();
        sort_keys(keys, size);
    }
    std::uint32_t to[kCapPer];  // sorted place within the bucket
#pragma unroll
    for (int k = 0; k < kCapPer; ++k) {
        const std::uint32_t j = k * kThreads + threadIdx.x;
        if (j < count) {
            std::uint32_t lo = sub[mine[k] >> down], hi = sub[(mine[k] >> down) + 1];
            to[k] = lo;
            if (crowded) {
                while (lo < hi) {  // the key's place among the sorted ones
                    const std::uint32_t m = (lo + hi) / 2;
                    lo = keys[m] < mine[k] ? m + 1 : lo;
                    hi = keys[m] < mine[k] ? hi : m;
                }
                to[k] = lo;
            } else {
                for (std::uint32_t m = lo; m < hi; ++m) {
                    to[k] += keys[m] < mine[k] ? 1u : 0u;
                }
            }
            pos[s + j] = static_cast<std::uint32_t>(mine[k]);
            place[s + j] = s + to[k];
        }
    }
    __syncthreads();
    std::uint32_t* from = reinterpret_cast<std::uint32_t*>(keys);
#pragma unroll
    for (int k = 0; k < kCapPer; ++k) {
        if (k * kThreads + threadIdx.x < count) {
            from[to[k]] = static_cast<std::uint32_t>(mine[k]);
        }
    }
    __syncthreads();
    for (std::uint32_t j = threadIdx.x; j < count; j += 4 * kThreads) {
        T r[4];
#pragma unroll
        for (int k = 0; k < 4; ++k) {
            const std::uint32_t at = j + k * kThreads;
            r[k] = rec[from[at < count ? at : j]];
        }
#pragma unroll
        for (int k = 0; k < 4; ++k) {
            if (j + k * kThreads < count) {
                out[s + j + k * kThreads] = r[k];
            }
        }
    }
}

// Lets a histogram kernel have `bytes` of dynamic LDS: beyond 64 KB, its static arrays
// included, it has to be allowed the size first (16,384 buckets take 64 KB by themselves).
template <typename F>
hipError_t allow_hist(F* kernel, std::size_t bytes)
{
    if (bytes <= (std::size_t{32} << 10)) {
        return hipSuccess;
    }
    return hipFuncSetAttribute(reinterpret_cast<const void*>(kernel),
                               hipFuncAttributeMaxDynamicSharedMemorySize,
                               static_cast<int>(bytes));
}

// Each kernel takes what the one before it wrote for granted (bucket numbers and places are
// indices), so nothing is launched after one that was refused.
template <typename T, bool kPacked>
hipError_t launch_buckets(const void* rec, std::size_t n, const Buckets& bk, ulonglong2* part,
                          std::uint64_t* key, std::uint32_t* pos, std::uint32_t* place, T* sorted,
                          hipStream_t stream)
{
    const std::size_t lds = (std::size_t{1} << bk.log2) * 4;
    const unsigned chunks = static_cast<unsigned>((n + kChunk - 1) / kChunk);
    const unsigned parts = std::min(blocks_for((n + 7) / 8), kRangeParts);
    hipError_t err = allow_hist(k_bucket_count<kPacked>, lds);
    if (err == hipSuccess) err = allow_hist(k_bucket_scatter<kPacked>, lds);
    if (err == hipSuccess) {
        hipLaunchKernelGGL(k_issue_range<kPacked>, dim3(parts), dim3(kThreads), 0, stream, rec, n,
                           part);
        err = hipGetLastError();
    }
    if (err == hipSuccess) {
        hipLaunchKernelGGL(k_bucket_count<kPacked>, dim3(chunks), dim3(kThreads), lds, stream, rec,
                           n, bk, part, parts);
        err = hipGetLastError();
    }
    if (err == hipSuccess) {
        hipLaunchKernelGGL(k_bucket_scan, dim3(1), dim3(1024), 0, stream, bk, n);
        err = hipGetLastError();
    }
    if (err == hipSuccess) {
        hipLaunchKernelGGL(k_bucket_scatter<kPacked>, dim3(chunks), dim3(kThreads), lds, stream,
                           rec, n, bk, key);
        err = hipGetLastError();
    }
    if (err == hipSuccess) {
        hipLaunchKernelGGL(k_bucket_sort<T>, dim3(1u << bk.log2), dim3(kThreads), 0, stream, bk,
                           key, static_cast<const T*>(rec), pos, place, sorted);
        err = hipGetLastError();
    }
    return err;
}

// The stable order by radix sort: pos receives the positions.
int radix_order(const void* rec, bool packed, std::size_t n, std::uint32_t* pos,
                hipStream_t stream)
{
    const unsigned end_bit = packed ? 56u : 64u;
    std::size_t temp_bytes = 0;
    hipError_t err = rocprim::radix_sort_pairs(nullptr, temp_bytes,
                                               static_cast<std::uint64_t*>(nullptr),
                                               static_cast<std::uint64_t*>(nullptr),
                                               static_cast<std::uint32_t*>(nullptr),
                                               static_cast<std::uint32_t*>(nullptr), n, 0, end_bit,
                                               stream);
    if (err != hipSuccess) {
        return HBFSIM_CUDA_ERROR;
    }
    ScratchPlan plan;
    const std::size_t o_key_a = plan.add<std::uint64_t>(n);
    const std::size_t o_key_b = plan.add<std::uint64_t>(n);
    const std::size_t o_pos = plan.add<std::uint32_t>(n);
    const std::size_t o_temp = plan.add<unsigned char>(temp_bytes);
    ScratchLease lease(plan.bytes, stream);
    if (!lease.ok()) {
        return HBFSIM_CUDA_ERROR;
    }
    auto* key_a = lease.at<std::uint64_t>(o_key_a);
    auto* pos_a = lease.at<std::uint32_t>(o_pos);
    if (packed) {
        hipLaunchKernelGGL(k_issue_keys<true>, dim3(blocks_for(n)), dim3(kThreads), 0, stream, rec,
                           n, key_a, pos_a);
    } else {
        hipLaunchKernelGGL(k_issue_keys<false>, dim3(blocks_for(n)), dim3(kThreads), 0, stream,
                           rec, n, key_a, pos_a);
    }
    err = hipGetLastError();
    if (err == hipSuccess) {
        err = rocprim::radix_sort_pairs(lease.at<unsigned char>(o_temp), temp_bytes, key_a,
                                        lease.at<std::uint64_t>(o_key_b), pos_a, pos, n, 0,
                                        end_bit, stream);
    }
    // (the lease waits for the stream)
    return err == hipSuccess ? HBFSIM_OK : HBFSIM_CUDA_ERROR;
}

// Results of the sorted copy back to the records' stream positions.
hipError_t scatter_back(const std::uint32_t* pos, const std::uint32_t* place, std::size_t n,
                        const std::uint64_t* scomp, const std::uint8_t* sstatus,
                        std::uint64_t* comp, std::uint8_t* status, hipStream_t stream)
{
    const unsigned eighths = (std::min(blocks_for(n), 8192u) + 7) / 8;  // whole rounds of XCDs
    hipLaunchKernelGGL(k_scatter, dim3(8 * eighths), dim3(kThreads), 0, stream, pos, place, n,
                       scomp, sstatus, comp, status);
    const hipError_t err = hipGetLastError();
    return err == hipSuccess ? hipStreamSynchronize(stream) : err;
}

// The run by the bucket sort.  `done` stays false, and nothing has changed, where it does not
// apply: no memory for all its arrays at once, a launch refused, or buckets that do not fit.
int run_bucketed(const void* d_rec, bool packed, std::size_t n, std::uint64_t* d_comp,
                 std::uint8_t* d_status, hipStream_t stream, const sorted_runner& run, bool& done)
{
    std::uint32_t log2 = 4;
    while ((kBucketMean << log2) < n && (std::size_t{1} << log2) < kMaxBuckets) {
        ++log2;
    }
    const std::size_t buckets = std::size_t{1} << log2;
    const std::size_t rec_bytes = packed ? sizeof(hbf_record16) : sizeof(hbf_record32);
    ScratchPlan plan;
    const std::size_t o_words = plan.add<unsigned long long>(3);
    const std::size_t o_count = plan.add<std::uint32_t>(buckets);
    const std::size_t o_first = plan.add<std::uint32_t>(buckets + 1);
    const std::size_t o_part = plan.add<ulonglong2>(kRangeParts);
    const std::size_t o_pos = plan.add<std::uint32_t>(n);
    const std::size_t o_place = plan.add<std::uint32_t>(n);
    const std::size_t o_key = plan.add<std::uint64_t>(n);  // keys, then completions
    const std::size_t o_rec = plan.add<unsigned char>(n * rec_bytes);
    const std::size_t o_status = plan.add<std::uint8_t>(d_status != nullptr ? n : 0);
    ScratchLease lease(plan.bytes, stream);
    if (!lease.ok()) {
        return HBFSIM_OK;
    }
    auto* words = lease.at<unsigned long long>(o_words);
    auto* pos = lease.at<std::uint32_t>(o_pos);
    auto* place = lease.at<std::uint32_t>(o_place);
    auto* key = lease.at<std::uint64_t>(o_key);
    void* sorted = lease.at<unsigned char>(o_rec);
    auto* sstatus = d_status != nullptr ? lease.at<std::uint8_t>(o_status) : nullptr;
    const Buckets bk{words, lease.at<std::uint32_t>(o_count), lease.at<std::uint32_t>(o_first),
                     reinterpret_cast<std::uint32_t*>(words + 2), log2};
    auto* part = lease.at<ulonglong2>(o_part);
    hipError_t err = hipMemsetAsync(words, 0, o_first - o_words, stream);
    if (err != hipSuccess) {
        return HBFSIM_CUDA_ERROR;
    }
    err = packed ? launch_buckets<hbf_record16, true>(d_rec, n, bk, part, key, pos, place,
                                                      static_cast<hbf_record16*>(sorted), stream)
                 : launch_buckets<hbf_record32, false>(d_rec, n, bk, part, key, pos, place,
                                                       static_cast<hbf_record32*>(sorted), stream);
    if (err != hipSuccess) {
        (void)hipGetLastError();
        return HBFSIM_OK;
    }
    std::uint32_t overflow = 0;
    err = hipMemcpyAsync(&overflow, bk.overflow, 4, hipMemcpyDeviceToHost, stream);
    if (err == hipSuccess) err = hipStreamSynchronize(stream);
    if (err != hipSuccess) {
        return HBFSIM_CUDA_ERROR;
    }
    if (overflow != 0) {
        lease.synced(err);
        return HBFSIM_OK;
    }
    done = true;
    const int st = run(sorted, key, sstatus);
    if (st != HBFSIM_OK) {
        return st;
    }
    err = scatter_back(pos, place, n, key, sstatus, d_comp, d_status, stream);
    lease.synced(err);
    return err == hipSuccess ? HBFSIM_OK : HBFSIM_CUDA_ERROR;
}

// The run by the radix sort.  Its keys (24 bytes a record, and the library's own scratch) are
// given back before the sorted copy and its results are laid out, so that a run needs the larger
// of the two and not their sum.
int run_radix(const void* d_rec, bool packed, std::size_t n, std::uint64_t* d_comp,
              std::uint8_t* d_status, hipStream_t stream, const sorted_runner& run)
{
    ScratchLease order(n * sizeof(std::uint32_t), stream);
    if (!order.ok()) {
        return HBFSIM_CUDA_ERROR;
    }
    auto* pos = order.at<std::uint32_t>(0);
    int st = radix_order(d_rec, packed, n, pos, stream);
    if (st != HBFSIM_OK) {
        return st;
    }
    ScratchPlan plan;
    const std::size_t rec_bytes = packed ? sizeof(hbf_record16) : sizeof(hbf_record32);
    const std::size_t o_comp = plan.add<std::uint64_t>(n);
    const std::size_t o_rec = plan.add<unsigned char>(n * rec_bytes);
    const std::size_t o_status = plan.add<std::uint8_t>(d_status != nullptr ? n : 0);
    ScratchLease lease(plan.bytes, stream);
    if (!lease.ok()) {
        return HBFSIM_CUDA_ERROR;
    }
    auto* scomp = lease.at<std::uint64_t>(o_comp);
    void* sorted = lease.at<unsigned char>(o_rec);
    auto* sstatus = d_status != nullptr ? lease.at<std::uint8_t>(o_status) : nullptr;
    if (packed) {
        hipLaunchKernelGGL(k_gather_records<hbf_record16>, dim3(blocks_for(n)), dim3(kThreads), 0,
                           stream, static_cast<const hbf_record16*>(d_rec), pos, n,
                           static_cast<hbf_record16*>(sorted));
    } else {
        hipLaunchKernelGGL(k_gather_records<hbf_record32>, dim3(blocks_for(n)), dim3(kThreads), 0,
                           stream, static_cast<const hbf_record32*>(d_rec), pos, n,
                           static_cast<hbf_record32*>(sorted));
    }
    if (hipGetLastError() != hipSuccess) {
        return HBFSIM_CUDA_ERROR;
    }
    st = run(sorted, scomp, sstatus);
    if (st != HBFSIM_OK) {
        return st;
    }
    const hipError_t err =
        scatter_back(pos, nullptr, n, scomp, sstatus, d_comp, d_status, stream);  // pos is sorted
    lease.synced(err);
    order.synced(err);
    return err == hipSuccess ? HBFSIM_OK : HBFSIM_CUDA_ERROR;
}

}  // namespace

int order_check(const void* d_rec, bool packed, std::size_t n, std::uint32_t* d_flag,
                void* stream_ptr)
{
    if (n < 2) {
        return HBFSIM_OK;
    }
    hipStream_t stream = static_cast<hipStream_t>(stream_ptr);
    if (packed) {
        hipLaunchKernelGGL(k_order_check<true>, dim3(blocks_for(n)), dim3(kThreads), 0, stream,
                           d_rec, n, d_flag);
    } else {
        hipLaunchKernelGGL(k_order_check<false>, dim3(blocks_for(n)), dim3(kThreads), 0, stream,
                           d_rec, n, d_flag);
    }
    return hipGetLastError() == hipSuccess ? HBFSIM_OK : HBFSIM_CUDA_ERROR;
}

int run_in_issue_order(const void* d_rec, bool packed, std::size_t n, std::uint64_t* d_comp,
                       std::uint8_t* d_status, void* stream_ptr, const sorted_runner& run)
{
    if (n >= (1ull << 32)) {
        return HBFSIM_UNSUPPORTED;  // positions travel as 32-bit payload
    }
    hipStream_t stream = static_cast<hipStream_t>(stream_ptr);
    if (n <= kMaxBucketed) {
        bool done = false;
        const int st = run_bucketed(d_rec, packed, n, d_comp, d_status, stream, run, done);
        if (done || st != HBFSIM_OK) {
            return st;
        }
    }
    return run_radix(d_rec, packed, n, d_comp, d_status, stream, run);
}

}  // namespace hbfamd
