// engine.hip -- HBF per-access timing engine for gfx950 (MI355X).
//
// Replaces the reference's per-access device resolver and its single global
// busy-until tail (src/cuda_runtime/device/hbf_device.cu:765-959, 963-1344)
// with a batch pipeline over access records resident in HBM:
//
//   k_summary  one wave per tile of records: classify against the range
//              table (binary search, fences staged in LDS), stripe the media
//              page onto channel/way/die/plane, and fold every record into a
//              per-resource (max,+) summary of the tile.  Planes also carry
//              their page-register tag; a tile's first record on a plane has
//              its page-buffer hit resolved later, from the carry.
//   k_carry_*  a three-level scan over the tile summaries gives the exact
//              busy-until / tag state at the start of every tile (and the
//              final state, kept for the next run); one launch for runs of
//              at most 4,096 tiles, three for larger ones.
//   k_apply    re-reads each tile, replays it from its carry-in state and
//              writes completion times, status bytes and accounting.
//
// Per resource, busy' = max(busy, issue) + service.  The map
// b -> max(b + A, B) composes associatively,
//   (A1, B1) then (A2, B2) = (A1 + A2, max(B1 + A2, B2)),
// which is what lets a wave fold a group of same-resource records in
// log2(64) shuffle rounds and lets tiles be summarised independently.
//
// Within a step of 64 records the wave groups lanes by resource with 64-bit
// ballots (one per key bit), orders each group by lane, and scans it by
// pointer jumping.  No atomics touch timing state, so results are
// deterministic and bit-identical to the sequential CPU model.
#include <hip/hip_runtime.h>

#include "engine.hpp"
#include "scratch.hpp"
#include "thermal.hpp"

#include <algorithm>
#include <cstring>
#include <mutex>
#include <optional>
#include <type_traits>
#include <vector>

namespace hbfamd {
namespace {

constexpr int kWave = 64;
// Top level of the two-level range lookup (find_range), staged in LDS by
// every per-record kernel.  256 fences (2 KiB) rather than 512 let the
// summary pass hold 8 waves per CU instead of 7 at 512 planes.
constexpr std::uint32_t kMaxFences = 256;
// Planes: the summary pass keeps 33 B of state per plane in LDS, which at
// 4,096 planes (135 KB) still fits gfx950's 160 KB per workgroup.
constexpr std::uint32_t kMaxPlanes = 4096;
constexpr std::uint32_t kMaxChannels = 256;
constexpr std::uint32_t kClsModeled = 0;
constexpr std::uint32_t kClsBypass = 1;
constexpr std::uint32_t kClsUnsupported = 2;
constexpr std::uint32_t kClsInvalid = 3;  // lane beyond the tile
constexpr std::uint32_t kClsFollower = 5;  // shares an earlier record's request
constexpr std::uint8_t kStGrouped = 32;

struct alignas(16) PlaneSum {
    std::uint64_t fpage1;  // page + 1 of the tile's first record (0: none)
    std::uint64_t fissue;  // its issue time
    std::uint64_t rA, rB;  // (max,+) map of the records after the first
    std::uint64_t lpage1;  // page + 1 of the tile's last record
    std::uint32_t fcls;    // first record: bit 0 op, bit 1 programs
    std::uint32_t pad;
};
struct alignas(16) ChanSum {
    std::uint64_t A, B;
};
struct alignas(16) PlaneCarry {
    std::uint64_t busy, tag1;
};

struct DevReport {
    unsigned long long v[14];
};
static_assert(offsetof(hbfsim_amd_report, grouped) == sizeof(DevReport), "report layout");
enum {
    R_RECORDS, R_MODELED, R_BYPASS, R_UNSUPPORTED, R_READS, R_WRITES, R_HITS,
    R_PROGRAMS, R_HYBRID, R_MAKESPAN, R_LAT_LO, R_LAT_HI, R_LAT_MAX, R_SERVICE
};

// A split step's second run (its media page + 1, the lane it starts at and
// its range id), beside the step's descriptor, whose byte count then carries
// kSplitFlag.
struct alignas(16) SplitDesc {
    std::uint32_t page1b;
    std::uint32_t k;
    std::uint32_t ridb;
    std::uint32_t pad;
};
constexpr std::uint32_t kSplitFlag = 0x80000000u;
constexpr std::uint8_t kTilePlain = 2;

// Kernel arguments, passed by value.
struct KArgs {
    // ranges (structure of arrays, sorted by base)
    const std::uint64_t* r_base;
    const std::uint64_t* r_length;
    const std::uint64_t* r_file_offset;
    const std::uint32_t* r_meta;  // mode | permissions << 8
    const std::uint32_t* r_id;
    std::uint32_t r_count, r_stride, r_nfence;
    // the per-record passes hold the whole range table in LDS (RangeView);
    // set where it fits the table's packed form and costs the passes no waves
    std::uint32_t r_lds;
    std::uint32_t r_top;  // the largest power of two up to r_count (r_lds only)
    // geometry
    std::uint32_t Rp, Rc;           // planes, channels (resource counts)
    std::uint32_t W, D, P;
    std::uint32_t pbits, cbits;     // key widths for grouping
    std::uint32_t pow2;             // all axis sizes powers of two
    std::uint32_t axis_size[4];     // C W D P
    std::uint64_t axis_div[4];      // product of faster axis sizes
    std::uint32_t axis_shift[4];    // log2 of axis_div (pow2 only)
    std::uint32_t flat;             // one channel, one plane
    std::uint32_t page_shift;
    std::uint32_t slots;
    std::uint32_t contention;
    std::uint32_t transfer_page;
    std::uint32_t every_write;
    std::uint32_t hybrid;
    std::uint32_t hybrid_warmup;
    std::uint64_t hybrid_threshold;
    std::uint64_t read_ps, program_ps;
    std::uint64_t xfer_num, xfer_den, xfer_q;
    std::uint64_t xfer_pow2[33];    // transfer ps for 2^k bytes
    std::uint64_t media_pages;      // device capacity in pages
    std::uint32_t tile;
    std::uint32_t ext_hits;         // page-buffer hits given per record (K = 2)
    // the per-record passes match lane keys through per-wave LDS tables (one
    // 64-bit lane mask per plane and per channel) instead of one ballot per
    // key bit; set where the tables cost the passes no occupancy
    std::uint32_t match_lds;
    // the per-record passes' general steps look a media page's plane and
    // channel up in a per-wave LDS table of Rp entries (power-of-two axes:
    // both depend on the page modulo Rp only) instead of striping it; set
    // where the table costs the passes no occupancy
    std::uint32_t stripe_lds;
    // warp grouping: per record, how many records back its group's request
    // was made (0: its own request); null when the run does not group
    const std::uint8_t* lead;
    // hybrid runs: the range id of each linear step beside its descriptor
    // (the sampler's key needs it); null otherwise
    std::uint32_t* desc_rid;
    // split steps' second runs beside their descriptors (with the descriptors)
    SplitDesc* desc_split;
    // set to 1 by the summary pass when some record's issue time is below its
    // predecessor's; the carry chain then leaves the engine state untouched
    // and the engine times the stream again from a sorted copy (null: the
    // stream is known to be in issue order)
    std::uint32_t* disorder;
    // per tile, written by the summary pass: 1 when the
    // tile holds a split step (the apply pass then takes its split-capable
    // body), kTilePlain when the scattered-record passes take it, else 0; null
    // for streams with refresh records
    std::uint8_t* tile_split;
    std::uint32_t mixed;  // the scattered-record passes ran before: skip their tiles
    // start times of the summary pass, the carry chain and the apply pass
    // (stamp_start)
    std::uint64_t* stamp;
};

// The first workgroup of a run's kernels notes when it starts, by the GPU's
// constant-rate clock.  (Event records between the kernels gave the same
// intervals but kept 5-6 us of idle time at each: 17 us of a short run.)
__device__ __forceinline__ void stamp_start(const KArgs& a, int which)
{
    if (blockIdx.x == 0 && threadIdx.x == 0) {
        a.stamp[which] = static_cast<std::uint64_t>(wall_clock64());
    }
}


// Record operations: 0 read, 1 write, and 2 refresh of media page `addr`
// (read out and programmed back), valid only with kMediaFlag.
constexpr std::uint32_t kOpRefresh = 2;
constexpr std::uint32_t kMediaFlag = 0x100;

struct Dec {
    std::uint32_t cls;
    std::uint32_t bits;    // bit 0 write or refresh, bit 1 programs, bit 2 refresh
    std::uint32_t plane, chan;
    std::uint32_t range_id;
    std::uint64_t page1;   // media page + 1
    std::uint64_t issue;
    std::uint64_t xfer;
    std::uint64_t xbytes;  // bytes the channel moves
};

__device__ __forceinline__ std::uint64_t shfl64(std::uint64_t v, int src)
{
    const int lo = __shfl(static_cast<int>(static_cast<std::uint32_t>(v)), src);
    const int hi = __shfl(static_cast<int>(static_cast<std::uint32_t>(v >> 32)), src);
    return (static_cast<std::uint64_t>(static_cast<std::uint32_t>(hi)) << 32) |
           static_cast<std::uint32_t>(lo);
}

__device__ __forceinline__ std::uint64_t umax64(std::uint64_t a, std::uint64_t b)
{
    return a > b ? a : b;
}

// Completion times are written once and not read again by the pass, so they
// are stored non-temporally: kept out of the caches, they leave the next
// step's records there (config 2: the apply pass 3% faster and the next
// summary pass 2-5%).
__device__ __forceinline__ void put_done(std::uint64_t* p, std::uint64_t v)
{
    __builtin_nontemporal_store(v, p);
}

__device__ __forceinline__ std::uint64_t lanemask_lt(int lane)
{
    return lane == 0 ? 0ull : (~0ull >> (64 - lane));
}

// SplitMix64 finaliser, the reference's fast_hash (hbf_device.cuh:729-736).
__device__ __forceinline__ std::uint64_t mix64(std::uint64_t v)
{
    v += 0x9e3779b97f4a7c15ull;
    v = (v ^ (v >> 30)) * 0xbf58476d1ce4e5b9ull;
    v = (v ^ (v >> 27)) * 0x94d049bb133111ebull;
    return v ^ (v >> 31);
}

// Lanes whose key equals this lane's key, among `active`: one ballot per key
// bit.  Every lane of the wave must call it (uniform control flow).
__device__ __forceinline__ std::uint64_t match_key(std::uint32_t key, std::uint32_t bits,
                                                   std::uint64_t active)
{
    std::uint64_t m = active;
    for (std::uint32_t b = 0; b < bits; ++b) {
        const bool bit = (key >> b) & 1u;
        const std::uint64_t ones = __ballot(bit);
        m &= bit ? ones : ~ones;
    }
    return m;
}

// Inclusive scan of (A, B) maps over each lane group, in lane order, by
// pointer jumping along `pred` (the previous lane of the same group, or -1).
__device__ __forceinline__ void group_scan(std::uint64_t& A, std::uint64_t& B, int pred,
                                           int lane)
{
    int ptr = pred;
    for (int s = 0; s < 6; ++s) {
        if (__ballot(ptr >= 0) == 0) {
            break;
        }
        const int src = ptr < 0 ? lane : ptr;
        const std::uint64_t pA = shfl64(A, src);
        const std::uint64_t pB = shfl64(B, src);
        const int pp = __shfl(ptr, src);
        if (ptr >= 0) {
            B = umax64(pB + A, B);
            A = pA + A;
            ptr = pp;
        }
    }
}

// Two independent group scans of 32-bit (A, B) maps, interleaved: pointer
// jumping along pred1 and pred2 (previous lane of the same group, or -1).
__device__ __forceinline__ void group_scan32x2(std::uint32_t& A1, std::uint32_t& B1, int pred1,
                                               std::uint32_t& A2, std::uint32_t& B2, int pred2,
                                               int lane)
{
    int p1 = pred1, p2 = pred2;
    for (int s = 0; s < 6; ++s) {
        if (__ballot(p1 >= 0 || p2 >= 0) == 0) {
            break;
        }
        const int s1 = p1 < 0 ? lane : p1;
        const int s2 = p2 < 0 ? lane : p2;
        const std::uint32_t a1 = static_cast<std::uint32_t>(__shfl(static_cast<int>(A1), s1));
        const std::uint32_t b1 = static_cast<std::uint32_t>(__shfl(static_cast<int>(B1), s1));
        const int q1 = __shfl(p1, s1);
        const std::uint32_t a2 = static_cast<std::uint32_t>(__shfl(static_cast<int>(A2), s2));
        const std::uint32_t b2 = static_cast<std::uint32_t>(__shfl(static_cast<int>(B2), s2));
        const int q2 = __shfl(p2, s2);
        if (p1 >= 0) {
            const std::uint32_t nb = b1 + A1;
            B1 = nb > B1 ? nb : B1;
            A1 = a1 + A1;
            p1 = q1;
        }
        if (p2 >= 0) {
            const std::uint32_t nb = b2 + A2;
            B2 = nb > B2 ? nb : B2;
            A2 = a2 + A2;
            p2 = q2;
        }
    }
}

// Whole-wave inclusive scan of (A, B) maps in lane order, for steps where
// every active lane belongs to one group (inactive lanes hold the identity
// (0, 0)).  DPP row shifts build 16-lane scans, then row broadcasts join the
// rows; no LDS traffic.  Controls are the GFX9 encodings gfx950 keeps:
// row_shr:n = 0x110 + n, row_bcast:15 = 0x142, row_bcast:31 = 0x143.
template <int Ctrl, int RowMask>
__device__ __forceinline__ std::uint64_t dpp64(std::uint64_t v)
{
    const int lo = __builtin_amdgcn_update_dpp(
        0, static_cast<int>(static_cast<std::uint32_t>(v)), Ctrl, RowMask, 0xF, false);
    const int hi = __builtin_amdgcn_update_dpp(
        0, static_cast<int>(static_cast<std::uint32_t>(v >> 32)), Ctrl, RowMask, 0xF, false);
    return (static_cast<std::uint64_t>(static_cast<std::uint32_t>(hi)) << 32) |
           static_cast<std::uint32_t>(lo);
}

template <int Ctrl, int RowMask>
__device__ __forceinline__ void dpp_scan_step(std::uint64_t& A, std::uint64_t& B)
{
    const std::uint64_t pA = dpp64<Ctrl, RowMask>(A);
    const std::uint64_t pB = dpp64<Ctrl, RowMask>(B);
    B = umax64(pB + A, B);
    A = pA + A;
}

__device__ __forceinline__ void wave_scan(std::uint64_t& A, std::uint64_t& B)
{
    dpp_scan_step<0x111, 0xF>(A, B);
    dpp_scan_step<0x112, 0xF>(A, B);
    dpp_scan_step<0x114, 0xF>(A, B);
    dpp_scan_step<0x118, 0xF>(A, B);
    dpp_scan_step<0x142, 0xA>(A, B);
    dpp_scan_step<0x143, 0xC>(A, B);
}

template <int Ctrl, int RowMask>
__device__ __forceinline__ void dpp_scan_step32(std::uint32_t& A, std::uint32_t& B)
{
    const std::uint32_t pA = static_cast<std::uint32_t>(
        __builtin_amdgcn_update_dpp(0, static_cast<int>(A), Ctrl, RowMask, 0xF, false));
    const std::uint32_t pB = static_cast<std::uint32_t>(
        __builtin_amdgcn_update_dpp(0, static_cast<int>(B), Ctrl, RowMask, 0xF, false));
    const std::uint32_t nb = pB + A;
    B = nb > B ? nb : B;
    A = pA + A;
}

// Two independent whole-wave scans in 32 bits, interleaved for ILP.
__device__ __forceinline__ void wave_scan32x2(std::uint32_t& A1, std::uint32_t& B1,
                                              std::uint32_t& A2, std::uint32_t& B2)
{
    dpp_scan_step32<0x111, 0xF>(A1, B1);
    dpp_scan_step32<0x111, 0xF>(A2, B2);
    dpp_scan_step32<0x112, 0xF>(A1, B1);
    dpp_scan_step32<0x112, 0xF>(A2, B2);
    dpp_scan_step32<0x114, 0xF>(A1, B1);
    dpp_scan_step32<0x114, 0xF>(A2, B2);
    dpp_scan_step32<0x118, 0xF>(A1, B1);
    dpp_scan_step32<0x118, 0xF>(A2, B2);
    dpp_scan_step32<0x142, 0xA>(A1, B1);
    dpp_scan_step32<0x142, 0xA>(A2, B2);
    dpp_scan_step32<0x143, 0xC>(A1, B1);
    dpp_scan_step32<0x143, 0xC>(A2, B2);
}

// Inclusive prefix maximum across the wave (DPP; lanes without a source take
// 0, the identity for unsigned max).
template <int Ctrl, int RowMask>
__device__ __forceinline__ std::uint32_t dpp32(std::uint32_t v)
{
    return static_cast<std::uint32_t>(
        __builtin_amdgcn_update_dpp(0, static_cast<int>(v), Ctrl, RowMask, 0xF, false));
}

__device__ __forceinline__ std::uint32_t wave_prefix_max32(std::uint32_t v)
{
    std::uint32_t t;
    t = dpp32<0x111, 0xF>(v); v = v > t ? v : t;
    t = dpp32<0x112, 0xF>(v); v = v > t ? v : t;
    t = dpp32<0x114, 0xF>(v); v = v > t ? v : t;
    t = dpp32<0x118, 0xF>(v); v = v > t ? v : t;
    t = dpp32<0x142, 0xA>(v); v = v > t ? v : t;
    t = dpp32<0x143, 0xC>(v); v = v > t ? v : t;
    return v;
}

__device__ __forceinline__ std::uint64_t wave_prefix_max64(std::uint64_t v)
{
    std::uint64_t t;
    t = dpp64<0x111, 0xF>(v); v = umax64(v, t);
    t = dpp64<0x112, 0xF>(v); v = umax64(v, t);
    t = dpp64<0x114, 0xF>(v); v = umax64(v, t);
    t = dpp64<0x118, 0xF>(v); v = umax64(v, t);
    t = dpp64<0x142, 0xA>(v); v = umax64(v, t);
    t = dpp64<0x143, 0xC>(v); v = umax64(v, t);
    return v;
}

__device__ __forceinline__ std::uint64_t readlane64(std::uint64_t v, int lane)
{
    const std::uint32_t lo = static_cast<std::uint32_t>(
        __builtin_amdgcn_readlane(static_cast<int>(static_cast<std::uint32_t>(v)), lane));
    const std::uint32_t hi = static_cast<std::uint32_t>(
        __builtin_amdgcn_readlane(static_cast<int>(static_cast<std::uint32_t>(v >> 32)), lane));
    return (static_cast<std::uint64_t>(hi) << 32) | lo;
}

// The lane below's value (0 in lane 0), by a DPP wave shift (wave_shr:1 = 0x138):
// two VALU moves where a shuffle is two LDS operations.
__device__ __forceinline__ std::uint64_t prev_lane64(std::uint64_t v)
{
    return dpp64<0x138, 0xF>(v);
}

// The range table as a kernel sees it: the fences in LDS and, where the whole
// table is held there too (KArgs::r_lds), each range's length | mode << 56 |
// permissions << 60, its first media page and, in hybrid runs, its id.  A
// lookup then makes no vector-memory load: those made a step of records spread
// over several ranges wait for the whole record pipeline.
struct RangeView {
    const std::uint64_t* fence;
    const std::uint64_t* len = nullptr;
    const std::uint32_t* page0 = nullptr;
    const std::uint32_t* id = nullptr;
    __device__ __forceinline__ RangeView(const std::uint64_t* f) : fence(f) {}
};
constexpr std::uint64_t kRangeLenMask = (1ull << 56) - 1;

// find_range_index (hbf_device.cuh:826-841): upper_bound(base) - 1 over the
// sorted range table.  The top level runs over every `stride`-th base,
// staged in LDS; the bottom level over at most `stride` bases in memory.
__device__ __forceinline__ std::uint32_t find_range(const KArgs& a, const RangeView& rv,
                                                    std::uint64_t addr)
{
    std::uint32_t lo = 0, hi = a.r_nfence;
    while (lo < hi) {
        const std::uint32_t mid = (lo + hi) >> 1;
        if (rv.fence[mid] <= addr) {
            lo = mid + 1;
        } else {
            hi = mid;
        }
    }
    if (lo == 0) {
        return a.r_count;
    }
    if (a.r_lds != 0) {
        return lo - 1;  // every base is a fence
    }
    const std::uint32_t start = (lo - 1) * a.r_stride;
    std::uint32_t end = start + a.r_stride;
    end = end < a.r_count ? end : a.r_count;
    std::uint32_t l2 = start + 1, h2 = end;
    while (l2 < h2) {
        const std::uint32_t mid = (l2 + h2) >> 1;
        if (a.r_base[mid] <= addr) {
            l2 = mid + 1;
        } else {
            h2 = mid;
        }
    }
    return l2 - 1;
}

// range_overlaps (hbf_device.cuh:873-884)
__device__ __forceinline__ bool overlaps(std::uint64_t base, std::uint64_t length,
                                         std::uint64_t addr, std::uint64_t bytes)
{
    if (bytes == 0 || length == 0 || base > ~0ull - length || addr > ~0ull - bytes) {
        return false;
    }
    return addr < base + length && base < addr + bytes;
}

__device__ __forceinline__ std::uint64_t xfer_ps(const KArgs& a, std::uint64_t bytes)
{
    if ((bytes & (bytes - 1)) == 0 && bytes != 0 && bytes <= (1ull << 32)) {
        return a.xfer_pow2[63 - __clzll(bytes)];
    }
    return a.xfer_q * ((bytes * a.xfer_num + a.xfer_den - 1) / a.xfer_den);
}

// The same with the power-of-two table in LDS, for per-lane byte counts: a
// lane-indexed read of the kernel arguments would be a vector memory load,
// and the record pipeline keeps those out of the step loop.
__device__ __forceinline__ std::uint64_t xfer_ps_lds(const KArgs& a, const std::uint64_t* xp,
                                                     std::uint64_t bytes)
{
    if ((bytes & (bytes - 1)) == 0 && bytes != 0 && bytes <= (1ull << 32)) {
        return xp[63 - __clzll(bytes)];
    }
    return a.xfer_q * ((bytes * a.xfer_num + a.xfer_den - 1) / a.xfer_den);
}

// Copies the power-of-two transfer table into LDS (`xp`, 33 entries).
__device__ __forceinline__ void load_xfer_table(const KArgs& a, std::uint64_t* xp, int lane)
{
    if (lane < 33) {
        xp[lane] = a.xfer_pow2[lane];
    }
}

// The same in two halves, so that later loads can be issued in between.
__device__ __forceinline__ std::uint64_t fetch_xfer(const KArgs& a, int lane)
{
    return lane < 33 ? a.xfer_pow2[lane] : 0ull;
}

__device__ __forceinline__ void store_xfer(std::uint64_t* xp, std::uint64_t v, int lane)
{
    if (lane < 33) {
        xp[lane] = v;
    }
}

// Waits for every outstanding vector memory operation (s_waitcnt vmcnt(0)).
// Called where a step has just made its own per-lane loads, so that none of
// them is still outstanding when the next step starts: the record pipeline's
// group in flight is then waited on only when the wave needs it.
__device__ __forceinline__ void wait_vector_loads()
{
    __builtin_amdgcn_s_waitcnt(0x0f70);  // vmcnt 0, expcnt 7, lgkmcnt 15: vmcnt only
}

// Range last found by this lane.  Ranges are disjoint, so an address inside
// the cached range is inside no other one and the search can be skipped.
struct RangeCache {
    std::uint64_t base;
    std::uint64_t end;
    std::uint64_t file_offset;
    std::uint32_t meta;
    std::uint32_t id;
};

__device__ __forceinline__ RangeCache empty_cache()
{
    RangeCache c;
    c.base = 1;
    c.end = 0;
    c.file_offset = 0;
    c.meta = 0;
    c.id = 0;
    return c;
}

__device__ __forceinline__ void load_record(const hbf_record32* rec, std::size_t i, uint4& x,
                                            uint4& y)
{
    const uint4* p = reinterpret_cast<const uint4*>(rec + i);
    x = p[0];
    y = p[1];
}

// Records reach a wave in groups of kPipe steps: while the wave works through
// one group (held in registers), the next group's loads are in flight, so
// each wave keeps kPipe * 2 KiB of reads outstanding for kPipe steps of
// work.  (A load queue rotated one step at a time would wait on the newest
// load at every step, since the rotation copies it.)  A step's 2 KiB arrive
// coalesced, 16 B per lane: half A holds records 0..31 and half B records
// 32..63, lane l holding word pair l & 1 of record l >> 1 (even lanes address
// and bytes, odd lanes issue time and operation).  Loading record-per-lane
// instead (32 B stride) caps the read rate at ~4.8 TB/s; the coalesced form
// streams at ~6.3 TB/s.  Within the current group the next step is always
// slot 0: taking a step shifts the group down by one slot, register moves
// with constant indices that wait on nothing in flight (a selection by step
// index would put the group in scratch memory).
constexpr int kPipe = 4;
// The summary pass of 32-byte records, whose occupancy its per-plane LDS
// state limits (not its registers), keeps twice as many steps in flight per
// wave.
constexpr int kSumPipe = 8;
// Packed records in the summary pass: four waves per SIMD with three steps in
// flight each.  Measured against three waves with eight steps: general
// streams +8% per step (k_summary 4.15 -> 3.57 ms at 2^28 records) and the
// paged-KV step +15%, the TinyLlama step 2% slower; the LDS-bound variant
// (kDeep) keeps 2 * kSumPipe at two waves.  A run whose tiles all fit in one
// round of three-wave slots (kFewTiles) leaves SIMDs without a fourth wave
// anyway: it keeps three waves with kSumPipe steps in flight (kFew).
constexpr int kPackedSumPipe = 3;
constexpr std::size_t kFewTiles = 3 * 4 * 256;  // waves per SIMD x SIMDs per CU x CUs
// Linear-step detection on streams that show none: after kLinGiveUp steps in
// a row fail it, a wave probes only every kLinProbe-th step until one
// passes (every step is exact on the general path too; random streams stop
// paying for the check).
constexpr std::uint32_t kLinGiveUp = 8;
constexpr std::size_t kLinProbe = 32;

// A step in the registers of one lane: the coalesced halves of 32-byte
// records, or one packed 16-byte record.
struct Step32 {
    uint4 A, B;
};
struct Step16 {
    uint4 R;
};

// Records are read once per pass and streamed, so their loads are
// non-temporal: they then leave the caches to what the passes read again (the
// tile summaries, descriptors and carries).  Config 2: the step 6% faster.
__device__ __forceinline__ uint4 load_stream(const uint4* p)
{
    typedef unsigned int u32x4 __attribute__((ext_vector_type(4)));
    const u32x4 v = __builtin_nontemporal_load(reinterpret_cast<const u32x4*>(p));
    return make_uint4(v.x, v.y, v.z, v.w);
}

template <int D>
struct RecordPipeT {
    using Step = Step32;
    uint4 ca[D], cb[D];  // the group being worked through
    uint4 na[D], nb[D];  // the next group, in flight

    __device__ __forceinline__ void issue(const void* rec, std::size_t g, std::size_t end,
                                          int lane)
    {
        const uint4* p = reinterpret_cast<const uint4*>(rec);
        if (g + static_cast<std::size_t>(D) * kWave <= end) {
            // the whole group lies inside the tile (every group but a tile's
            // last): plain loads, no per-load bounds or zero fill
            const uint4* q = p + 2 * g + static_cast<std::size_t>(lane);
#pragma unroll
            for (int j = 0; j < D; ++j) {
                na[j] = load_stream(q + static_cast<std::size_t>(2 * j) * kWave);
                nb[j] = load_stream(q + static_cast<std::size_t>(2 * j + 1) * kWave);
            }
            return;
        }
        const std::size_t words = 2 * end;  // 16-byte words in the tile's records
#pragma unroll
        for (int j = 0; j < D; ++j) {
            const std::size_t w = 2 * (g + static_cast<std::size_t>(j) * kWave) + lane;
            na[j] = make_uint4(0, 0, 0, 0);
            nb[j] = na[j];
            if (w < words) {
                na[j] = p[w];
            }
            if (w + kWave < words) {
                nb[j] = p[w + kWave];
            }
        }
    }
    // Makes the group in flight current (waiting for it).
    __device__ __forceinline__ void promote()
    {
#pragma unroll
        for (int j = 0; j < D; ++j) {
            ca[j] = na[j];
            cb[j] = nb[j];
        }
    }
    // Makes the group in flight current and issues the one after it.
    __device__ __forceinline__ void advance(const void* rec, std::size_t next, std::size_t end,
                                            int lane)
    {
        promote();
        if (next < end) {
            issue(rec, next, end, lane);
        }
    }
    // The current group's next step, in the coalesced halves.
    __device__ __forceinline__ void take(Step32& st)
    {
        st.A = ca[0];
        st.B = cb[0];
#pragma unroll
        for (int j = 0; j + 1 < D; ++j) {
            ca[j] = ca[j + 1];
            cb[j] = cb[j + 1];
        }
    }
};

// Packed records (hbf_record16, 16 B): word 0 holds the address (bits 0-47)
// and byte count (bits 48-63), word 1 the issue time (bits 0-55) and the
// operation (bits 56-63).  A step is 1 KiB and lane r loads record r whole,
// so no transpose is needed, and a group holds one register quad per step.
template <int D>
struct PackedPipeT {
    using Step = Step16;
    uint4 c[D];   // the group being worked through
    uint4 nx[D];  // the next group, in flight

    __device__ __forceinline__ void issue(const void* rec, std::size_t g, std::size_t end,
                                          int lane)
    {
        const uint4* p = reinterpret_cast<const uint4*>(rec);
        if (g + static_cast<std::size_t>(D) * kWave <= end) {
            const uint4* q = p + g + static_cast<std::size_t>(lane);
#pragma unroll
            for (int j = 0; j < D; ++j) {
                nx[j] = load_stream(q + static_cast<std::size_t>(j) * kWave);
            }
            return;
        }
#pragma unroll
        for (int j = 0; j < D; ++j) {
            const std::size_t i = g + static_cast<std::size_t>(j) * kWave + lane;
            nx[j] = make_uint4(0, 0, 0, 0);
            if (i < end) {
                nx[j] = p[i];
            }
        }
    }
    __device__ __forceinline__ void promote()
    {
#pragma unroll
        for (int j = 0; j < D; ++j) {
            c[j] = nx[j];
        }
    }
    __device__ __forceinline__ void advance(const void* rec, std::size_t next, std::size_t end,
                                            int lane)
    {
        promote();
        if (next < end) {
            issue(rec, next, end, lane);
        }
    }
    __device__ __forceinline__ void take(Step16& st)
    {
        st.R = c[0];
#pragma unroll
        for (int j = 0; j + 1 < D; ++j) {
            c[j] = c[j + 1];
        }
    }
};

// A packed record in the two word quads the decoder takes (x: address,
// bytes; y: issue time, operation).
__device__ __forceinline__ void unpack16(const uint4& r, uint4& x, uint4& y)
{
    x = make_uint4(r.x, r.y & 0xffffu, r.y >> 16, 0u);
    y = make_uint4(r.z, r.w & 0xffffffu, r.w >> 24, 0u);
}

using RecordPipe = RecordPipeT<kPipe>;

// Record-per-lane form of a step (lane r gets record r's two word pairs).
__device__ __forceinline__ void to_records(const uint4& A, const uint4& B, int lane, uint4& x,
                                           uint4& y)
{
    const int sx = ((2 * lane) & 63) << 2;  // bpermute byte addresses
    const int sy = ((2 * lane + 1) & 63) << 2;
    const bool lo = lane < 32;
    const auto pick = [&](std::uint32_t a, std::uint32_t b, int src) {
        const std::uint32_t ta =
            static_cast<std::uint32_t>(__builtin_amdgcn_ds_bpermute(src, static_cast<int>(a)));
        const std::uint32_t tb =
            static_cast<std::uint32_t>(__builtin_amdgcn_ds_bpermute(src, static_cast<int>(b)));
        return lo ? ta : tb;
    };
    x = make_uint4(pick(A.x, B.x, sx), pick(A.y, B.y, sx), pick(A.z, B.z, sx),
                   pick(A.w, B.w, sx));
    y = make_uint4(pick(A.x, B.x, sy), pick(A.y, B.y, sy), pick(A.z, B.z, sy), 0);
}

__device__ __forceinline__ void step_records(const Step32& st, int lane, uint4& x, uint4& y)
{
    to_records(st.A, st.B, lane, x, y);
}

__device__ __forceinline__ void step_records(const Step16& st, int, uint4& x, uint4& y)
{
    unpack16(st.R, x, y);
}

// Channel and global plane id of a media page (the profile's allocation
// scheme, fastest axis first).
__device__ __forceinline__ void stripe(const KArgs& a, std::uint64_t page, Dec& d)
{
    if (a.flat) {
        return;
    }
    std::uint32_t c[4];
    if (a.pow2) {
#pragma unroll
        for (int ax = 0; ax < 4; ++ax) {
            c[ax] = static_cast<std::uint32_t>((page >> a.axis_shift[ax]) &
                                               (a.axis_size[ax] - 1));
        }
    } else {
#pragma unroll
        for (int ax = 0; ax < 4; ++ax) {
            c[ax] = static_cast<std::uint32_t>((page / a.axis_div[ax]) % a.axis_size[ax]);
        }
    }
    d.chan = c[0];
    d.plane = ((c[0] * a.W + c[1]) * a.D + c[2]) * a.P + c[3];
}

// A wave's stripe table: entry r = plane | channel << 20 of media page r,
// r < Rp.  With power-of-two axes every axis digit is a bit field of the
// page's low log2(Rp) bits, so page p stripes as p mod Rp does.
__device__ __forceinline__ void fill_stripe_table(const KArgs& a, std::uint32_t* stab, int lane)
{
    for (std::uint32_t r = static_cast<std::uint32_t>(lane); r < a.Rp; r += kWave) {
        Dec d;
        d.plane = 0;
        d.chan = 0;
        stripe(a, r, d);
        stab[r] = d.plane | (d.chan << 20);
    }
}

// The operation a decoded record carries (hybrid sampler key).
__device__ __forceinline__ std::uint32_t dec_op(std::uint32_t bits)
{
    return (bits & 4u) ? kOpRefresh : (bits & 1u);
}

// Classification in the resolver's order (hbf_device.cu:1081-1165) followed
// by striping of the media page.  Refresh records are recognised only in
// the kRefresh instantiation (streams the thermal-coupled run merged them
// into); the other streams keep the branch out of the hot loop.  `stab`:
// the wave's stripe table (fill_stripe_table), when the run keeps one.
template <bool kRefresh, bool kUniform = false>
__device__ __forceinline__ Dec decode(const KArgs& a, const RangeView& fence, RangeCache& rc,
                                      const uint4& x, const uint4& y, std::uint64_t base_ps,
                                      const std::uint32_t* stab = nullptr)
{
    const std::uint64_t addr = x.x | (static_cast<std::uint64_t>(x.y) << 32);
    const std::uint64_t bytes = x.z | (static_cast<std::uint64_t>(x.w) << 32);
    const std::uint64_t issue_rel = y.x | (static_cast<std::uint64_t>(y.y) << 32);
    const std::uint32_t op = y.z & 0xffu;
    Dec d;
    d.issue = base_ps + issue_rel;
    d.bits = op & 1u;
    d.plane = 0;
    d.chan = 0;
    d.range_id = 0;
    d.page1 = 0;
    d.xfer = 0;
    d.xbytes = 0;
    if (kRefresh && op == kOpRefresh && (y.z & kMediaFlag) != 0) {
        if (bytes == 0 || bytes > 0xffffffffull || addr >= a.media_pages) {
            d.cls = kClsUnsupported;
            return d;
        }
        d.cls = kClsModeled;
        d.bits = 7u;
        d.page1 = addr + 1;
        d.xbytes = bytes;
        stripe(a, addr, d);
        return d;
    }
    if (!(addr >= rc.base && addr < rc.end)) {
        std::uint32_t idx = find_range(a, fence, addr);
        if (kUniform) {
            // wave-uniform record: keep the range in scalar registers
            idx = static_cast<std::uint32_t>(__builtin_amdgcn_readfirstlane(static_cast<int>(idx)));
        }
        if (a.r_lds != 0) {
            const std::uint64_t base = idx == a.r_count ? 0ull : fence.fence[idx];
            const std::uint64_t lm = idx == a.r_count ? 0ull : fence.len[idx];
            if (idx == a.r_count || addr - base >= (lm & kRangeLenMask)) {
                const std::uint32_t succ = idx == a.r_count ? 0u : idx + 1u;
                d.cls = bytes > 0xffffffffull ||
                                (succ < a.r_count &&
                                 overlaps(fence.fence[succ], fence.len[succ] & kRangeLenMask, addr,
                                          bytes))
                            ? kClsUnsupported
                            : kClsBypass;
                return d;
            }
            rc.base = base;
            rc.end = base + (lm & kRangeLenMask);
            rc.file_offset = static_cast<std::uint64_t>(fence.page0[idx]) << a.page_shift;
            rc.meta = static_cast<std::uint32_t>(lm >> 56) & 0xfu;
            rc.meta |= static_cast<std::uint32_t>(lm >> 60) << 8;
            rc.id = a.hybrid != 0 ? fence.id[idx] : 0u;
        } else {
        if (idx == a.r_count || addr < a.r_base[idx] ||
            addr - a.r_base[idx] >= a.r_length[idx]) {
            const std::uint32_t succ = idx == a.r_count ? 0u : idx + 1u;
            if (bytes > 0xffffffffull ||
                (succ < a.r_count && overlaps(a.r_base[succ], a.r_length[succ], addr, bytes))) {
                d.cls = kClsUnsupported;
            } else {
                d.cls = kClsBypass;
            }
            return d;
        }
        rc.base = a.r_base[idx];
        rc.end = rc.base + a.r_length[idx];
        rc.file_offset = a.r_file_offset[idx];
        rc.meta = a.r_meta[idx];
        rc.id = a.r_id[idx];
        if (!kUniform) {
            wait_vector_loads();
        }
        }
    }
    const std::uint32_t mode = rc.meta & 0xffu;
    const std::uint32_t perms = rc.meta >> 8;
    const std::uint64_t page_mask = (1ull << a.page_shift) - 1;
    // access_supported (hbf_device.cuh:843-860); the range's own bounds and
    // page size are validated at registration.
    if (bytes == 0 || bytes > 0xffffffffull || op > 1 || (mode != 1 && mode != 2) ||
        bytes > ~0ull - addr || addr + bytes > rc.end || (perms & (1u << op)) == 0) {
        d.cls = kClsUnsupported;
        return d;
    }
    const std::uint64_t off = addr - rc.base;
    if ((off >> a.page_shift) != ((off + bytes - 1) >> a.page_shift)) {
        d.cls = kClsUnsupported;
        return d;
    }
    if ((off & ~page_mask) > ~0ull - rc.file_offset) {
        d.cls = kClsUnsupported;
        return d;
    }
    d.cls = kClsModeled;
    d.range_id = rc.id;
    const std::uint64_t media = rc.file_offset + off;
    const std::uint64_t page = media >> a.page_shift;
    d.page1 = page + 1;
    const std::uint64_t page_bytes = 1ull << a.page_shift;
    if (op == 1 && (a.every_write || (media & page_mask) + bytes == page_bytes)) {
        d.bits |= 2u;
    }
    d.xbytes = a.transfer_page ? page_bytes : bytes;
    // (striping written out here rather than through stripe(): the helper
    // costs the summary kernel a quarter of its speed)
    if (!a.flat && stab != nullptr) {
        // plane | channel << 20 of the page modulo Rp (a power of two)
        const std::uint32_t e = stab[static_cast<std::uint32_t>(page) & (a.Rp - 1)];
        d.chan = e >> 20;
        d.plane = e & 0xfffffu;
    } else if (!a.flat) {
        std::uint32_t c[4];
        if (a.pow2) {
#pragma unroll
            for (int ax = 0; ax < 4; ++ax) {
                c[ax] = static_cast<std::uint32_t>((page >> a.axis_shift[ax]) &
                                                   (a.axis_size[ax] - 1));
            }
        } else {
#pragma unroll
            for (int ax = 0; ax < 4; ++ax) {
                c[ax] = static_cast<std::uint32_t>((page / a.axis_div[ax]) % a.axis_size[ax]);
            }
        }
        d.chan = c[0];
        d.plane = ((c[0] * a.W + c[1]) * a.D + c[2]) * a.P + c[3];
    }
    return d;
}

__device__ __forceinline__ Dec invalid_dec()
{
    Dec d;
    d.cls = kClsInvalid;
    d.bits = 0;
    d.plane = d.chan = d.range_id = 0;
    d.page1 = d.issue = d.xfer = d.xbytes = 0;
    return d;
}

// Transfer time of every lane's access.  When all modeled lanes move the same
// byte count (the usual case) it is computed once, in scalar registers.
__device__ __forceinline__ std::uint64_t lane_xfer(const KArgs& a, const std::uint64_t* xp,
                                                   const Dec& d, bool m, std::uint64_t active,
                                                   bool& uniform)
{
    const int first = __ffsll(static_cast<long long>(active)) - 1;
    const std::uint32_t lo = static_cast<std::uint32_t>(
        __builtin_amdgcn_readlane(static_cast<int>(static_cast<std::uint32_t>(d.xbytes)), first));
    const std::uint32_t hi = static_cast<std::uint32_t>(__builtin_amdgcn_readlane(
        static_cast<int>(static_cast<std::uint32_t>(d.xbytes >> 32)), first));
    const std::uint64_t xb0 = (static_cast<std::uint64_t>(hi) << 32) | lo;
    uniform = __ballot(m && d.xbytes != xb0) == 0;
    if (uniform) {
        return xfer_ps(a, xb0);
    }
    return m ? xfer_ps_lds(a, xp, d.xbytes) : 0ull;
}

// Time origin for 32-bit scans: the first active lane's issue time.  The
// narrow path is taken only when, for every modeled lane, issue - origin is
// in [0, 2^30) and both services are below 2^24, so every partial sum of a
// step fits 32 bits.  (0, 0) in relative form stands for (0, origin), which
// acts as the identity on every state reachable in the step.
struct Narrow {
    std::uint64_t origin;
    bool ok;
};

__device__ __forceinline__ Narrow narrow_check(const Dec& d, bool m, std::uint64_t active,
                                               std::uint64_t svc1, std::uint64_t svc2)
{
    const int first = __ffsll(static_cast<long long>(active)) - 1;
    Narrow n;
    n.origin = readlane64(d.issue, first);
    const bool bad = m && (d.issue < n.origin || d.issue - n.origin >= (1ull << 30) ||
                           svc1 >= (1ull << 24) || svc2 >= (1ull << 24));
    n.ok = __ballot(bad) == 0;
    return n;
}

// A sequential run step: all 64 lanes are modeled reads of one media page,
// with the same byte count, in non-decreasing issue order (weight and KV
// streaming produce these).  With at least one page register, lanes 1..63
// hit the page their predecessor just read (plane map (0, issue_i)), and with
// a constant transfer x the channel maps fold to one prefix maximum:
//   lane i's channel map = (x (i + 1), x (i + 1) + max_{k<=i} (issue_k - x k)).
// Wave-uniform.
__device__ __forceinline__ bool run_step(const KArgs& a, const Dec& d, std::uint64_t active,
                                         int lane)
{
    if (active != ~0ull || a.slots == 0) {
        return false;
    }
    const std::uint32_t page0 = static_cast<std::uint32_t>(
        __builtin_amdgcn_readlane(static_cast<int>(static_cast<std::uint32_t>(d.page1)), 0));
    if (__ballot(static_cast<std::uint32_t>(d.page1) != page0) != 0) {
        return false;  // (scattered streams leave here)
    }
    const std::uint64_t bytes0 = readlane64(d.xbytes, 0);
    const std::uint64_t prev = prev_lane64(d.issue);
    const bool bad = (d.bits & 1u) != 0 || d.xbytes != bytes0 || (lane != 0 && d.issue < prev);
    return __ballot(bad) == 0;
}

// W_i = max_{k<=i} (issue_k + x (63 - k)) for a run step, so that the channel
// completion of lane i is max(cursor + x (i + 1), W_i - x (62 - i)).  Runs in
// 32 bits relative to lane 0's issue when the step's span allows.
__device__ __forceinline__ std::uint64_t run_channel_max(const Dec& d, std::uint64_t x, int lane)
{
    const std::uint64_t w = d.issue + x * static_cast<std::uint64_t>(63 - lane);
    const std::uint64_t i0 = readlane64(d.issue, 0);
    const std::uint64_t i63 = readlane64(d.issue, 63);
    if (i63 - i0 + 64 * x < (1ull << 31) && x < (1ull << 24)) {
        return i0 + wave_prefix_max32(static_cast<std::uint32_t>(w - i0));
    }
    return wave_prefix_max64(w);
}

__device__ __forceinline__ std::uint32_t rfl32(std::uint32_t v)
{
    return static_cast<std::uint32_t>(__builtin_amdgcn_readfirstlane(static_cast<int>(v)));
}

// A linear step: 64 reads addr_0 + k * bytes_0 with one issue time, inside
// one page of one range (weight streaming issues whole page-halves in one
// slot).  Such a step touches one plane and one channel; lanes 1..63 hit the
// page lane 0 opened, so its effect has a closed form given lane 0's record.
// linear_detect checks a step in scalar registers against the wave-uniform
// range cache (the full decode runs only when the cache misses) and returns
// the step's media page + 1, issue time and byte count.  Anything else (and
// any step with fewer than 64 records) takes the general paths.
__device__ __forceinline__ std::uint32_t rl32(std::uint32_t v, int k)
{
    return static_cast<std::uint32_t>(__builtin_amdgcn_readlane(static_cast<int>(v), k));
}

// The range and page checks of a step whose 64 records already follow
// record 0 (xu: its address and bytes, yu: its issue time and operation).
template <bool kRefresh>
__device__ __forceinline__ bool linear_tail(const KArgs& a, const RangeView& fence,
                                            RangeCache& rcu, const uint4& xu, const uint4& yu,
                                            std::uint64_t base_ps, std::uint32_t& page1,
                                            std::uint64_t& issue0, std::uint32_t& bytes0);

template <bool kRefresh>
__device__ __forceinline__ bool linear_detect(const KArgs& a, const RangeView& fence,
                                              RangeCache& rcu, const Step32& st,
                                              std::uint64_t base_ps, bool full, int lane,
                                              std::uint32_t& page1, std::uint64_t& issue0,
                                              std::uint32_t& bytes0)
{
    if (!full) {
        return false;
    }
    const uint4& A = st.A;
    const uint4& B = st.B;
    // record 0: address and bytes in lane 0, issue and operation in lane 1
    const uint4 xu = make_uint4(rfl32(A.x), rfl32(A.y), rfl32(A.z), rfl32(A.w));
    const uint4 yu = make_uint4(rl32(A.x, 1), rl32(A.y, 1), rl32(A.z, 1), 0);
    if ((yu.z & 0xffu) != 0 || xu.w != 0 || xu.z == 0) {
        return false;  // reads of 1 .. 2^32 - 1 bytes only
    }
    const std::uint64_t a0 = xu.x | (static_cast<std::uint64_t>(xu.y) << 32);
    // lane l checks word pair l & 1 of records l >> 1 (half A) and 32 + (l >> 1) (half B)
    const std::uint64_t ea = a0 + static_cast<std::uint64_t>(lane >> 1) * xu.z;
    const std::uint64_t eb = ea + 32ull * xu.z;
    const std::uint64_t wa = A.x | (static_cast<std::uint64_t>(A.y) << 32);
    const std::uint64_t wb = B.x | (static_cast<std::uint64_t>(B.y) << 32);
    const bool odd = (lane & 1) != 0;
    const bool ok_even = wa == ea && A.z == xu.z && A.w == 0 && wb == eb && B.z == xu.z &&
                         B.w == 0;
    const bool ok_odd = A.x == yu.x && A.y == yu.y && A.z == yu.z && B.x == yu.x &&
                        B.y == yu.y && B.z == yu.z;
    if (__ballot(odd ? !ok_odd : !ok_even) != 0) {
        return false;
    }
    return linear_tail<kRefresh>(a, fence, rcu, xu, yu, base_ps, page1, issue0, bytes0);
}

// A packed step: lane l checks its own record against record 0.
template <bool kRefresh>
__device__ __forceinline__ bool linear_detect(const KArgs& a, const RangeView& fence,
                                              RangeCache& rcu, const Step16& st,
                                              std::uint64_t base_ps, bool full, int lane,
                                              std::uint32_t& page1, std::uint64_t& issue0,
                                              std::uint32_t& bytes0)
{
    if (!full) {
        return false;
    }
    const uint4& R = st.R;
    const uint4 r0 = make_uint4(rfl32(R.x), rfl32(R.y), rfl32(R.z), rfl32(R.w));
    uint4 xu, yu;
    unpack16(r0, xu, yu);
    if (yu.z != 0 || xu.z == 0) {
        return false;  // reads of at least one byte only
    }
    const std::uint64_t a0 = xu.x | (static_cast<std::uint64_t>(xu.y) << 32);
    const std::uint64_t mine = a0 + static_cast<std::uint64_t>(lane) * xu.z;
    const bool ok = R.x == static_cast<std::uint32_t>(mine) &&
                    (R.y & 0xffffu) == (mine >> 32) && (R.y >> 16) == xu.z && R.z == r0.z &&
                    R.w == r0.w;
    if (__ballot(!ok) != 0) {
        return false;
    }
    return linear_tail<kRefresh>(a, fence, rcu, xu, yu, base_ps, page1, issue0, bytes0);
}

template <bool kRefresh>
__device__ __forceinline__ bool linear_tail(const KArgs& a, const RangeView& fence,
                                            RangeCache& rcu, const uint4& xu, const uint4& yu,
                                            std::uint64_t base_ps, std::uint32_t& page1,
                                            std::uint64_t& issue0, std::uint32_t& bytes0)
{
    const std::uint64_t a0 = xu.x | (static_cast<std::uint64_t>(xu.y) << 32);
    if (!(a0 >= rcu.base && a0 < rcu.end)) {
        // refill the cache through the full classification
        const Dec d = decode<kRefresh, true>(a, fence, rcu, xu, yu, base_ps);
        if (d.cls != kClsModeled) {
            return false;
        }
    }
    // every record inside the cached range, which admits reads, and in one
    // page whose media offset does not wrap (access_supported,
    // hbf_device.cuh:843-860, for all 64 records at once)
    const std::uint32_t mode = rcu.meta & 0xffu;
    const std::uint64_t span = 64ull * xu.z;
    if ((mode != 1 && mode != 2) || (rcu.meta & (1u << 8)) == 0 || span > rcu.end - a0) {
        return false;
    }
    const std::uint64_t off0 = a0 - rcu.base;
    const std::uint64_t page_mask = (1ull << a.page_shift) - 1;
    if ((off0 >> a.page_shift) != ((off0 + span - 1) >> a.page_shift) ||
        (off0 & ~page_mask) > ~0ull - rcu.file_offset) {
        return false;
    }
    page1 = static_cast<std::uint32_t>(((rcu.file_offset + off0) >> a.page_shift) + 1);
    issue0 = base_ps + (yu.x | (static_cast<std::uint64_t>(yu.y) << 32));
    bytes0 = xu.z;
    return true;
}

// A linear step (k = 0: one run of 64) or a split step (two linear runs,
// lanes 0 .. k-1 and k .. 63, with one issue time and byte count).
struct LinStep {
    std::uint32_t page1, page1b, k, bytes, rid, ridb;
    std::uint64_t issue;
};

// A step whose records all share record 0's byte count (b0), issue
// time and read operation, and whose addresses continue record 0's (one run,
// split where a page boundary falls inside it) or continue record 0's up to
// a lane k and lane k's after it (two spans joined).  Each run must lie in
// one page of a range that admits reads (access_supported,
// hbf_device.cuh:843-860, for the run's records at once); a run whose first
// address lies outside the wave-uniform range cache refills it through the
// full classification (one call site for both runs).
template <bool kRefresh>
__device__ __forceinline__ bool split_runs(const KArgs& a, const RangeView& fence,
                                           RangeCache& rcu, std::uint64_t addr,
                                           std::uint32_t b0, const uint4& yu,
                                           std::uint64_t base_ps, int lane, LinStep& ls)
{
    const std::uint64_t a0 = readlane64(addr, 0);
    const std::uint64_t breaks = __ballot(addr != a0 + static_cast<std::uint64_t>(lane) * b0);
    std::uint32_t k = 0;  // the split lane (0: none)
    std::uint64_t a1 = 0;
    if (breaks != 0) {
        k = static_cast<std::uint32_t>(__ffsll(static_cast<long long>(breaks)) - 1);
        a1 = readlane64(addr, static_cast<int>(k));
        const std::uint64_t own =
            a1 + static_cast<std::uint64_t>(lane - static_cast<int>(k)) * b0;
        if (__ballot(lane >= static_cast<int>(k) && addr != own) != 0) {
            return false;
        }
    }
    ls.issue = base_ps + (yu.x | (static_cast<std::uint64_t>(yu.y) << 32));
    ls.bytes = b0;
    ls.page1b = 0;
    ls.ridb = 0;
    const std::uint64_t page_mask = (1ull << a.page_shift) - 1;
    std::uint64_t at = a0;
    std::uint32_t cnt = k != 0 ? k : static_cast<std::uint32_t>(kWave);
    for (int part = 0; part < 2; ++part) {
        if (!(at >= rcu.base && at < rcu.end)) {
            const uint4 xa = make_uint4(static_cast<std::uint32_t>(at),
                                        static_cast<std::uint32_t>(at >> 32), b0, 0u);
            const Dec d = decode<kRefresh, true>(a, fence, rcu, xa, yu, base_ps);
            if (d.cls != kClsModeled) {
                return false;
            }
        }
        const std::uint32_t mode = rcu.meta & 0xffu;
        if ((mode != 1 && mode != 2) || (rcu.meta & (1u << 8)) == 0) {
            return false;
        }
        const std::uint64_t off = at - rcu.base;
        std::uint64_t span = static_cast<std::uint64_t>(cnt) * b0;
        if ((off >> a.page_shift) != ((off + span - 1) >> a.page_shift)) {
            // one run crossing a page boundary: split it there when the
            // boundary falls between two records
            const std::uint64_t room = (off | page_mask) + 1 - off;
            if (part != 0 || k != 0 || room % b0 != 0) {
                return false;
            }
            k = static_cast<std::uint32_t>(room / b0);
            a1 = a0 + room;
            cnt = k;
            span = room;
        }
        if (span > rcu.end - at || (off & ~page_mask) > ~0ull - rcu.file_offset) {
            return false;
        }
        const std::uint32_t page1 =
            static_cast<std::uint32_t>(((rcu.file_offset + off) >> a.page_shift) + 1);
        if (part == 0) {
            ls.page1 = page1;
            ls.rid = rcu.id;
            if (k == 0) {
                break;  // a whole linear step
            }
        } else {
            ls.page1b = page1;
            ls.ridb = rcu.id;
        }
        at = a1;
        cnt = static_cast<std::uint32_t>(kWave) - k;
    }
    ls.k = k;
    return true;
}

template <bool kRefresh>
__device__ __forceinline__ bool linear_detect_split(const KArgs& a, const RangeView& fence,
                                                    RangeCache& rcu, const Step16& st,
                                                    std::uint64_t base_ps, bool full, int lane,
                                                    LinStep& ls)
{
    if (!full) {
        return false;
    }
    const uint4& R = st.R;
    const uint4 r0 = make_uint4(rfl32(R.x), rfl32(R.y), rfl32(R.z), rfl32(R.w));
    uint4 xu, yu;
    unpack16(r0, xu, yu);
    if (yu.z != 0 || xu.z == 0) {
        return false;  // reads of at least one byte only
    }
    if (__ballot((R.y >> 16) != xu.z || R.z != r0.z || R.w != r0.w) != 0) {
        return false;
    }
    return split_runs<kRefresh>(a, fence, rcu,
                                R.x | (static_cast<std::uint64_t>(R.y & 0xffffu) << 32), xu.z, yu,
                                base_ps, lane, ls);
}

// 32-byte records: a whole step is found in the halves as they lie; only a
// step that is none is laid out record-per-lane for its runs.
template <bool kRefresh>
__device__ __forceinline__ bool linear_detect_split(const KArgs& a, const RangeView& fence,
                                                    RangeCache& rcu, const Step32& st,
                                                    std::uint64_t base_ps, bool full, int lane,
                                                    LinStep& ls)
{
    if (!full) {
        return false;
    }
    const std::uint32_t b0 = rfl32(st.A.z);
    const uint4 yu = make_uint4(rl32(st.A.x, 1), rl32(st.A.y, 1), rl32(st.A.z, 1), 0);
    if ((yu.z & 0xffu) != 0 || rfl32(st.A.w) != 0 || b0 == 0) {
        return false;  // reads of 1 .. 2^32 - 1 bytes only
    }
    // every even lane's byte count, every odd lane's issue time and flags
    const bool odd = (lane & 1) != 0;
    const bool ok_even = st.A.z == b0 && st.A.w == 0 && st.B.z == b0 && st.B.w == 0;
    const bool ok_odd = st.A.x == yu.x && st.A.y == yu.y && st.A.z == yu.z && st.B.x == yu.x &&
                        st.B.y == yu.y && st.B.z == yu.z;
    if (__ballot(odd ? !ok_odd : !ok_even) != 0) {
        return false;
    }
    const int src = ((2 * lane) & 63) << 2;
    const auto pick = [&](std::uint32_t u, std::uint32_t v) {
        const std::uint32_t tu =
            static_cast<std::uint32_t>(__builtin_amdgcn_ds_bpermute(src, static_cast<int>(u)));
        const std::uint32_t tv =
            static_cast<std::uint32_t>(__builtin_amdgcn_ds_bpermute(src, static_cast<int>(v)));
        return lane < 32 ? tu : tv;
    };
    const std::uint64_t addr = pick(st.A.x, st.B.x) |
                               (static_cast<std::uint64_t>(pick(st.A.y, st.B.y)) << 32);
    return split_runs<kRefresh>(a, fence, rcu, addr, b0, yu, base_ps, lane, ls);
}

// The step detection: with kSplit steps may be split; otherwise they are whole
// linear steps or none.
template <bool kRefresh, bool kSplit, typename Step>
__device__ __forceinline__ bool detect_step(const KArgs& a, const RangeView& fence,
                                            RangeCache& rcu, const Step& st,
                                            std::uint64_t base_ps, bool full, int lane,
                                            LinStep& ls)
{
    if constexpr (kSplit) {
        return linear_detect_split<kRefresh>(a, fence, rcu, st, base_ps, full, lane, ls);
    }
    ls.k = 0;
    ls.page1b = 0;
    ls.ridb = 0;
    const bool lin = linear_detect<kRefresh>(a, fence, rcu, st, base_ps, full, lane, ls.page1,
                                             ls.issue, ls.bytes);
    ls.rid = rcu.id;
    return lin;
}

// A linear group: D consecutive linear steps continuing one another
// (record r of the group at address a0 + r * bytes0), each step with its own
// issue time, all inside the cached range.  Checked at once on the group's
// registers: lane l looks at word pair l & 1 of records 64 j + 32 h + (l >> 1)
// for every step j and half h.  The step values live one step per lane
// (lane j < D: step j), not in D wave-uniform registers each: per-step
// scalar arrays would hold about 3 D scalar registers across the group's
// checks, more than the wave has beside the kernel's own, and the overflow
// goes to VGPR lanes one write and one read at a time.
template <int D>
struct GroupLin {
    std::uint32_t page1;  // lane j < D: step j's media page + 1
    std::uint64_t issue;  // lane j < D: step j's issue time
    std::uint32_t bytes;
};

template <bool kRefresh, int D>
__device__ __forceinline__ bool group_tail(const KArgs& a, const RangeView& fence,
                                           RangeCache& rcu, std::uint64_t base_ps,
                                           const uint4& xu, std::uint32_t op0, std::uint32_t vlo,
                                           std::uint32_t vhi, int lane, GroupLin<D>& gl);

template <bool kRefresh, int D>
__device__ __forceinline__ bool group_linear(const KArgs& a, const RangeView& fence,
                                             RangeCache& rcu, const RecordPipeT<D>& pipe,
                                             std::uint64_t base_ps, int lane, GroupLin<D>& gl)
{
    const uint4 xu = make_uint4(rfl32(pipe.ca[0].x), rfl32(pipe.ca[0].y), rfl32(pipe.ca[0].z),
                                rfl32(pipe.ca[0].w));
    const std::uint32_t op0 = rl32(pipe.ca[0].z, 1);
    if ((op0 & 0xffu) != 0 || xu.w != 0 || xu.z == 0) {
        return false;  // reads of 1 .. 2^32 - 1 bytes only
    }
    const std::uint64_t a0 = xu.x | (static_cast<std::uint64_t>(xu.y) << 32);
    const std::uint64_t b0 = xu.z;
    const std::uint64_t half = 32ull * b0;  // bytes between the two halves of a step
    const std::uint64_t mine = a0 + static_cast<std::uint64_t>(lane >> 1) * b0;
    const bool odd = (lane & 1) != 0;
    std::uint32_t vlo = 0, vhi = 0;  // lane j < D: step j's issue time
    bool ok = true;
#pragma unroll
    for (int j = 0; j < D; ++j) {
        const std::uint32_t ilo = rl32(pipe.ca[j].x, 1);
        const std::uint32_t ihi = rl32(pipe.ca[j].y, 1);
        vlo = lane == j ? ilo : vlo;
        vhi = lane == j ? ihi : vhi;
        const uint4& A = pipe.ca[j];
        const uint4& B = pipe.cb[j];
        const std::uint64_t ea = mine + static_cast<std::uint64_t>(2 * j) * half;
        const std::uint64_t eb = ea + half;
        const std::uint64_t wa = A.x | (static_cast<std::uint64_t>(A.y) << 32);
        const std::uint64_t wb = B.x | (static_cast<std::uint64_t>(B.y) << 32);
        const bool ev = wa == ea && A.z == xu.z && A.w == 0 && wb == eb && B.z == xu.z &&
                        B.w == 0;
        const bool od = A.x == ilo && A.y == ihi && A.z == op0 && B.x == ilo && B.y == ihi &&
                        B.z == op0;
        ok = ok && (odd ? od : ev);
    }
    if (__ballot(!ok) != 0) {
        return false;
    }
    return group_tail<kRefresh, D>(a, fence, rcu, base_ps, xu, op0, vlo, vhi, lane, gl);
}

// A packed group: lane l checks its own record of every step.
template <bool kRefresh, int D>
__device__ __forceinline__ bool group_linear(const KArgs& a, const RangeView& fence,
                                             RangeCache& rcu, const PackedPipeT<D>& pipe,
                                             std::uint64_t base_ps, int lane, GroupLin<D>& gl)
{
    const uint4 r0 = make_uint4(rfl32(pipe.c[0].x), rfl32(pipe.c[0].y), rfl32(pipe.c[0].z),
                                rfl32(pipe.c[0].w));
    uint4 xu, yu;
    unpack16(r0, xu, yu);
    if (yu.z != 0 || xu.z == 0) {
        return false;  // reads of at least one byte only
    }
    const std::uint64_t a0 = xu.x | (static_cast<std::uint64_t>(xu.y) << 32);
    const std::uint64_t b0 = xu.z;
    const std::uint64_t mine = a0 + static_cast<std::uint64_t>(lane) * b0;
    std::uint32_t vlo = 0, vhi = 0;  // lane j < D: step j's issue time
    bool ok = true;
#pragma unroll
    for (int j = 0; j < D; ++j) {
        const uint4& R = pipe.c[j];
        const std::uint32_t w = rfl32(R.w);  // record 0 of step j: issue high, operation
        const std::uint32_t ilo = rfl32(R.z);
        vlo = lane == j ? ilo : vlo;
        vhi = lane == j ? (w & 0xffffffu) : vhi;
        const std::uint64_t e = mine + static_cast<std::uint64_t>(j) * 64ull * b0;
        ok = ok && (w >> 24) == 0 && R.x == static_cast<std::uint32_t>(e) &&
             (R.y & 0xffffu) == (e >> 32) && (R.y >> 16) == b0 && R.z == ilo && R.w == w;
    }
    if (__ballot(!ok) != 0) {
        return false;
    }
    return group_tail<kRefresh, D>(a, fence, rcu, base_ps, xu, 0u, vlo, vhi, lane, gl);
}

// The range and page checks of a group whose records already continue one
// another from record 0 (xu: its address and bytes; op0: its operation;
// vlo, vhi: lane j < D holds step j's issue time), and the group's step
// values, lane j checking and holding step j.
template <bool kRefresh, int D>
__device__ __forceinline__ bool group_tail(const KArgs& a, const RangeView& fence,
                                           RangeCache& rcu, std::uint64_t base_ps,
                                           const uint4& xu, std::uint32_t op0, std::uint32_t vlo,
                                           std::uint32_t vhi, int lane, GroupLin<D>& gl)
{
    static_assert(D <= kWave, "one lane per step");
    const std::uint64_t a0 = xu.x | (static_cast<std::uint64_t>(xu.y) << 32);
    const std::uint64_t b0 = xu.z;
    if (!(a0 >= rcu.base && a0 < rcu.end)) {
        const uint4 yu = make_uint4(rl32(vlo, 0), rl32(vhi, 0), op0, 0);
        const Dec d = decode<kRefresh, true>(a, fence, rcu, xu, yu, base_ps);
        if (d.cls != kClsModeled) {
            return false;
        }
    }
    const std::uint32_t mode = rcu.meta & 0xffu;
    const std::uint64_t step = 64ull * b0;
    const std::uint64_t span = D * step;
    if ((mode != 1 && mode != 2) || (rcu.meta & (1u << 8)) == 0 || span > rcu.end - a0) {
        return false;
    }
    const std::uint64_t page_mask = (1ull << a.page_shift) - 1;
    const std::uint64_t off = a0 - rcu.base + static_cast<std::uint64_t>(lane) * step;
    // a step crossing a page, or a page whose file offset overflows
    const bool bad = lane < D && ((off >> a.page_shift) != ((off + step - 1) >> a.page_shift) ||
                                  (off & ~page_mask) > ~0ull - rcu.file_offset);
    if (__ballot(bad) != 0) {
        return false;
    }
    gl.page1 = static_cast<std::uint32_t>(((rcu.file_offset + off) >> a.page_shift) + 1);
    gl.issue = base_ps + (vlo | (static_cast<std::uint64_t>(vhi) << 32));
    gl.bytes = xu.z;
    return true;
}

// What the summary pass learned about a step, for the apply pass: a linear
// step's media page + 1, byte count and issue time (bytes == 0: any other
// step).  Indexed by record index / 64.
struct alignas(16) StepDesc {
    std::uint32_t page1;
    std::uint32_t bytes;
    std::uint64_t issue;
};

// Linear steps waiting to be folded, as runs: lane r (r < n) holds run r --
// m consecutive records of one step, issued together and reading one page
// (its media page + 1, byte count and issue time), starting at lane lo of
// that step.  A whole linear step is one run (m = 64, lo = 0); a split step
// (two linear runs, split at lane k: a page boundary inside the step, or two
// spans joined) is two, (m = k, lo = 0) and (m = 64 - k, lo = k).  Pending
// steps are always consecutive steps of the tile, `rows` of them, the first
// starting at record `first`; `split` says whether any is a split step.
// Only packed records form split steps (kRuns); in a batch of 32-byte
// records every run is a whole step, which len() and at() give as constants.
template <bool kRuns>
struct LinBatchT {
    std::uint32_t page1;
    std::uint32_t bytes;
    std::uint64_t issue;
    std::uint32_t rid;  // range id (kept by the apply pass, for hybrid sampling)
    std::uint32_t m;    // records of the run
    std::uint32_t lo;   // lane of its first record in its step
    std::size_t first;
    int n;
    int rows;
    bool split;

    __device__ __forceinline__ void push(std::uint32_t p1, std::uint64_t i0, std::uint32_t b0,
                                         std::size_t s, std::uint32_t r = 0)
    {
        if (n == 0) {
            first = s;
        }
        if (static_cast<int>(threadIdx.x) == n) {
            page1 = p1;
            bytes = b0;
            issue = i0;
            rid = r;
            m = kWave;
            lo = 0;
        }
        ++n;
        ++rows;
    }
    // A split step: lanes 0 .. k-1 read page pa - 1, lanes k .. 63 page pb - 1
    // (needs n <= 62).
    __device__ __forceinline__ void push_split(std::uint32_t pa, std::uint32_t pb, std::uint32_t k,
                                               std::uint64_t i0, std::uint32_t b0, std::size_t s,
                                               std::uint32_t ra, std::uint32_t rb)
    {
        if (n == 0) {
            first = s;
        }
        const int l = static_cast<int>(threadIdx.x);
        if (l == n || l == n + 1) {
            const bool second = l == n + 1;
            page1 = second ? pb : pa;
            bytes = b0;
            issue = i0;
            rid = second ? rb : ra;
            m = second ? kWave - k : k;
            lo = second ? k : 0u;
        }
        n += 2;
        ++rows;
        split = true;
    }
    // Appends a linear group's D steps (needs n <= 64 - D).
    template <int D>
    __device__ __forceinline__ void push_group(const GroupLin<D>& gl, std::size_t s,
                                               std::uint32_t r = 0)
    {
        if (n == 0) {
            first = s;
        }
        const int j = static_cast<int>(threadIdx.x) - n;
        // batch lane n + j takes step j from the group's lane j (every lane
        // takes part in the shuffles)
        const int src = j >= 0 && j < D ? j : 0;
        const std::uint32_t p1 =
            static_cast<std::uint32_t>(__shfl(static_cast<int>(gl.page1), src));
        const std::uint64_t i0 = shfl64(gl.issue, src);
        if (j >= 0 && j < D) {
            page1 = p1;
            issue = i0;
            bytes = gl.bytes;
            rid = r;
            m = kWave;
            lo = 0;
        }
        n += D;
        rows += D;
    }
    __device__ __forceinline__ void clear()
    {
        n = 0;
        rows = 0;
        split = false;
    }
    __device__ __forceinline__ std::uint32_t len() const { return kRuns ? m : kWave; }
    __device__ __forceinline__ std::uint32_t at() const { return kRuns ? lo : 0u; }
    __device__ __forceinline__ bool any_split() const { return kRuns && split; }
};

template <bool kRuns>
__device__ __forceinline__ LinBatchT<kRuns> empty_batch()
{
    LinBatchT<kRuns> b;
    b.page1 = 0;
    b.bytes = 0;
    b.issue = 0;
    b.rid = 0;
    b.m = kWave;
    b.lo = 0;
    b.first = 0;
    b.n = 0;
    b.rows = 0;
    b.split = false;
    return b;
}

// Lane grouping by key for one step: the previous lane of the same key
// (pred, -1 for the first), and the group's first and last lanes.  When every
// active lane has the same key (sequential streams) the ballot match is
// skipped.
struct Group {
    int pred, leader, last;
    bool uniform;         // every active lane has the same key (wave-uniform)
    std::uint64_t peers;  // the group's lanes (group_by only)
};

// Lanes whose key equals this lane's key, through a per-wave LDS table of
// lane masks (tab[key] is 0 between calls): every lane ORs its bit into its
// key's slot, reads the slot back, and clears it.  A wave's LDS operations
// complete in issue order, so each read sees every lane's bit and each clear
// follows every read.  Every lane of the wave must call it.
__device__ __forceinline__ std::uint64_t match_lds(std::uint64_t* tab, std::uint32_t key, bool m,
                                                   int lane)
{
    std::uint64_t peers = 0;
    if (m) {
        __hip_atomic_fetch_or(&tab[key], 1ull << lane, __ATOMIC_RELAXED,
                              __HIP_MEMORY_SCOPE_WORKGROUP);
    }
    if (m) {
        peers = __hip_atomic_load(&tab[key], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
    }
    if (m) {
        __hip_atomic_store(&tab[key], 0ull, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
    }
    return peers;
}

__device__ __forceinline__ Group group_by(std::uint32_t key, std::uint32_t bits, bool m,
                                          std::uint64_t active, int lane,
                                          std::uint64_t* tab = nullptr)
{
    const int first = __ffsll(static_cast<long long>(active)) - 1;
    const std::uint32_t key0 =
        static_cast<std::uint32_t>(__builtin_amdgcn_readlane(static_cast<int>(key), first));
    Group g;
    std::uint64_t peers;
    g.uniform = __ballot(m && key == key0) == active;
    if (g.uniform) {
        peers = active;
    } else if (tab != nullptr) {
        peers = match_lds(tab, key, m, lane);
    } else {
        peers = match_key(key, bits, active);
    }
    const std::uint64_t below = peers & lanemask_lt(lane);
    g.pred = (m && below) ? 63 - __clzll(below) : -1;
    g.leader = m ? __ffsll(static_cast<long long>(peers)) - 1 : lane;
    g.last = m ? 63 - __clzll(peers) : lane;
    g.peers = peers;
    return g;
}

// General steps whose records all move the same byte count (the usual case).
// The services of a group of lanes are then counts times constants, so a
// lane's sums over the group's lanes before or after it are population counts
// of the group's mask, not scans:
//   miss, prog   lanes whose record senses (a read that misses) or programs.
// What is left to scan is a maximum.  (Scans of (A, B) pairs by pointer
// jumping, six LDS shuffles a round for the two chains, were 40% of the
// summary pass on random records.)
struct StepCounts {
    std::uint64_t miss, prog;
};

__device__ __forceinline__ StepCounts count_services(bool counts, std::uint32_t bits, bool hit)
{
    StepCounts c;
    c.miss = __ballot(counts && (bits & 1u) == 0 && !hit);
    c.prog = __ballot(counts && (bits & 2u) != 0);
    return c;
}

// Service of the group's lanes in `lanes`.
__device__ __forceinline__ std::uint64_t count_service(const KArgs& a, const StepCounts& c,
                                                       std::uint64_t lanes)
{
    std::uint64_t s =
        static_cast<std::uint64_t>(static_cast<std::uint32_t>(__popcll(lanes & c.miss))) *
        a.read_ps;
    if (c.prog != 0) {
        s += static_cast<std::uint64_t>(static_cast<std::uint32_t>(__popcll(lanes & c.prog))) *
             a.program_ps;
    }
    return s;
}

// Prefix maxima of v1 and v2 along two lane groups, by pointer jumping (a
// chain that is not wanted is passed pred -1 in every lane).
__device__ __forceinline__ void group_prefix_max(std::uint32_t& v1, int p1, std::uint32_t& v2,
                                                 int p2, int lane)
{
    for (int s = 0; s < 6; ++s) {
        const bool any1 = __ballot(p1 >= 0) != 0, any2 = __ballot(p2 >= 0) != 0;
        if (!any1 && !any2) {
            break;
        }
        if (any1) {
            const int s1 = p1 < 0 ? lane : p1;
            const std::uint32_t x =
                static_cast<std::uint32_t>(__shfl(static_cast<int>(v1), s1));
            const int q = __shfl(p1, s1);
            v1 = p1 >= 0 && x > v1 ? x : v1;
            p1 = p1 >= 0 ? q : p1;
        }
        if (any2) {
            const int s2 = p2 < 0 ? lane : p2;
            const std::uint32_t x =
                static_cast<std::uint32_t>(__shfl(static_cast<int>(v2), s2));
            const int q = __shfl(p2, s2);
            v2 = p2 >= 0 && x > v2 ? x : v2;
            p2 = p2 >= 0 ? q : p2;
        }
    }
}

__device__ __forceinline__ void lds_add(std::uint64_t* p, std::uint64_t v)
{
    (void)__hip_atomic_fetch_add(p, v, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
}

__device__ __forceinline__ void lds_max(std::uint64_t* p, std::uint64_t v)
{
    (void)__hip_atomic_fetch_max(p, v, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
}

// Plane grouping of a batch of linear steps (lane k: step k, active lanes a
// prefix).  Steps on one media page share a plane.  Striping maps the page
// modulo C W D P = Rp one-to-one onto the planes (mixed-radix digits), so
// when the batch's pages never fall from lane to lane and span fewer than Rp
// pages, the runs of equal page are exactly the plane groups: one shuffle and
// two ballots instead of a ballot per key bit.  Otherwise, by key.
__device__ __forceinline__ Group group_plane_runs(const KArgs& a, std::uint32_t page1,
                                                  std::uint32_t key, bool m,
                                                  std::uint64_t active, int lane,
                                                  std::uint64_t* tab)
{
    const std::uint32_t prev =
        static_cast<std::uint32_t>(__shfl(static_cast<int>(page1), lane > 0 ? lane - 1 : 0));
    const int last_lane = 63 - __clzll(active);
    const std::uint32_t p0 = rfl32(page1);
    const std::uint32_t pl = rl32(page1, last_lane);
    const bool falls = m && lane > 0 && prev > page1;
    if (__ballot(falls) != 0 || pl - p0 >= a.Rp) {
        return group_by(key, a.pbits, m, active, lane, tab);
    }
    const bool head = m && (lane == 0 || prev != page1);
    const std::uint64_t heads = __ballot(head);
    const std::uint64_t upto = lane == 63 ? ~0ull : ((2ull << lane) - 1);
    const std::uint64_t later = heads & ~upto;
    Group g;
    g.peers = 0;
    g.uniform = heads == 1ull;
    g.pred = (m && !head) ? lane - 1 : -1;
    g.leader = m ? 63 - __clzll(heads & upto) : lane;
    g.last = m ? (later != 0 ? __ffsll(static_cast<long long>(later)) - 2 : last_lane) : lane;
    return g;
}

__device__ __forceinline__ void scan_group(const Group& g, std::uint64_t& A, std::uint64_t& B,
                                           int lane)
{
    if (g.uniform) {
        wave_scan(A, B);
    } else {
        group_scan(A, B, g.pred, lane);
    }
}

// Scans a step's plane maps and channel maps.  When the narrow check passes
// both run in 32 bits relative to the step's time origin: as interleaved DPP
// scans when both are single-key steps, else as interleaved pointer-jumping
// group scans.  Otherwise each runs exactly in 64 bits.
__device__ __forceinline__ void scan_pair(const Group& gp, std::uint64_t& Ap, std::uint64_t& Bp,
                                          const Group& gc, std::uint64_t& Ac, std::uint64_t& Bc,
                                          const Dec& d, bool m, std::uint64_t active,
                                          std::uint64_t svc, std::uint64_t xfer, int lane)
{
    const Narrow nw = narrow_check(d, m, active, svc, xfer);
    if (nw.ok) {
        std::uint32_t ap = static_cast<std::uint32_t>(Ap);
        std::uint32_t bp = Bp == 0 ? 0u : static_cast<std::uint32_t>(Bp - nw.origin);
        std::uint32_t ac = static_cast<std::uint32_t>(Ac);
        std::uint32_t bc = Bc == 0 ? 0u : static_cast<std::uint32_t>(Bc - nw.origin);
        if (gp.uniform && gc.uniform) {
            wave_scan32x2(ap, bp, ac, bc);
        } else {
            group_scan32x2(ap, bp, gp.pred, ac, bc, gc.pred, lane);
        }
        Ap = ap;
        Bp = nw.origin + bp;
        Ac = ac;
        Bc = nw.origin + bc;
        return;
    }
    scan_group(gp, Ap, Bp, lane);
    scan_group(gc, Ac, Bc, lane);
}

__device__ __forceinline__ std::uint64_t plane_service(const KArgs& a, std::uint32_t bits,
                                                       bool hit)
{
    if ((bits & 1u) == 0) {
        return hit ? 0ull : a.read_ps;
    }
    if (bits & 4u) {
        return a.read_ps + a.program_ps;
    }
    return (bits & 2u) ? a.program_ps : 0ull;
}

// The range table in LDS (a.r_lds): at most kLdsRanges ranges, two per lane,
// loaded and stored in two halves as the fences are.
constexpr std::uint32_t kLdsRanges = 128;
constexpr int kRangesPerLane = static_cast<int>(kLdsRanges) / kWave;

struct RangeRegs {
    std::uint64_t len[kRangesPerLane], off[kRangesPerLane];
    std::uint32_t meta[kRangesPerLane], id[kRangesPerLane];
};

__host__ __device__ __forceinline__ std::size_t range_lds_bytes(const KArgs& a)
{
    return a.r_lds != 0 ? 8ull * a.r_count + (a.hybrid != 0 ? 8ull : 4ull) * a.r_count : 0ull;
}

__device__ __forceinline__ RangeRegs fetch_ranges(const KArgs& a, int lane)
{
    RangeRegs r{};
    if (a.r_lds != 0) {
#pragma unroll
        for (int k = 0; k < kRangesPerLane; ++k) {
            const std::uint32_t j = static_cast<std::uint32_t>(k * kWave + lane);
            if (j < a.r_count) {
                r.len[k] = a.r_length[j];
                r.off[k] = a.r_file_offset[j];
                r.meta[k] = a.r_meta[j];
                r.id[k] = a.hybrid != 0 ? a.r_id[j] : 0u;
            }
        }
    }
    return r;
}

// Writes the table at `at` (8-byte aligned) and completes the view.
__device__ __forceinline__ void store_ranges(const KArgs& a, const RangeRegs& r, void* at,
                                             RangeView& rv, int lane)
{
    if (a.r_lds == 0) {
        return;
    }
    auto* len = static_cast<std::uint64_t*>(at);
    auto* page0 = reinterpret_cast<std::uint32_t*>(len + a.r_count);
    auto* id = page0 + a.r_count;
    rv.len = len;
    rv.page0 = page0;
    rv.id = id;
#pragma unroll
    for (int k = 0; k < kRangesPerLane; ++k) {
        const std::uint32_t j = static_cast<std::uint32_t>(k * kWave + lane);
        if (j < a.r_count) {
            len[j] = r.len[k] | (static_cast<std::uint64_t>(r.meta[k] & 0xfu) << 56) |
                     (static_cast<std::uint64_t>((r.meta[k] >> 8) & 0xfu) << 60);
            page0[j] = static_cast<std::uint32_t>(r.off[k] >> a.page_shift);
            if (a.hybrid != 0) {
                id[j] = r.id[k];
            }
        }
    }
}

// The range fences (r_nfence <= kMaxFences), a lane's share in registers:
// fetch_fences issues every load before store_fences writes any of them, so
// a tile's set-up waits for memory once rather than once per 64 fences.
constexpr int kFencesPerLane = static_cast<int>(kMaxFences) / kWave;

struct FenceRegs {
    std::uint64_t v[kFencesPerLane];
};

__device__ __forceinline__ FenceRegs fetch_fences(const KArgs& a, int lane)
{
    FenceRegs f;
#pragma unroll
    for (int k = 0; k < kFencesPerLane; ++k) {
        const std::uint32_t j = static_cast<std::uint32_t>(lane + k * kWave);
        f.v[k] = j < a.r_nfence ? a.r_base[static_cast<std::size_t>(j) * a.r_stride] : 0ull;
    }
    return f;
}

__device__ __forceinline__ void store_fences(const KArgs& a, const FenceRegs& f,
                                             std::uint64_t* fence, int lane)
{
#pragma unroll
    for (int k = 0; k < kFencesPerLane; ++k) {
        const std::uint32_t j = static_cast<std::uint32_t>(lane + k * kWave);
        if (j < a.r_nfence) {
            fence[j] = f.v[k];
        }
    }
}

__device__ __forceinline__ void load_fences(const KArgs& a, std::uint64_t* fence, int lane)
{
    store_fences(a, fetch_fences(a, lane), fence, lane);
}

// Step view of a batch of linear steps: lane k < n stands for step k, with
// lane 0's record of that step (plane and channel from the media page, the
// byte count the channel moves per record and its transfer time).
struct StepView {
    Dec d;
    bool m;
    std::uint64_t active;
    std::uint64_t x;  // transfer of one record
};

template <bool kR>
__device__ __forceinline__ StepView step_view(const KArgs& a, const std::uint64_t* xp,
                                              const LinBatchT<kR>& q, int lane)
{
    StepView v;
    v.m = lane < q.n;
    v.active = q.n == kWave ? ~0ull : ((1ull << q.n) - 1);
    v.d.cls = v.m ? kClsModeled : kClsInvalid;
    v.d.bits = 0;
    v.d.plane = 0;
    v.d.chan = 0;
    v.d.range_id = 0;
    v.d.page1 = q.page1;
    v.d.issue = q.issue;
    v.d.xbytes = a.transfer_page ? (1ull << a.page_shift) : q.bytes;
    v.d.xfer = 0;
    if (v.m) {
        stripe(a, static_cast<std::uint64_t>(q.page1) - 1, v.d);
    }
    v.x = v.m ? xfer_ps_lds(a, xp, v.d.xbytes) : 0ull;
    return v;
}

// The summary pass keeps its per-plane LDS state at slot pslot(plane) =
// plane ^ ((plane >> 5) & 31), a permutation within each aligned block of 32
// planes (the arrays are padded to whole blocks, plane_slots).  A batch of
// linear steps walks the striping's fastest axis: its planes lie 32 apart on
// the 16 x 8 x 4 geometry (8 apart on 8 x 4 x 2), so plain indexing puts every
// lane of a fold on one LDS bank; the swizzle spreads them over distinct ones.
__host__ __device__ __forceinline__ std::uint32_t plane_slots(const KArgs& a)
{
    return (a.Rp + 31u) & ~31u;
}
__device__ __forceinline__ std::uint32_t pslot(std::uint32_t plane)
{
    return plane ^ ((plane >> 5) & 31u);
}

// Issue order across a batch of linear steps (one issue time per step):
// every step's time must be at least the one before it, the first step's at
// least `last` (the last issue time the wave saw before the batch).
template <bool kR>
__device__ __forceinline__ void batch_order(const LinBatchT<kR>& q, int lane, std::uint64_t& last,
                                            bool& back)
{
    const std::uint64_t prev = shfl64(q.issue, lane == 0 ? 0 : lane - 1);
    back = back || __ballot(lane < q.n && q.issue < (lane == 0 ? last : prev)) != 0;
    last = readlane64(q.issue, q.n - 1);
}

// Folds a batch of linear runs into the tile summary: the per-record fold of
// the general path applied to whole runs.  A run of m records after another
// record of its plane has plane map (sense, issue + sense) -- its first record
// senses unless its page is the one the plane last read, the others hit; a
// run that holds the tile's first record on its plane records that record
// and folds the m - 1 hits after it, map (0, issue) (the identity for m = 1).
// The channel map of a run is (m x, issue + m x).  kGiven: page-register
// hits come per record from `hits` (two page registers): a run's first record
// hits as hits[] says, and a run that holds the tile's first record on its
// plane records that hit in its class (bit 3), as the
// per-record path does.
// Stream position of the first record of lane r's run.
template <bool kR>
__device__ __forceinline__ std::size_t run_record(const LinBatchT<kR>& q, int lane)
{
    int row = lane;
    std::uint32_t at = 0;
    if constexpr (kR) {
        const std::uint64_t heads = __ballot(lane < q.n && q.lo == 0);
        row = __popcll(heads & (lanemask_lt(lane) | (1ull << lane))) - 1;
        at = q.lo;
    }
    return q.first + static_cast<std::size_t>(row) * kWave + at;
}

template <bool kR, bool kGiven = false>
__device__ __forceinline__ void fold_summary(const KArgs& a, const std::uint64_t* xp,
                                             const LinBatchT<kR>& q, int lane, std::uint64_t* p_fi,
                                             std::uint64_t* p_rA, std::uint64_t* p_rB,
                                             std::uint64_t* c_A, std::uint64_t* c_B,
                                             std::uint32_t* p_f1, std::uint32_t* p_l1,
                                             std::uint8_t* p_fc, std::uint64_t* mt_p,
                                             std::uint64_t* mt_c,
                                             const std::uint8_t* hits = nullptr)
{
    const StepView v = step_view(a, xp, q, lane);
    const bool m = v.m;
    const std::uint32_t pkey = m ? v.d.plane : 0u;
    const std::uint32_t ckey = m ? v.d.chan : 0u;
    const Group gp = group_plane_runs(a, q.page1, pkey, m, v.active, lane, mt_p);
    const Group gc = group_by(ckey, a.cbits, m, v.active, lane, mt_c);
    const std::uint32_t pk = pslot(pkey);
    const std::uint32_t f1 = m ? p_f1[pk] : 0u;
    const std::uint32_t last_page = m ? p_l1[pk] : 0u;
    const bool has = f1 != 0;
    const bool tfirst = m && gp.pred < 0 && !has;
    std::uint32_t prev1 = static_cast<std::uint32_t>(
        __shfl(static_cast<int>(q.page1), gp.pred < 0 ? lane : gp.pred));
    if (gp.pred < 0) {
        prev1 = last_page;
    }
    bool hit0 = prev1 == q.page1;
    if constexpr (kGiven) {
        const std::size_t at = run_record(q, lane);
        hit0 = m && hits[at] != 0;
    }
    const std::uint64_t ls = hit0 ? 0ull : a.read_ps;
    const std::uint64_t cx = q.len() * v.x;
    std::uint64_t Ap = 0, Bp = 0, Ac = 0, Bc = 0;
    if (m) {
        // a run that holds the tile's first record on its plane records that
        // one apart; the map of the run's others is (0, issue), the identity
        // when it has none
        Ap = tfirst ? 0ull : ls;
        Bp = tfirst ? (q.len() >= 2 ? q.issue : 0ull) : q.issue + ls;
        Ac = cx;
        Bc = q.issue + cx;
    }
    scan_pair(gp, Ap, Bp, gc, Ac, Bc, v.d, m, v.active, ls, cx, lane);
    const std::uint32_t l1 =
        static_cast<std::uint32_t>(__shfl(static_cast<int>(q.page1), gp.leader));
    const std::uint64_t li = shfl64(q.issue, gp.leader);
    std::uint32_t lc = 0;  // the leader's class: a read (bit 3: its given hit)
    if constexpr (kGiven) {
        lc = static_cast<std::uint32_t>(__shfl(hit0 ? 8 : 0, gp.leader));
    }
    if (m && lane == gp.last) {
        if (!has) {
            p_f1[pk] = l1;
            p_fi[pk] = li;
            p_fc[pk] = static_cast<std::uint8_t>(lc);
        }
        const std::uint64_t sA = p_rA[pk];
        const std::uint64_t sB = p_rB[pk];
        p_rB[pk] = umax64(sB + Ap, Bp);
        p_rA[pk] = sA + Ap;
        p_l1[pk] = q.page1;
    }
    if (m && lane == gc.last) {
        const std::uint64_t sA = c_A[ckey];
        const std::uint64_t sB = c_B[ckey];
        c_B[ckey] = umax64(sB + Ac, Bc);
        c_A[ckey] = sA + Ac;
    }
}

// Writes a folded batch's step descriptors.  The summary pass calls it just
// before issuing a group's loads: vector memory operations complete in
// issue order, so a store placed after a group's loads would hold up the
// wait for that group.
template <bool kR>
__device__ __forceinline__ void write_descs(StepDesc* desc, SplitDesc* split, std::uint32_t* rid,
                                            LinBatchT<kR>& dq, int lane)
{
    if (dq.n != 0 && desc != nullptr) {
        // one descriptor per step, written by its first run's lane; a split
        // step's second run is the next lane
        // (32-byte batches hold whole steps only: row = lane, no second runs)
        const bool head = lane < dq.n && dq.at() == 0;
        const int row = kR ? __popcll(__ballot(head) & lanemask_lt(lane)) : lane;
        const int nx = lane + 1 < kWave ? lane + 1 : lane;
        std::uint32_t nlo = 0, np1 = 0, nrid = 0;
        if constexpr (kR) {
            nlo = static_cast<std::uint32_t>(__shfl(static_cast<int>(dq.at()), nx));
            np1 = static_cast<std::uint32_t>(__shfl(static_cast<int>(dq.page1), nx));
            nrid = static_cast<std::uint32_t>(__shfl(static_cast<int>(dq.rid), nx));
        }
        const bool second = kR && head && lane + 1 < dq.n && nlo != 0;
        if (head) {
            const std::size_t at = dq.first / kWave + static_cast<std::size_t>(row);
            StepDesc sd;
            sd.page1 = dq.page1;
            sd.bytes = dq.bytes | (second ? kSplitFlag : 0u);
            sd.issue = dq.issue;
            if (second && split == nullptr) {
                sd = StepDesc{0, 0, 0};  // no side array: replayed from its records
            }
            desc[at] = sd;
            if (second && split != nullptr) {
                split[at] = SplitDesc{np1, nlo, nrid, 0u};
            }
            if (rid != nullptr) {
                rid[at] = dq.rid;
            }
        }
    }
    dq.clear();
}

// 64-bit words of a tile's touched-plane mask.
__host__ __device__ __forceinline__ std::uint32_t mask_words(const KArgs& a)
{
    return (a.Rp + 63) / 64;
}

// A tile's plane summaries are packed: word w of its mask holds the touched
// planes r in [64 w, 64 w + 64) and how many touched planes come before them.
struct alignas(16) MaskWord {
    std::uint64_t bits;
    std::uint32_t base;
    std::uint32_t pad;
};

// Where plane r's entry sits among tile `tile`'s packed summaries (and carry-
// ins), or -1 when the tile does not touch the plane.
__device__ __forceinline__ int slot(const MaskWord* tmask, std::uint32_t words, std::size_t tile,
                                    std::uint32_t r)
{
    const MaskWord m = tmask[tile * words + r / 64];
    const std::uint32_t bit = r % 64;
    if (((m.bits >> bit) & 1u) == 0) {
        return -1;
    }
    return static_cast<int>(m.base) + __popcll(m.bits & ((1ull << bit) - 1));
}

// Byte offset of the summary pass's lane-matching tables (plane table, then
// channel table) after its state: fences, three 64-bit and two 32-bit plane
// arrays, two 64-bit channel arrays and the plane class bytes; 8-byte aligned.
__host__ __device__ __forceinline__ std::size_t summary_match_offset(const KArgs& a)
{
    const std::uint64_t rp = plane_slots(a);
    return 8ull * (a.r_nfence + 3ull * rp + 2ull * a.Rc) + 8ull * rp + ((rp + 7ull) & ~7ull);
}

// Byte offset of the summary pass's stripe table (Rp words), after the
// lane-matching tables when the run keeps them.
__host__ __device__ __forceinline__ std::size_t summary_stripe_offset(const KArgs& a)
{
    return summary_match_offset(a) + (a.match_lds ? 8ull * (a.Rp + a.Rc) : 0ull);
}
__host__ __device__ __forceinline__ std::size_t summary_range_offset(const KArgs& a)
{
    return (summary_stripe_offset(a) + (a.stripe_lds ? 4ull * a.Rp : 0ull) + 7ull) & ~7ull;
}

// Summary pass.  Per plane the tile keeps: the first record (page, issue,
// class), the (max,+) map of the records after it, and the last page; per
// channel the map of all its records.  Pages are stored as page + 1 in 32
// bits (capacity / page_bytes < 2^32 is checked on the host).
template <bool kRefresh, bool kHits, bool kPacked = false, bool kDeep = false, bool kFew = false>
__global__ __launch_bounds__(64) __attribute__((amdgpu_waves_per_eu(kPacked ? (kDeep ? 2 : (kFew ? 3 : 4)) : 1))) void k_summary(KArgs a, const void* rec, std::size_t n,
                                                std::uint64_t base_ps, PlaneSum* psum,
                                                MaskWord* tmask, ChanSum* csum,
                                                std::uint64_t* tile_count,
                                                const std::uint8_t* hits, StepDesc* desc)
{
    extern __shared__ std::uint64_t sm[];
    constexpr bool kRuns = !kRefresh;  // batches hold runs: steps may be split
    // per-plane state at slot pslot(plane) of plane_slots(a) entries
    const std::uint32_t rpp = plane_slots(a);
    RangeView fence(sm);
    std::uint64_t* p_fi = sm + a.r_nfence;
    std::uint64_t* p_rA = p_fi + rpp;
    std::uint64_t* p_rB = p_rA + rpp;
    std::uint64_t* c_A = p_rB + rpp;
    std::uint64_t* c_B = c_A + a.Rc;
    std::uint32_t* p_f1 = reinterpret_cast<std::uint32_t*>(c_B + a.Rc);
    std::uint32_t* p_l1 = p_f1 + rpp;
    std::uint8_t* p_fc = reinterpret_cast<std::uint8_t*>(p_l1 + rpp);  // class bits < 16
    std::uint64_t* mt_p = a.match_lds ? reinterpret_cast<std::uint64_t*>(
                                            reinterpret_cast<unsigned char*>(sm) +
                                            summary_match_offset(a))
                                      : nullptr;
    std::uint64_t* mt_c = a.match_lds ? mt_p + a.Rp : nullptr;
    __shared__ std::uint64_t xp[33];
    const int lane = threadIdx.x;
    const std::size_t tile = blockIdx.x;
    const std::size_t begin = tile * a.tile;
    const std::size_t end = begin + a.tile < n ? begin + a.tile : n;
    if (a.mixed != 0 && a.tile_split[tile] == kTilePlain) {
        return;  // k_plain_summary took it
    }
    if (a.mixed == 0) {
        stamp_start(a, 0);
    }
    // set-up loads and the first group of records are in flight together
    const FenceRegs fr = fetch_fences(a, lane);
    const RangeRegs rr = fetch_ranges(a, lane);
    const std::uint64_t xv = fetch_xfer(a, lane);
    // The record before the tile: every record's issue time must be at least
    // its predecessor's for stream position to be the service order.  Steps
    // check their records against the last issue time seen (wave-uniform);
    // any that goes back sets a.disorder.
    std::uint64_t last_issue = 0;
    if (begin > 0) {
        last_issue = base_ps + (kPacked ? (static_cast<const hbf_record16*>(rec)[begin - 1].issue_op &
                                           ((1ull << 56) - 1))
                                        : static_cast<const hbf_record32*>(rec)[begin - 1].issue_ps);
    }
    bool disorder = false;
    bool any_split = false;  // some step of the tile was split (wave-uniform)
    // (packed records keep kPackedSumPipe steps at four waves per SIMD)
    // (kDeep: packed records where LDS already holds the pass at two waves
    // per SIMD, whose registers then allow 2 * kSumPipe steps in flight)
    constexpr int kDepth =
        (kDeep ? 2 * kSumPipe : (kPacked && !kFew ? kPackedSumPipe : kSumPipe));
    constexpr std::size_t kSpan = static_cast<std::size_t>(kDepth) * kWave;
    using Pipe = std::conditional_t<kPacked, PackedPipeT<kDepth>, RecordPipeT<kDepth>>;
    Pipe pipe;
    pipe.issue(rec, begin, end, lane);
    store_fences(a, fr, sm, lane);
    store_ranges(a, rr, reinterpret_cast<unsigned char*>(sm) + summary_range_offset(a), fence,
                 lane);
    store_xfer(xp, xv, lane);
    for (std::uint32_t r = lane; r < rpp; r += kWave) {
        p_fi[r] = 0;
        p_rA[r] = 0;
        p_rB[r] = 0;
        p_f1[r] = 0;
        p_l1[r] = 0;
        p_fc[r] = 0;
    }
    for (std::uint32_t r = lane; r < a.Rc; r += kWave) {
        c_A[r] = 0;
        c_B[r] = 0;
    }
    if (a.match_lds) {
        for (std::uint32_t r = lane; r < a.Rp + a.Rc; r += kWave) {
            mt_p[r] = 0;
        }
    }
    std::uint32_t* stab = nullptr;
    if (a.stripe_lds) {
        stab = reinterpret_cast<std::uint32_t*>(reinterpret_cast<unsigned char*>(sm) +
                                                summary_stripe_offset(a));
        fill_stripe_table(a, stab, lane);
    }
    __syncthreads();
    RangeCache rc = empty_cache();
    RangeCache rcu = empty_cache();  // wave-uniform copy for linear steps
    LinBatchT<kRuns> q = empty_batch<kRuns>();
    LinBatchT<kRuns> dq = empty_batch<kRuns>();  // folded, descriptors not written yet
    // a batch is folded once it holds kFull runs: two lanes stay free for a
    // split step's runs
    constexpr int kFull = kRuns ? kWave - 1 : kWave;
    std::uint64_t modeled = 0;
    std::uint32_t lin_miss = 0;  // steps in a row that were not linear (wave-uniform)
    // descriptors of steps replayed from their records are zeroed up to 64
    // at a time, one lane per step: steps zbase + l for the bits l of zmask
    std::size_t zbase = 0;
    std::uint64_t zmask = 0;
    const auto flush_zero = [&]() {
        if (((zmask >> lane) & 1u) != 0) {
            desc[zbase + lane] = StepDesc{0, 0, 0};
        }
        zmask = 0;
    };
    for (std::size_t g = begin; g < end; g += kSpan) {
        pipe.promote();
        write_descs(desc, a.desc_split, a.desc_rid, dq, lane);
        if (g + kSpan < end) {
            pipe.issue(rec, g + kSpan, end, lane);
        }
        const std::size_t gend = g + kSpan < end ? g + kSpan : end;
        if ((kHits || a.slots == 1) && a.lead == nullptr && g + kSpan <= end &&
            q.n <= kWave - kDepth && lin_miss < kLinGiveUp) {
            // a whole group of linear steps joins the batch at once
            GroupLin<kDepth> gl;
            if (group_linear<kRefresh>(a, fence, rcu, pipe, base_ps, lane, gl)) {
                q.push_group(gl, g, rcu.id);
                if (q.n >= kFull || gend >= end) {
                    batch_order(q, lane, last_issue, disorder);
                    fold_summary<kRuns, kHits>(a, xp, q, lane, p_fi, p_rA, p_rB, c_A, c_B,
                                                 p_f1, p_l1, p_fc, mt_p, mt_c, hits);
                    modeled += static_cast<std::uint64_t>(q.rows) * kWave;
                    dq = q;  // (its descriptors wait for the next group's loads)
                    q.clear();
                }
                continue;
            }
        }
        for (std::size_t s = g; s < gend; s += kWave) {
            typename Pipe::Step st;
            pipe.take(st);
            const std::size_t i = s + lane;
            const bool valid = i < end;
            if ((kHits || a.slots == 1) && a.lead == nullptr) {
                // linear steps wait in a batch; the batch is folded when full, at
                // the tile's last step, and before any other step (order matters)
                LinStep ls;
                bool lin = false;
                if (lin_miss < kLinGiveUp || (s / kWave) % kLinProbe == 0) {
                    lin = detect_step<kRefresh, kRuns>(a, fence, rcu, st, base_ps, s + kWave <= end,
                                                lane, ls);
                    lin_miss = lin ? 0u : lin_miss + 1u;
                }
                if (lin) {
                    if (!kRuns || ls.k == 0) {
                        q.push(ls.page1, ls.issue, ls.bytes, s, ls.rid);
                    } else if constexpr (kRuns) {
                        q.push_split(ls.page1, ls.page1b, ls.k, ls.issue, ls.bytes, s, ls.rid,
                                     ls.ridb);
                        any_split = true;
                    }
                }
                if (q.n != 0 && (!lin || q.n >= kFull || s + kWave >= end)) {
                    batch_order(q, lane, last_issue, disorder);
                    fold_summary<kRuns, kHits>(a, xp, q, lane, p_fi, p_rA, p_rB, c_A, c_B,
                                                 p_f1, p_l1, p_fc, mt_p, mt_c, hits);
                    modeled += static_cast<std::uint64_t>(q.rows) * kWave;
                    write_descs(desc, a.desc_split, a.desc_rid, dq, lane);  // at most one waits
                    dq = q;
                    q.clear();
                }
                if (lin) {
                    continue;
                }
                if (desc != nullptr) {  // replayed from its records
                    const std::size_t step = s / kWave;
                    if (zmask != 0 && step - zbase >= static_cast<std::size_t>(kWave)) {
                        flush_zero();
                    }
                    if (zmask == 0) {
                        zbase = step;
                    }
                    zmask |= 1ull << (step - zbase);
                }
            }
            uint4 x, y;
            step_records(st, lane, x, y);
            Dec d = valid ? decode<kRefresh>(a, fence, rc, x, y, base_ps, stab) : invalid_dec();
            {
                const std::uint64_t prev = prev_lane64(d.issue);
                const bool back = valid && d.issue < (lane == 0 ? last_issue : prev);
                disorder = disorder || __ballot(back) != 0;
                const std::uint64_t vmask = __ballot(valid);  // lanes 0 .. k
                last_issue = readlane64(d.issue, 63 - __clzll(static_cast<long long>(vmask)));
            }
            if (!kPacked && a.lead != nullptr && valid && a.lead[i] != 0) {
                d.cls = kClsFollower;
            }
            const bool m = valid && d.cls == kClsModeled;
            const bool hbit = kHits && valid && hits[i] != 0;
            const std::uint64_t active = __ballot(m);
            modeled += __popcll(active);
            if (active == 0) {
                continue;
            }
            bool same_x = false;
            const std::uint64_t xfer = lane_xfer(a, xp, d, m, active, same_x);
            if (!kHits && run_step(a, d, active, lane)) {
                const std::uint64_t W = run_channel_max(d, xfer, lane);
                if (lane == 63) {
                    const std::uint32_t pkey = pslot(d.plane);
                    const std::uint32_t ckey = d.chan;
                    const std::uint32_t page1 = static_cast<std::uint32_t>(d.page1);
                    const std::uint64_t i0 = readlane64(d.issue, 0);
                    if (p_f1[pkey] == 0) {  // lane 0 is the tile's first record here
                        p_f1[pkey] = page1;
                        p_fi[pkey] = i0;
                        p_fc[pkey] = 0;
                        p_rA[pkey] = 0;
                        p_rB[pkey] = d.issue;
                    } else {
                        const bool lhit = p_l1[pkey] == page1;
                        const std::uint64_t ls = lhit ? 0ull : a.read_ps;
                        const std::uint64_t sA = p_rA[pkey] + ls;
                        const std::uint64_t sB = umax64(p_rB[pkey] + ls, i0 + ls);
                        p_rA[pkey] = sA;
                        p_rB[pkey] = umax64(sB, d.issue);
                    }
                    p_l1[pkey] = page1;
                    const std::uint64_t tA = 64 * xfer;
                    const std::uint64_t tB = W + xfer;
                    const std::uint64_t sA = c_A[ckey];
                    const std::uint64_t sB = c_B[ckey];
                    c_B[ckey] = umax64(sB + tA, tB);
                    c_A[ckey] = sA + tA;
                }
                continue;
            }
            const std::uint32_t page1 = static_cast<std::uint32_t>(d.page1);
            const std::uint32_t pkey = m ? d.plane : 0u;
            const std::uint32_t ckey = m ? d.chan : 0u;
            const Group gp = group_by(pkey, a.pbits, m, active, lane, mt_p);
            const Group gc = group_by(ckey, a.cbits, m, active, lane, mt_c);
            // state reads come before this step's writes
            const std::uint32_t pk = pslot(pkey);
            const std::uint32_t f1 = m ? p_f1[pk] : 0u;
            const std::uint32_t last_page = m ? p_l1[pk] : 0u;
            const bool has = f1 != 0;
            const bool tfirst = m && gp.pred < 0 && !has;
            std::uint32_t prev1 = static_cast<std::uint32_t>(
                __shfl(static_cast<int>(page1), gp.pred < 0 ? lane : gp.pred));
            if (gp.pred < 0) {
                prev1 = last_page;
            }
            const bool hit = kHits ? (m && hbit) : (a.slots != 0 && m && prev1 == page1);
            // the leader's class; with given hits, bit 3 carries its hit
            const std::uint32_t lbits = kHits && hit ? (d.bits | 8u) : d.bits;
            if (!kRefresh && same_x) {
                // Per group, (A, B) becomes (A + S, max(B + S, issue_k + S_k)
                // over its lanes k), with S the service of all of them and S_k
                // that of lane k and later: the group's last lane adds S, then
                // every lane joins its own term, all by LDS atomics (a wave's
                // LDS operations complete in issue order).
                const StepCounts sc = count_services(m && !tfirst, d.bits, hit);
                const std::uint64_t from = ~lanemask_lt(lane);
                if (tfirst) {
                    p_f1[pk] = page1;
                    p_fi[pk] = d.issue;
                    p_fc[pk] = static_cast<std::uint8_t>(lbits);
                }
                if (m && lane == gp.last) {
                    const std::uint64_t S = count_service(a, sc, gp.peers);
                    lds_add(&p_rA[pk], S);
                    lds_add(&p_rB[pk], S);
                    p_l1[pk] = page1;
                }
                if (m && !tfirst) {
                    lds_max(&p_rB[pk], d.issue + count_service(a, sc, gp.peers & from));
                }
                if (m && lane == gc.last) {
                    const std::uint64_t S =
                        static_cast<std::uint64_t>(
                            static_cast<std::uint32_t>(__popcll(gc.peers))) * xfer;
                    lds_add(&c_A[ckey], S);
                    lds_add(&c_B[ckey], S);
                }
                if (m) {
                    lds_max(&c_B[ckey], d.issue + static_cast<std::uint64_t>(static_cast<std::uint32_t>(
                                                      __popcll(gc.peers & from))) * xfer);
                }
                continue;
            }
            const std::uint64_t svc = plane_service(a, d.bits, hit);
            std::uint64_t Ap = 0, Bp = 0;
            if (m && !tfirst) {
                Ap = svc;
                Bp = d.issue + svc;
            }
            std::uint64_t Ac = m ? xfer : 0ull;
            std::uint64_t Bc = m ? d.issue + xfer : 0ull;
            scan_pair(gp, Ap, Bp, gc, Ac, Bc, d, m, active, svc, xfer, lane);
            const std::uint32_t l1 =
                static_cast<std::uint32_t>(__shfl(static_cast<int>(page1), gp.leader));
            const std::uint64_t li = shfl64(d.issue, gp.leader);
            const std::uint32_t lc =
                static_cast<std::uint32_t>(__shfl(static_cast<int>(lbits), gp.leader));
            if (m && lane == gp.last) {
                if (!has) {
                    p_f1[pk] = l1;
                    p_fi[pk] = li;
                    p_fc[pk] = static_cast<std::uint8_t>(lc);
                }
                const std::uint64_t sA = p_rA[pk];
                const std::uint64_t sB = p_rB[pk];
                p_rB[pk] = umax64(sB + Ap, Bp);
                p_rA[pk] = sA + Ap;
                p_l1[pk] = page1;
            }
            if (m && lane == gc.last) {
                const std::uint64_t sA = c_A[ckey];
                const std::uint64_t sB = c_B[ckey];
                c_B[ckey] = umax64(sB + Ac, Bc);
                c_A[ckey] = sA + Ac;
            }
        }
    }
    write_descs(desc, a.desc_split, a.desc_rid, dq, lane);
    if (desc != nullptr) {
        flush_zero();
    }
    if (disorder && a.disorder != nullptr && lane == 0) {
        *a.disorder = 1u;
    }
    if (kRuns && a.tile_split != nullptr && lane == 0) {
        a.tile_split[tile] = any_split ? 1u : 0u;
    }
    __syncthreads();
    // Only planes the tile touched get a summary, packed in plane order; the
    // tile's mask words say which (the others are identities, and the carry
    // chain skips them).
    PlaneSum* ps = psum + tile * a.Rp;
    MaskWord* tm = tmask + tile * mask_words(a);
    std::uint32_t count = 0;
    for (std::uint32_t r0 = 0; r0 < a.Rp; r0 += kWave) {
        const std::uint32_t r = r0 + lane;
        const std::uint32_t k = pslot(r);
        const bool touched = r < a.Rp && p_f1[k] != 0;
        const std::uint64_t bits = __ballot(touched);
        if (lane == 0) {
            MaskWord m;
            m.bits = bits;
            m.base = count;
            m.pad = 0;
            tm[r0 / kWave] = m;
        }
        if (touched) {
            PlaneSum v;
            v.fpage1 = p_f1[k];
            v.fissue = p_fi[k];
            v.rA = p_rA[k];
            v.rB = p_rB[k];
            v.lpage1 = p_l1[k];
            v.fcls = p_fc[k];
            v.pad = 0;
            ps[count + __popcll(bits & lanemask_lt(lane))] = v;
        }
        count += static_cast<std::uint32_t>(__popcll(bits));
    }
    ChanSum* cs = csum + tile * a.Rc;
    for (std::uint32_t r = lane; r < a.Rc; r += kWave) {
        ChanSum v;
        v.A = c_A[r];
        v.B = c_B[r];
        cs[r] = v;
    }
    if (lane == 0) {
        tile_count[tile] = modeled;
    }
}

__device__ __forceinline__ void add128(std::uint64_t& lo, std::uint64_t& hi, std::uint64_t v)
{
    const std::uint64_t n = lo + v;
    hi += n < lo ? 1u : 0u;
    lo = n;
}

__device__ __forceinline__ std::uint64_t wave_sum(std::uint64_t v)
{
    for (int o = 32; o > 0; o >>= 1) {
        v += shfl64(v, threadIdx.x ^ o);
    }
    return v;
}

// ---- carry chain: a three-level scan over tile summaries ---------------
//
// A plane summary is a (first record, (max,+) map of the rest, last page)
// triple.  Two summaries compose associatively: the later summary's first
// record resolves its page-register hit against the earlier one's last page,
// then joins the map.  Level 1 folds groups of kGroup tiles, level 2 walks
// the groups of each resource in order from the engine state, level 3 walks
// each group's tiles from the group's carry-in.  One thread per (group,
// resource) at levels 1 and 3, one per resource at level 2.

constexpr std::uint32_t kGroup = 16;
constexpr int kChunk = 8;  // loads a carry thread keeps in flight

__device__ __forceinline__ PlaneSum plane_compose(const KArgs& a, const PlaneSum& s1,
                                                  const PlaneSum& s2)
{
    if (s2.fpage1 == 0) {
        return s1;
    }
    if (s1.fpage1 == 0) {
        return s2;
    }
    PlaneSum r = s1;
    const bool hit = a.ext_hits ? (s2.fcls & 8u) != 0 : (a.slots != 0 && s2.fpage1 == s1.lpage1);
    const std::uint64_t svc = plane_service(a, s2.fcls, hit);
    // rest1, then the later first record (svc, issue + svc), then rest2; A
    // is also the service total of the records after the first
    const std::uint64_t A = s1.rA + svc;
    const std::uint64_t B = umax64(s1.rB + svc, s2.fissue + svc);
    r.rB = umax64(B + s2.rA, s2.rB);
    r.rA = A + s2.rA;
    r.lpage1 = s2.lpage1;
    return r;
}

// Applies a summary to a plane's state; returns the service it charged.
__device__ __forceinline__ std::uint64_t plane_apply(const KArgs& a, const PlaneSum& s,
                                                     std::uint64_t& busy, std::uint64_t& tag1)
{
    if (s.fpage1 == 0) {
        return 0;
    }
    const bool hit = a.ext_hits ? (s.fcls & 8u) != 0 : (a.slots != 0 && tag1 == s.fpage1);
    const std::uint64_t svc = plane_service(a, s.fcls, hit);
    if (a.contention) {
        const std::uint64_t b = umax64(busy, s.fissue) + svc;
        busy = umax64(b + s.rA, s.rB);
    }
    tag1 = s.lpage1;
    return svc + s.rA;
}

__device__ __forceinline__ ChanSum chan_compose(const ChanSum& s1, const ChanSum& s2)
{
    ChanSum r;
    r.A = s1.A + s2.A;
    r.B = umax64(s1.B + s2.A, s2.B);
    return r;
}

// Level 1: thread (g, r) folds the summaries of group g's tiles.
// Slots of plane r in tiles t .. t + kChunk - 1 (those below t1; -1 where
// a tile did not touch r).  The chunk's mask words are loaded whole and
// together before any is decoded: decoding each word as it arrives would
// put a memory round trip per tile in front of the summaries' loads.
__device__ __forceinline__ void chunk_slots(const MaskWord* tmask, std::uint32_t words,
                                            std::size_t t, std::size_t t1, std::uint32_t r,
                                            int (&at)[kChunk])
{
    MaskWord mw[kChunk];
#pragma unroll
    for (int k = 0; k < kChunk; ++k) {
        mw[k] = t + k < t1 ? tmask[(t + k) * words + r / 64] : MaskWord{0, 0, 0};
    }
    const std::uint32_t bit = r % 64;
    const std::uint64_t below = (1ull << bit) - 1;
#pragma unroll
    for (int k = 0; k < kChunk; ++k) {
        at[k] = ((mw[k].bits >> bit) & 1u) != 0
                    ? static_cast<int>(mw[k].base) + __popcll(mw[k].bits & below)
                    : -1;
    }
}

// Level-1 work of thread (g, r): the composition of group g's tile
// summaries of plane r, of channel c, and its tiles' modeled-record count.
// Loads go out kChunk at a time ahead of the (serial) composition, so a
// thread waits once per chunk rather than once per tile.
__device__ __forceinline__ PlaneSum plane_fold(const KArgs& a, const PlaneSum* psum,
                                               const MaskWord* tmask, std::size_t ntiles,
                                               std::size_t g, std::uint32_t r)
{
    const std::size_t t0 = g * kGroup;
    const std::size_t t1 = t0 + kGroup < ntiles ? t0 + kGroup : ntiles;
    const std::uint32_t words = mask_words(a);
    PlaneSum acc{};  // the identity: no first record
#pragma unroll
    for (std::uint32_t c = 0; c < kGroup / kChunk; ++c) {
        const std::size_t t = t0 + static_cast<std::size_t>(c) * kChunk;
        if (t >= t1) {
            break;
        }
        int at[kChunk];
        PlaneSum buf[kChunk];
        chunk_slots(tmask, words, t, t1, r, at);
#pragma unroll
        for (int k = 0; k < kChunk; ++k) {
            if (at[k] >= 0) {
                buf[k] = psum[(t + k) * a.Rp + at[k]];
            }
        }
#pragma unroll
        for (int k = 0; k < kChunk; ++k) {
            if (at[k] >= 0) {
                acc = plane_compose(a, acc, buf[k]);
            }
        }
    }
    return acc;
}

__device__ __forceinline__ ChanSum chan_fold(const KArgs& a, const ChanSum* csum,
                                             std::size_t ntiles, std::size_t g, std::uint32_t c)
{
    const std::size_t t0 = g * kGroup;
    const std::size_t t1 = t0 + kGroup < ntiles ? t0 + kGroup : ntiles;
    ChanSum acc{0, 0};  // the identity
    for (std::size_t t = t0; t < t1; t += kChunk) {
        ChanSum buf[kChunk];
#pragma unroll
        for (int k = 0; k < kChunk; ++k) {
            buf[k] = t + k < t1 ? csum[(t + k) * a.Rc + c] : ChanSum{0, 0};
        }
#pragma unroll
        for (int k = 0; k < kChunk; ++k) {
            acc = chan_compose(acc, buf[k]);
        }
    }
    return acc;
}

__device__ __forceinline__ std::uint64_t count_fold(const std::uint64_t* tile_count,
                                                    std::size_t ntiles, std::size_t g)
{
    const std::size_t t0 = g * kGroup;
    const std::size_t t1 = t0 + kGroup < ntiles ? t0 + kGroup : ntiles;
    std::uint64_t sum = 0;
    for (std::size_t t = t0; t < t1; ++t) {
        sum += tile_count[t];
    }
    return sum;
}

__global__ __launch_bounds__(256) void k_carry_up(KArgs a, std::size_t ntiles, std::size_t ngroups,
                                                  const PlaneSum* psum,
                                                  const MaskWord* tmask, const ChanSum* csum,
                                                  const std::uint64_t* tile_count,
                                                  PlaneSum* gpsum, ChanSum* gcsum,
                                                  std::uint64_t* gcount)
{
    const std::uint32_t rt = a.Rp + a.Rc + 1;
    const std::size_t id = static_cast<std::size_t>(blockIdx.x) * blockDim.x + threadIdx.x;
    stamp_start(a, 1);
    if (id >= ngroups * rt) {
        return;
    }
    const std::size_t g = id / rt;
    const std::uint32_t r = static_cast<std::uint32_t>(id - g * rt);
    if (r < a.Rp) {
        gpsum[g * a.Rp + r] = plane_fold(a, psum, tmask, ntiles, g, r);
    } else if (r < a.Rp + a.Rc) {
        const std::uint32_t c = r - a.Rp;
        gcsum[g * a.Rc + c] = chan_fold(a, csum, ntiles, g, c);
    } else {
        gcount[g] = count_fold(tile_count, ntiles, g);
    }
}

// Level 2: block r scans resource r's group summaries (an exclusive scan by
// composition, kMidBlock groups per pass with a running carry) and applies
// each prefix to the engine state: every group's carry-in, the final state,
// and the service total.
constexpr int kMidBlock = 512;
// runs of at most this many tiles take the one-launch chain (k_carry_one)
constexpr std::size_t kOneCarryTiles = static_cast<std::size_t>(kMidBlock) * kChunk;

// one entry per wave of the block: the waves' inclusive totals
union MidShared {
    PlaneSum p[kMidBlock / kWave];
    ChanSum c[kMidBlock / kWave];
    std::uint64_t s[kMidBlock / kWave];
};

// Lane `src`'s value of a scanned type.
__device__ __forceinline__ std::uint64_t lane_value(std::uint64_t v, int src)
{
    return shfl64(v, src);
}

__device__ __forceinline__ ChanSum lane_value(const ChanSum& v, int src)
{
    return ChanSum{shfl64(v.A, src), shfl64(v.B, src)};
}

__device__ __forceinline__ PlaneSum lane_value(const PlaneSum& v, int src)
{
    PlaneSum r;
    r.fpage1 = shfl64(v.fpage1, src);
    r.fissue = shfl64(v.fissue, src);
    r.rA = shfl64(v.rA, src);
    r.rB = shfl64(v.rB, src);
    r.lpage1 = shfl64(v.lpage1, src);
    r.fcls = static_cast<std::uint32_t>(__shfl(static_cast<int>(v.fcls), src));
    r.pad = 0;
    return r;
}

// Inclusive scan of x over the block, earlier elements first: each wave
// scans its lanes through shuffles (Hillis-Steele), then every thread
// composes the totals of the waves before its own from LDS; two barriers in
// all.  `excl` receives the exclusive prefix (identity for thread 0).
template <typename T, typename F>
__device__ __forceinline__ T block_scan(T x, T* wsh, T identity, F compose, T& excl)
{
    const int tid = threadIdx.x;
    const int lane = tid & (kWave - 1);
    const int w = tid / kWave;
    for (int off = 1; off < kWave; off <<= 1) {
        const T y = lane_value(x, lane >= off ? lane - off : lane);
        if (lane >= off) {
            x = compose(y, x);
        }
    }
    T before_lane = lane_value(x, lane > 0 ? lane - 1 : 0);
    if (lane == kWave - 1) {
        wsh[w] = x;
    }
    __syncthreads();
    T before = identity;
    for (int k = 0; k < w; ++k) {
        before = compose(before, wsh[k]);
    }
    __syncthreads();  // (wsh may be written again after the return)
    excl = lane > 0 ? compose(before, before_lane) : before;
    return compose(before, x);
}

__device__ __forceinline__ std::uint64_t block_sum(std::uint64_t v, std::uint64_t* sh)
{
    const std::uint64_t w = wave_sum(v);
    const int tid = threadIdx.x;
    if ((tid & (kWave - 1)) == 0) {
        sh[tid / kWave] = w;
    }
    __syncthreads();
    std::uint64_t total = 0;
    for (int k = 0; k < kMidBlock / kWave; ++k) {
        total += sh[k];
    }
    __syncthreads();
    return total;
}

__global__ __launch_bounds__(kMidBlock) void k_carry_mid(
    KArgs a, std::size_t ngroups, const PlaneSum* gpsum, const ChanSum* gcsum,
    const std::uint64_t* gcount, PlaneCarry* gpcarry, std::uint64_t* gccarry,
    std::uint64_t* gseq, std::uint64_t* st_pbusy, std::uint64_t* st_ptag,
    std::uint64_t* st_cbusy, std::uint64_t* st_seq, std::uint64_t* ptotal, std::uint64_t* ctotal)
{
    __shared__ MidShared sh;
    __shared__ std::uint64_t red[kMidBlock / kWave];
    __shared__ std::uint64_t next[2];
    const std::uint32_t r = blockIdx.x;
    const int tid = threadIdx.x;
    // a stream whose issue time goes back is timed again from a sorted copy:
    // this run then leaves the engine state as it found it
    const bool commit = a.disorder == nullptr || *a.disorder == 0u;
    if (r < a.Rp) {
        std::uint64_t busy = st_pbusy[r];
        std::uint64_t tag1 = st_ptag[static_cast<std::size_t>(r) * 2];
        std::uint64_t total = 0;
        const PlaneSum id{};
        const auto compose = [&](const PlaneSum& s1, const PlaneSum& s2) {
            return plane_compose(a, s1, s2);
        };
        for (std::size_t g0 = 0; g0 < ngroups; g0 += kMidBlock) {
            const std::size_t g = g0 + tid;
            PlaneSum own = id;
            if (g < ngroups) {
                own = gpsum[g * a.Rp + r];
            }
            PlaneSum before;
            (void)block_scan(own, sh.p, id, compose, before);
            std::uint64_t b = busy, t1 = tag1;
            (void)plane_apply(a, before, b, t1);  // the state this group starts from
            std::uint64_t svc = 0;
            if (g < ngroups) {
                PlaneCarry c;
                c.busy = b;
                c.tag1 = t1;
                gpcarry[g * a.Rp + r] = c;
                svc = plane_apply(a, own, b, t1);
            }
            const std::size_t last = (ngroups - g0 < kMidBlock ? ngroups - g0 : kMidBlock) - 1;
            if (static_cast<std::size_t>(tid) == last) {
                next[0] = b;
                next[1] = t1;
            }
            total += block_sum(svc, red);
            busy = next[0];
            tag1 = next[1];
            __syncthreads();
        }
        if (tid == 0 && commit) {
            st_pbusy[r] = busy;
            st_ptag[static_cast<std::size_t>(r) * 2] = tag1;
            ptotal[r] += total;
        }
    } else if (r < a.Rp + a.Rc) {
        const std::uint32_t c = r - a.Rp;
        std::uint64_t busy = st_cbusy[c];
        std::uint64_t total = 0;
        const ChanSum id{0, 0};
        for (std::size_t g0 = 0; g0 < ngroups; g0 += kMidBlock) {
            const std::size_t g = g0 + tid;
            ChanSum own = id;
            if (g < ngroups) {
                own = gcsum[g * a.Rc + c];
            }
            ChanSum before;
            const ChanSum inc = block_scan(own, sh.c, id, chan_compose, before);
            if (g < ngroups) {
                gccarry[g * a.Rc + c] = umax64(busy + before.A, before.B);
            }
            const std::size_t last = (ngroups - g0 < kMidBlock ? ngroups - g0 : kMidBlock) - 1;
            if (static_cast<std::size_t>(tid) == last) {
                next[0] = umax64(busy + inc.A, inc.B);
            }
            total += block_sum(g < ngroups ? own.A : 0ull, red);
            busy = next[0];
            __syncthreads();
        }
        if (tid == 0 && commit) {
            st_cbusy[c] = busy;
            ctotal[c] += total;
        }
    } else if (r == a.Rp + a.Rc) {
        std::uint64_t seq = *st_seq;
        const auto add = [](std::uint64_t x, std::uint64_t y) { return x + y; };
        for (std::size_t g0 = 0; g0 < ngroups; g0 += kMidBlock) {
            const std::size_t g = g0 + tid;
            const std::uint64_t own = g < ngroups ? gcount[g] : 0ull;
            std::uint64_t before;
            const std::uint64_t inc = block_scan(own, sh.s, std::uint64_t{0}, add, before);
            if (g < ngroups) {
                gseq[g] = seq + before;
            }
            const std::size_t last = (ngroups - g0 < kMidBlock ? ngroups - g0 : kMidBlock) - 1;
            if (static_cast<std::size_t>(tid) == last) {
                next[0] = seq + inc;
            }
            __syncthreads();
            seq = next[0];
            __syncthreads();
        }
        if (tid == 0 && commit) {
            *st_seq = seq;
        }
    }
}

// Level-3 work of thread (g, r): walks group g's tiles from the group's
// carry-in and writes every tile's carry-in.
__device__ __forceinline__ void plane_walk(const KArgs& a, const PlaneSum* psum,
                                           const MaskWord* tmask, std::size_t ntiles,
                                           std::size_t g, std::uint32_t r, PlaneCarry c0,
                                           PlaneCarry* pcarry)
{
    const std::size_t t0 = g * kGroup;
    const std::size_t t1 = t0 + kGroup < ntiles ? t0 + kGroup : ntiles;
    const std::uint32_t words = mask_words(a);
    std::uint64_t busy = c0.busy, tag1 = c0.tag1;
#pragma unroll
    for (std::uint32_t c = 0; c < kGroup / kChunk; ++c) {
        const std::size_t t = t0 + static_cast<std::size_t>(c) * kChunk;
        if (t >= t1) {
            break;
        }
        int at[kChunk];
        PlaneSum buf[kChunk];
        chunk_slots(tmask, words, t, t1, r, at);
#pragma unroll
        for (int k = 0; k < kChunk; ++k) {
            if (at[k] >= 0) {
                buf[k] = psum[(t + k) * a.Rp + at[k]];
            }
        }
#pragma unroll
        for (int k = 0; k < kChunk; ++k) {
            // an untouched tile neither reads nor changes this plane
            if (at[k] >= 0) {
                PlaneCarry c;
                c.busy = busy;
                c.tag1 = tag1;
                pcarry[(t + k) * a.Rp + at[k]] = c;  // packed like the summaries
                (void)plane_apply(a, buf[k], busy, tag1);
            }
        }
    }
}

__device__ __forceinline__ void chan_walk(const KArgs& a, const ChanSum* csum, std::size_t ntiles,
                                          std::size_t g, std::uint32_t c, std::uint64_t busy,
                                          std::uint64_t* ccarry)
{
    const std::size_t t0 = g * kGroup;
    const std::size_t t1 = t0 + kGroup < ntiles ? t0 + kGroup : ntiles;
    for (std::size_t t = t0; t < t1; t += kChunk) {
        ChanSum buf[kChunk];
#pragma unroll
        for (int k = 0; k < kChunk; ++k) {
            buf[k] = t + k < t1 ? csum[(t + k) * a.Rc + c] : ChanSum{0, 0};
        }
#pragma unroll
        for (int k = 0; k < kChunk; ++k) {
            if (t + k < t1) {
                ccarry[(t + k) * a.Rc + c] = busy;
                busy = umax64(busy + buf[k].A, buf[k].B);
            }
        }
    }
}

__device__ __forceinline__ void seq_walk(const std::uint64_t* tile_count, std::size_t ntiles,
                                         std::size_t g, std::uint64_t s, std::uint64_t* tile_seq)
{
    const std::size_t t0 = g * kGroup;
    const std::size_t t1 = t0 + kGroup < ntiles ? t0 + kGroup : ntiles;
    for (std::size_t t = t0; t < t1; ++t) {
        tile_seq[t] = s;
        s += tile_count[t];
    }
}

// Level 3: thread (g, r) walks group g's tiles from the group carry-in.
__global__ __launch_bounds__(256) void k_carry_down(KArgs a, std::size_t ntiles,
                                                    std::size_t ngroups, const PlaneSum* psum,
                                                    const MaskWord* tmask,
                                                    const ChanSum* csum,
                                                    const std::uint64_t* tile_count,
                                                    const PlaneCarry* gpcarry,
                                                    const std::uint64_t* gccarry,
                                                    const std::uint64_t* gseq, PlaneCarry* pcarry,
                                                    std::uint64_t* ccarry, std::uint64_t* tile_seq)
{
    const std::uint32_t rt = a.Rp + a.Rc + 1;
    const std::size_t id = static_cast<std::size_t>(blockIdx.x) * blockDim.x + threadIdx.x;
    if (id >= ngroups * rt) {
        return;
    }
    const std::size_t g = id / rt;
    const std::uint32_t r = static_cast<std::uint32_t>(id - g * rt);
    if (r < a.Rp) {
        plane_walk(a, psum, tmask, ntiles, g, r, gpcarry[g * a.Rp + r], pcarry);
    } else if (r < a.Rp + a.Rc) {
        const std::uint32_t c = r - a.Rp;
        chan_walk(a, csum, ntiles, g, c, gccarry[g * a.Rc + c], ccarry);
    } else {
        seq_walk(tile_count, ntiles, g, gseq[g], tile_seq);
    }
}

// The whole chain in one launch, for runs of at most kMidBlock * kChunk
// tiles.  Thread g of block r owns tiles [g span, g span + span) (span <=
// kChunk): it loads their summaries of resource r in one round, folds them,
// the block scans the folds from the engine state, and the thread walks its
// tiles from its carry-in with the summaries still in registers.  Two
// rounds of dependent loads in all, where the three kernels above take
// eight; the compositions, and so the results, are the same.
__global__ __launch_bounds__(kMidBlock) void k_carry_one(
    KArgs a, std::size_t ntiles, std::uint32_t span, const PlaneSum* psum,
    const MaskWord* tmask, const ChanSum* csum, const std::uint64_t* tile_count,
    PlaneCarry* pcarry, std::uint64_t* ccarry, std::uint64_t* tile_seq,
    std::uint64_t* st_pbusy, std::uint64_t* st_ptag, std::uint64_t* st_cbusy,
    std::uint64_t* st_seq, std::uint64_t* ptotal, std::uint64_t* ctotal)
{
    __shared__ MidShared sh;
    __shared__ std::uint64_t red[kMidBlock / kWave];
    stamp_start(a, 1);
    const std::uint32_t r = blockIdx.x;
    const std::size_t t0 = static_cast<std::size_t>(threadIdx.x) * span;
    const std::size_t t1 = t0 + span < ntiles ? t0 + span : ntiles;
    const bool in = t0 < ntiles;
    const bool last = in && t1 == ntiles;
    const bool commit = a.disorder == nullptr || *a.disorder == 0u;
    if (r < a.Rp) {
        std::uint64_t busy = st_pbusy[r];
        std::uint64_t tag1 = st_ptag[static_cast<std::size_t>(r) * 2];
        const auto compose = [&](const PlaneSum& s1, const PlaneSum& s2) {
            return plane_compose(a, s1, s2);
        };
        int at[kChunk];
        PlaneSum buf[kChunk];
        chunk_slots(tmask, mask_words(a), t0, in ? t1 : t0, r, at);
#pragma unroll
        for (int k = 0; k < kChunk; ++k) {
            if (at[k] >= 0) {
                buf[k] = psum[(t0 + k) * a.Rp + at[k]];
            }
        }
        PlaneSum own{};
#pragma unroll
        for (int k = 0; k < kChunk; ++k) {
            if (at[k] >= 0) {
                own = compose(own, buf[k]);
            }
        }
        PlaneSum before;
        (void)block_scan(own, sh.p, PlaneSum{}, compose, before);
        (void)plane_apply(a, before, busy, tag1);  // the state this thread's tiles start from
        std::uint64_t svc = 0;
        {
            std::uint64_t b = busy, t = tag1;
            svc = plane_apply(a, own, b, t);
        }
#pragma unroll
        for (int k = 0; k < kChunk; ++k) {
            // an untouched tile neither reads nor changes this plane
            if (at[k] >= 0) {
                pcarry[(t0 + k) * a.Rp + at[k]] = PlaneCarry{busy, tag1};
                (void)plane_apply(a, buf[k], busy, tag1);
            }
        }
        const std::uint64_t total = block_sum(svc, red);
        if (last && commit) {
            st_pbusy[r] = busy;
            st_ptag[static_cast<std::size_t>(r) * 2] = tag1;
        }
        if (threadIdx.x == 0 && commit) {
            ptotal[r] += total;
        }
    } else if (r < a.Rp + a.Rc) {
        const std::uint32_t c = r - a.Rp;
        std::uint64_t busy = st_cbusy[c];
        ChanSum buf[kChunk];
#pragma unroll
        for (int k = 0; k < kChunk; ++k) {
            buf[k] = t0 + k < t1 ? csum[(t0 + k) * a.Rc + c] : ChanSum{0, 0};
        }
        ChanSum own{0, 0};
#pragma unroll
        for (int k = 0; k < kChunk; ++k) {
            own = chan_compose(own, buf[k]);
        }
        ChanSum before;
        const ChanSum inc = block_scan(own, sh.c, ChanSum{0, 0}, chan_compose, before);
        const std::uint64_t fin = umax64(busy + inc.A, inc.B);
        busy = umax64(busy + before.A, before.B);
#pragma unroll
        for (int k = 0; k < kChunk; ++k) {
            if (t0 + k < t1) {
                ccarry[(t0 + k) * a.Rc + c] = busy;
                busy = umax64(busy + buf[k].A, buf[k].B);
            }
        }
        const std::uint64_t total = block_sum(own.A, red);
        if (last && commit) {
            st_cbusy[c] = fin;
        }
        if (threadIdx.x == 0 && commit) {
            ctotal[c] += total;
        }
    } else if (r == a.Rp + a.Rc) {
        const std::uint64_t seq = *st_seq;
        std::uint64_t cnt[kChunk];
#pragma unroll
        for (int k = 0; k < kChunk; ++k) {
            cnt[k] = t0 + k < t1 ? tile_count[t0 + k] : 0ull;
        }
        std::uint64_t own = 0;
#pragma unroll
        for (int k = 0; k < kChunk; ++k) {
            own += cnt[k];
        }
        std::uint64_t before;
        const std::uint64_t inc = block_scan(
            own, sh.s, std::uint64_t{0}, [](std::uint64_t x, std::uint64_t y) { return x + y; },
            before);
        std::uint64_t q = seq + before;
#pragma unroll
        for (int k = 0; k < kChunk; ++k) {
            if (t0 + k < t1) {
                tile_seq[t0 + k] = q;
                q += cnt[k];
            }
        }
        if (last && commit) {
            *st_seq = seq + inc;
        }
    }
}


__device__ __forceinline__ std::uint64_t wave_max(std::uint64_t v)
{
    for (int o = 32; o > 0; o >>= 1) {
        v = umax64(v, shfl64(v, threadIdx.x ^ o));
    }
    return v;
}

// Replays a batch of linear steps from the plane and channel state and writes
// their completions.  Per step, lane 0 senses unless its page is the one the
// plane last read (with contention the plane is busy from max(busy, issue)
// for the sense, and the hits after it end at the same time); the channel
// moves the 64 records back to back from max(channel busy, issue).  The
// step-level maps are scanned across the batch exactly as records are in the
// general path; then every step's 64 completions follow in closed form:
//   plane  lane 0: lead = max(busy, issue) + sense (busy ignored without
//          contention); lanes 1..63: lead with contention, else issue;
//   channel lane j: top - x (63 - j), top = max(busy, issue) + 64 x.
struct ApplySums {
    std::uint64_t n_rec, n_mod, n_rd, n_hit, mk, lat_lo, lat_hi, lat_max, svc_sum, seq, n_hyb;
};

// kGiven: page-register hits per record from `given` (two page registers):
// a step's first record hits as given[] says.
template <bool kR, bool kGiven = false>
__device__ __forceinline__ void fold_apply(const KArgs& a, const std::uint64_t* xp,
                                           const LinBatchT<kR>& q, int lane, std::uint64_t* p_busy,
                                           std::uint64_t* c_busy, std::uint32_t* p_tag,
                                           std::uint64_t* completion, std::uint8_t* status,
                                           ApplySums& t, std::uint64_t* mt_p,
                                           std::uint64_t* mt_c, const std::uint8_t* given = nullptr)
{
    const StepView v = step_view(a, xp, q, lane);
    const bool m = v.m;
    const std::uint32_t pkey = m ? v.d.plane : 0u;
    const std::uint32_t ckey = m ? v.d.chan : 0u;
    const Group gp = group_plane_runs(a, q.page1, pkey, m, v.active, lane, mt_p);
    const Group gc = group_by(ckey, a.cbits, m, v.active, lane, mt_c);
    const std::uint32_t tag = m ? p_tag[pkey] : 0u;
    const std::uint64_t pbusy = m ? p_busy[pkey] : 0ull;
    const std::uint64_t cbusy = m ? c_busy[ckey] : 0ull;
    std::uint32_t prev1 = static_cast<std::uint32_t>(
        __shfl(static_cast<int>(q.page1), gp.pred < 0 ? lane : gp.pred));
    if (gp.pred < 0) {
        prev1 = tag;
    }
    bool lhit = m && prev1 == q.page1;
    if constexpr (kGiven) {
        lhit = m && given[q.first + static_cast<std::size_t>(lane) * kWave] != 0;
    }
    const std::uint64_t ls = lhit ? 0ull : a.read_ps;
    const std::uint64_t cx = 64 * v.x;
    std::uint64_t Ap = 0, Bp = 0, Ac = 0, Bc = 0;
    if (m) {
        Ap = ls;
        Bp = q.issue + ls;
        Ac = cx;
        Bc = q.issue + cx;
    }
    if (a.contention) {
        scan_pair(gp, Ap, Bp, gc, Ac, Bc, v.d, m, v.active, ls, cx, lane);
    } else {
        scan_group(gc, Ac, Bc, lane);
    }
    const std::uint64_t lead = a.contention ? umax64(pbusy + Ap, Bp) : q.issue + ls;
    const std::uint64_t top = umax64(cbusy + Ac, Bc);
    if (m && lane == gp.last) {
        if (a.contention) {
            p_busy[pkey] = lead;
        }
        p_tag[pkey] = q.page1;
    }
    if (m && lane == gc.last) {
        c_busy[ckey] = top;
    }
    // accounting: every lane gets one record of each step; all are modeled
    // reads, lanes 1..63 hit, lane 0 hits when its page was buffered
    const std::uint64_t nq = static_cast<std::uint64_t>(q.n);
    const std::uint64_t hits = __ballot(lhit);  // (every lane takes part)
    t.n_rec += nq;
    t.n_mod += nq;
    t.n_rd += nq;
    t.n_hit += lane == 0 ? static_cast<std::uint64_t>(__popcll(hits)) : nq;
    const std::uint64_t sx = wave_sum(v.x);                        // lanes 1..63: service x
    const std::uint64_t s0 = wave_sum(m ? umax64(ls, v.x) : 0ull);  // lane 0: max(sense, x)
    t.svc_sum += lane == 0 ? s0 : sx;
    const std::uint64_t seq0 = t.seq;  // sequence number of the batch's first record
    t.seq += 64 * nq;
    // Per-step totals of the 64 records, in closed form (lane k: step k).
    // Record j completes at done_j = max(pd_j, top - x (63 - j)), with pd_0 =
    // lead and pd_j = P for j >= 1 (P = lead with contention, else the issue
    // time).  The channel term grows with j, so among j = 1..63 the last cnt
    // records follow it and the others wait for P; the largest such record is
    // max(lead, top).
    if (m) {
        const std::uint64_t x = v.x;
        const std::uint64_t P = a.contention ? lead : q.issue;
        const std::uint64_t d0 = umax64(lead, top - 63 * x);
        std::uint64_t cnt = 0;  // records 1..63 on the channel side
        if (top >= P) {
            const std::uint64_t D = top - P;
            std::uint64_t tmax = 0;  // largest t <= 62 with x t <= D (x t <= 64 x <= top)
            for (std::uint64_t stp = 32; stp != 0; stp >>= 1) {
                if (tmax + stp <= 62 && x * (tmax + stp) <= D) {
                    tmax += stp;
                }
            }
            cnt = tmax + 1;
        }
        // sum_j done_j - 64 issue, exactly in 128 bits
        std::uint64_t lo = d0, hi = 0;
        const auto add = [&](std::uint64_t f, std::uint64_t w) {  // += f * w
            const std::uint64_t pl = f * w;
            const std::uint64_t ph = __umul64hi(f, w);
            const std::uint64_t n2 = lo + pl;
            hi += ph + (n2 < lo ? 1u : 0u);
            lo = n2;
        };
        const auto sub = [&](std::uint64_t f, std::uint64_t w) {  // -= f * w
            const std::uint64_t pl = f * w;
            const std::uint64_t ph = __umul64hi(f, w);
            hi -= ph + (lo < pl ? 1u : 0u);
            lo -= pl;
        };
        add(63 - cnt, P);
        add(cnt, top);
        sub(x, cnt * (cnt - (cnt != 0 ? 1 : 0)) / 2);
        sub(64, q.issue);
        const std::uint64_t n2 = t.lat_lo + lo;
        t.lat_hi += hi + (n2 < t.lat_lo ? 1u : 0u);
        t.lat_lo = n2;
        const std::uint64_t most = umax64(lead, top);
        t.mk = umax64(t.mk, most);
        t.lat_max = umax64(t.lat_max, most - q.issue);
    }
    // Completions.  Record j >= 1 of step k completes at max(P_k, top_k -
    // x_k (63 - j)) and record 0 at D0_k.  Lane j writes record j of every
    // step (whole 512-B rows: a row left partly written for a later store
    // costs more than the selects), taking P_k, top_k and D0_k from lane k by
    // shuffles; with one transfer time for the whole batch x (63 - j) is a
    // per-lane constant.  Nothing is outstanding here (the batch's values
    // were read above); saying so keeps a conservative wait for vector
    // memory out of the store loop, which would drain the stores.
    const std::uint64_t x0 = readlane64(v.x, 0);
    const bool xuni = __ballot(m && v.x != x0) == 0;
    const std::uint64_t back = static_cast<std::uint64_t>(63 - lane);
    const std::uint64_t P = a.contention ? lead : q.issue;
    const std::uint64_t D0 = umax64(lead, top - 63 * v.x);
    // Status bytes four steps at a time: 4 for a page-register hit (every
    // record but a sensing lane 0), 0 otherwise; with hybrid sampling, 8 more
    // for each record the sampler picks (record j of step k has sequence
    // number seq0 + 64 k + j and key (page, range, read), as in the general
    // path).  Lane l takes records 4 (l & 15) .. + 3 of step k + (l >> 4).
    // They are made next to the completion stores of the same four steps, so
    // that the sampler's hashes run while those stores drain.
    const bool stat = status != nullptr || a.hybrid;
    const bool words = status != nullptr && (reinterpret_cast<std::uintptr_t>(status) & 3u) == 0;
    const auto status4 = [&](int k) {
        const int ks = k + (lane >> 4);
        // every lane takes part in the shuffles
        const std::uint32_t kp = static_cast<std::uint32_t>(
            __shfl(static_cast<int>(q.page1), ks < q.n ? ks : 0));
        const std::uint32_t kr = static_cast<std::uint32_t>(
            __shfl(static_cast<int>(q.rid), ks < q.n ? ks : 0));
        if (ks < q.n) {
            const std::uint32_t r0 = 4u * static_cast<std::uint32_t>(lane & 15);
            const bool sense = r0 == 0 && ((hits >> ks) & 1u) == 0;
            std::uint32_t word = sense ? 0x04040400u : 0x04040404u;
            if (a.hybrid) {
                const std::uint64_t key =
                    ((static_cast<std::uint64_t>(kp) - 1) << a.page_shift) ^
                    (static_cast<std::uint64_t>(kr) << 32);
#pragma unroll
                for (int u = 0; u < 4; ++u) {
                    const std::uint64_t qn =
                        seq0 + static_cast<std::uint64_t>(ks) * kWave + r0 + u;
                    const bool sampled =
                        qn < a.hybrid_warmup ||
                        (a.hybrid_threshold != 0 && mix64(qn ^ key) <= a.hybrid_threshold);
                    if (sampled) {
                        word |= 8u << (8 * u);
                        ++t.n_hyb;
                    }
                }
            }
            if (status != nullptr) {
                std::uint8_t* out =
                    status + q.first + static_cast<std::size_t>(ks) * kWave + r0;
                if (words) {
                    *reinterpret_cast<std::uint32_t*>(out) = word;
                } else {
                    out[0] = static_cast<std::uint8_t>(word);
                    out[1] = static_cast<std::uint8_t>(word >> 8);
                    out[2] = static_cast<std::uint8_t>(word >> 16);
                    out[3] = static_cast<std::uint8_t>(word >> 24);
                }
            }
        }
    };
    std::uint64_t* out = completion + q.first + lane;
    wait_vector_loads();
    const bool z = lane == 0;
    if (xuni) {
        const std::uint64_t xm = x0 * back;
        int k = 0;
        for (; k + 4 <= q.n; k += 4) {
            std::uint64_t pk[4], tk[4], dk[4];
#pragma unroll
            for (int u = 0; u < 4; ++u) {
                pk[u] = shfl64(P, k + u);
                tk[u] = shfl64(top, k + u);
                dk[u] = shfl64(D0, k + u);
            }
#pragma unroll
            for (int u = 0; u < 4; ++u) {
                const std::uint64_t done = umax64(pk[u], tk[u] - xm);
                put_done(&out[static_cast<std::size_t>(k + u) * kWave], z ? dk[u] : done);
            }
            if (stat) {
                status4(k);
            }
        }
        const int kt = k;
        for (; k < q.n; ++k) {
            const std::uint64_t done = umax64(shfl64(P, k), shfl64(top, k) - xm);
            const std::uint64_t d = shfl64(D0, k);
            put_done(&out[static_cast<std::size_t>(k) * kWave], z ? d : done);
        }
        if (stat && kt < q.n) {
            status4(kt);
        }
    } else {
        for (int k = 0; k < q.n; ++k) {
            const std::uint64_t xm = shfl64(v.x, k) * back;
            const std::uint64_t done = umax64(shfl64(P, k), shfl64(top, k) - xm);
            const std::uint64_t d = shfl64(D0, k);
            put_done(&out[static_cast<std::size_t>(k) * kWave], z ? d : done);
        }
        if (stat) {
            for (int k = 0; k < q.n; k += 4) {
                status4(k);
            }
        }
    }
}

// fold_apply for a batch that holds split steps: lane r is run r, m records
// from lane lo of its step, all issued together and reading one page.  The
// run-level maps scan as in fold_apply with the channel moving m records;
// with e = lo + m - 1 the run's records complete at
//   record lo:           max(lead, top - x (m - 1))
//   record j > lo:       max(P, top - x (e - j))
// (P = lead with contention, else the issue time).  Rows are stored whole:
// lane j of a row takes the run its record belongs to, found by walking the
// runs row by row (a row's second run starts at a nonzero lane).
template <bool kGiven>
__device__ __forceinline__ void fold_apply_runs(const KArgs& a, const std::uint64_t* xp,
                                                const LinBatchT<true>& q, int lane,
                                                std::uint64_t* p_busy, std::uint64_t* c_busy,
                                                std::uint32_t* p_tag, std::uint64_t* completion,
                                                std::uint8_t* status, ApplySums& t,
                                                std::uint64_t* mt_p, std::uint64_t* mt_c,
                                                const std::uint8_t* hits)
{
    const StepView v = step_view(a, xp, q, lane);
    const bool m = v.m;
    const std::uint32_t pkey = m ? v.d.plane : 0u;
    const std::uint32_t ckey = m ? v.d.chan : 0u;
    const Group gp = group_plane_runs(a, q.page1, pkey, m, v.active, lane, mt_p);
    const Group gc = group_by(ckey, a.cbits, m, v.active, lane, mt_c);
    const std::uint32_t tag = m ? p_tag[pkey] : 0u;
    const std::uint64_t pbusy = m ? p_busy[pkey] : 0ull;
    const std::uint64_t cbusy = m ? c_busy[ckey] : 0ull;
    std::uint32_t prev1 = static_cast<std::uint32_t>(
        __shfl(static_cast<int>(q.page1), gp.pred < 0 ? lane : gp.pred));
    if (gp.pred < 0) {
        prev1 = tag;
    }
    bool lhit = m && prev1 == q.page1;
    if constexpr (kGiven) {
        const std::size_t at = run_record(q, lane);
        lhit = m && hits[at] != 0;
    }
    const std::uint64_t ls = lhit ? 0ull : a.read_ps;
    const std::uint64_t rm = m ? q.m : 1u;
    const std::uint64_t x = v.x;
    const std::uint64_t cx = rm * x;
    std::uint64_t Ap = 0, Bp = 0, Ac = 0, Bc = 0;
    if (m) {
        Ap = ls;
        Bp = q.issue + ls;
        Ac = cx;
        Bc = q.issue + cx;
    }
    if (a.contention) {
        scan_pair(gp, Ap, Bp, gc, Ac, Bc, v.d, m, v.active, ls, cx, lane);
    } else {
        scan_group(gc, Ac, Bc, lane);
    }
    const std::uint64_t lead = a.contention ? umax64(pbusy + Ap, Bp) : q.issue + ls;
    const std::uint64_t top = umax64(cbusy + Ac, Bc);
    if (m && lane == gp.last) {
        if (a.contention) {
            p_busy[pkey] = lead;
        }
        p_tag[pkey] = q.page1;
    }
    if (m && lane == gc.last) {
        c_busy[ckey] = top;
    }
    const std::uint64_t P = a.contention ? lead : q.issue;
    const std::uint64_t D0 = umax64(lead, top - (rm - 1) * x);
    // accounting: all modeled reads; every record after a run's first hits,
    // the first when its page was buffered
    const std::uint64_t recs = static_cast<std::uint64_t>(q.rows) * kWave;
    if (lane == 0) {
        t.n_rec += recs;
        t.n_mod += recs;
        t.n_rd += recs;
    }
    if (m) {
        t.n_hit += rm - 1 + (lhit ? 1u : 0u);
        t.svc_sum += umax64(ls, x) + (rm - 1) * x;
        // sum of the run's completions - m issue, exactly in 128 bits: among
        // records lo + 1 .. e the last cnt follow the channel, the others P
        std::uint64_t cnt = 0;
        if (rm >= 2 && top >= P) {
            const std::uint64_t D = top - P;
            std::uint64_t tmax = 0;  // largest t <= m - 2 with x t <= D
            for (std::uint64_t stp = 32; stp != 0; stp >>= 1) {
                if (tmax + stp <= rm - 2 && x * (tmax + stp) <= D) {
                    tmax += stp;
                }
            }
            cnt = tmax + 1;
        }
        std::uint64_t lo = D0, hi = 0;
        const auto add = [&](std::uint64_t f, std::uint64_t w) {  // += f * w
            const std::uint64_t pl = f * w;
            const std::uint64_t ph = __umul64hi(f, w);
            const std::uint64_t n2 = lo + pl;
            hi += ph + (n2 < lo ? 1u : 0u);
            lo = n2;
        };
        const auto sub = [&](std::uint64_t f, std::uint64_t w) {  // -= f * w
            const std::uint64_t pl = f * w;
            const std::uint64_t ph = __umul64hi(f, w);
            hi -= ph + (lo < pl ? 1u : 0u);
            lo -= pl;
        };
        add(rm - 1 - cnt, P);
        add(cnt, top);
        sub(x, cnt * (cnt - (cnt != 0 ? 1 : 0)) / 2);
        sub(rm, q.issue);
        const std::uint64_t n2 = t.lat_lo + lo;
        t.lat_hi += hi + (n2 < t.lat_lo ? 1u : 0u);
        t.lat_lo = n2;
        const std::uint64_t most = umax64(lead, top);
        t.mk = umax64(t.mk, most);
        t.lat_max = umax64(t.lat_max, most - q.issue);
    }
    const std::uint64_t seq0 = t.seq;
    t.seq += recs;
    const std::uint32_t e = m ? q.lo + q.m - 1 : 0u;
    const std::uint32_t hit1 = lhit ? 1u : 0u;
    wait_vector_loads();
    int ra = 0;  // the row's first run (wave-uniform)
    for (int r = 0; r < q.rows; ++r) {
        const bool two = ra + 1 < q.n && rl32(q.lo, ra + 1) != 0;
        const int rb = two ? ra + 1 : ra;
        const std::uint32_t kb = two ? rl32(q.lo, rb) : 0u;
        const bool second = two && static_cast<std::uint32_t>(lane) >= kb;
        const auto pick64 = [&](std::uint64_t val) {
            const std::uint64_t va = readlane64(val, ra);
            const std::uint64_t vb = readlane64(val, rb);
            return second ? vb : va;
        };
        const auto pick32 = [&](std::uint32_t val) {
            const std::uint32_t va = rl32(val, ra);
            const std::uint32_t vb = rl32(val, rb);
            return second ? vb : va;
        };
        const std::uint64_t rP = pick64(P);
        const std::uint64_t rtop = pick64(top);
        const std::uint64_t rD0 = pick64(D0);
        const std::uint64_t rx = pick64(x);
        const std::uint32_t re = pick32(e);
        const std::uint32_t j = static_cast<std::uint32_t>(lane);
        const bool first = j == (second ? kb : 0u);
        const std::uint64_t done =
            first ? rD0 : umax64(rP, rtop - rx * static_cast<std::uint64_t>(re - j));
        const std::size_t at = q.first + static_cast<std::size_t>(r) * kWave + lane;
        put_done(&completion[at], done);
        if (status != nullptr || a.hybrid) {
            std::uint8_t st = first && pick32(hit1) == 0 ? 0u : 4u;
            if (a.hybrid) {
                const std::uint64_t key =
                    ((static_cast<std::uint64_t>(pick32(q.page1)) - 1) << a.page_shift) ^
                    (static_cast<std::uint64_t>(pick32(q.rid)) << 32);
                const std::uint64_t qn = seq0 + static_cast<std::uint64_t>(r) * kWave + j;
                if (qn < a.hybrid_warmup ||
                    (a.hybrid_threshold != 0 && mix64(qn ^ key) <= a.hybrid_threshold)) {
                    st |= 8u;
                    ++t.n_hyb;
                }
            }
            if (status != nullptr) {
                status[at] = st;
            }
        }
        ra = rb + 1;
    }
}

// The apply pass copies a tile's step descriptors into LDS with its other
// set-up loads (tiles of up to kStageSteps steps, 4 KiB): read per window
// from memory instead, each read would wait for the previous window's
// completion stores, vector memory completing in issue order.
constexpr std::uint32_t kStageSteps = 256;

__host__ __device__ __forceinline__ std::uint32_t staged_steps(const KArgs& a)
{
    return a.tile <= kStageSteps * kWave ? a.tile / kWave : 0u;
}

// Byte offset of the staged descriptors in the apply pass's LDS (after the
// fences, plane busy, channel busy and plane tags; 16-byte aligned).
__host__ __device__ __forceinline__ std::size_t apply_desc_offset(const KArgs& a)
{
    return (8ull * (a.r_nfence + a.Rp + a.Rc) + 4ull * a.Rp + 15ull) & ~15ull;
}

// Byte offset of the apply pass's lane-matching tables (plane table, then
// channel table) after its state; 16-byte aligned.
__host__ __device__ __forceinline__ std::size_t apply_match_offset(const KArgs& a)
{
    return apply_desc_offset(a) + 16ull * staged_steps(a);
}

// Byte offset of the apply pass's stripe table (Rp words), after the
// lane-matching tables when the run keeps them.
__host__ __device__ __forceinline__ std::size_t apply_stripe_offset(const KArgs& a)
{
    return apply_match_offset(a) + (a.match_lds ? 8ull * (a.Rp + a.Rc) : 0ull);
}
__host__ __device__ __forceinline__ std::size_t apply_range_offset(const KArgs& a)
{
    return (apply_stripe_offset(a) + (a.stripe_lds ? 4ull * a.Rp : 0ull) + 7ull) & ~7ull;
}

// A tile's plane carry-ins are packed like its summaries: word w of the
// mask covers planes [64 w, 64 w + 64), so lane l reads bit l of each word.
// Eight words' carries are in flight before any is written.
template <int kWords = 8>
__device__ __forceinline__ void load_plane_carry(const KArgs& a, const MaskWord* tmask,
                                                 const PlaneCarry* pcarry, std::size_t tile,
                                                 std::uint64_t* p_busy, std::uint32_t* p_tag,
                                                 int lane)
{
    const std::uint32_t words = mask_words(a);
    const MaskWord* tm = tmask + tile * words;
    const PlaneCarry* pc = pcarry + tile * a.Rp;
    const std::uint64_t below = lanemask_lt(lane);
    // (unrolled over the at most kMaxPlanes / 64 words: a loop back edge
    // would make the compiler wait for every carry load before the next)
#pragma unroll
    for (std::uint32_t w0 = 0; w0 < kMaxPlanes / kWave; w0 += kWords) {
        if (w0 >= words) {
            break;
        }
        // the mask words first, then the carries: vector loads complete in
        // issue order, so a word loaded after a carry would wait for it
        MaskWord mw[kWords];
#pragma unroll
        for (int k = 0; k < kWords; ++k) {
            mw[k] = w0 + k < words ? tm[w0 + k] : MaskWord{0, 0, 0};
        }
        PlaneCarry c[kWords];
        bool has[kWords];
#pragma unroll
        for (int k = 0; k < kWords; ++k) {
            has[k] = ((mw[k].bits >> lane) & 1ull) != 0;
            if (has[k]) {
                c[k] = pc[mw[k].base + static_cast<std::uint32_t>(__popcll(mw[k].bits & below))];
            }
        }
#pragma unroll
        for (int k = 0; k < kWords; ++k) {
            if (has[k]) {
                const std::uint32_t r = (w0 + k) * kWave + static_cast<std::uint32_t>(lane);
                p_busy[r] = c[k].busy;
                p_tag[r] = static_cast<std::uint32_t>(c[k].tag1);
            }
        }
    }
}

__device__ __forceinline__ void load_chan_carry(const KArgs& a, const std::uint64_t* ccarry,
                                                std::size_t tile, std::uint64_t* c_busy, int lane)
{
    constexpr int kPer = 4;
    const std::uint64_t* cc = ccarry + tile * a.Rc;
    for (std::uint32_t r0 = 0; r0 < a.Rc; r0 += kPer * kWave) {
        std::uint64_t v[kPer];
#pragma unroll
        for (int k = 0; k < kPer; ++k) {
            const std::uint32_t r = r0 + k * kWave + static_cast<std::uint32_t>(lane);
            v[k] = r < a.Rc ? cc[r] : 0ull;
        }
#pragma unroll
        for (int k = 0; k < kPer; ++k) {
            const std::uint32_t r = r0 + k * kWave + static_cast<std::uint32_t>(lane);
            if (r < a.Rc) {
                c_busy[r] = v[k];
            }
        }
    }
}

// Runs of descriptor rows r0 .. r1 - 1 of a window (lane r holding row r's
// descriptor sd, its split side entry sp and range id; smask: the split
// rows) laid out one run per lane, at most 64: row r's first run sits at
// lane (r - r0) + the split rows in [r0, r), its second run after it.
__device__ __forceinline__ void expand_rows(LinBatchT<true>& q, const StepDesc& sd,
                                            const SplitDesc& sp,
                                            std::uint32_t rid, std::uint64_t smask, int r0,
                                            int r1, std::size_t w0, int lane)
{
    const std::uint64_t below0 = lanemask_lt(r0);
    const auto before = [&](int r) {  // runs of rows r0 .. r - 1
        return (r - r0) + __popcll(smask & lanemask_lt(r) & ~below0);
    };
    int r = r0;  // the last row whose first run is at or before this lane
    for (int stp = 32; stp != 0; stp >>= 1) {
        if (r + stp < r1 && before(r + stp) <= lane) {
            r += stp;
        }
    }
    const int nruns = before(r1 - 1) + 1 + static_cast<int>((smask >> (r1 - 1)) & 1ull);
    const bool second = lane > before(r);
    const bool two = ((smask >> r) & 1ull) != 0;
    const std::uint32_t p1 = static_cast<std::uint32_t>(__shfl(static_cast<int>(sd.page1), r));
    const std::uint32_t by = static_cast<std::uint32_t>(__shfl(static_cast<int>(sd.bytes), r));
    const std::uint64_t is = shfl64(sd.issue, r);
    const std::uint32_t ra = static_cast<std::uint32_t>(__shfl(static_cast<int>(rid), r));
    const std::uint32_t pb = static_cast<std::uint32_t>(__shfl(static_cast<int>(sp.page1b), r));
    const std::uint32_t k = static_cast<std::uint32_t>(__shfl(static_cast<int>(sp.k), r));
    const std::uint32_t rb = static_cast<std::uint32_t>(__shfl(static_cast<int>(sp.ridb), r));
    const bool in = lane < nruns;
    q.page1 = in ? (second ? pb : p1) : 0u;
    q.bytes = by & ~kSplitFlag;
    q.issue = is;
    q.rid = second ? rb : ra;
    q.m = two ? (second ? kWave - k : k) : kWave;
    q.lo = second ? k : 0u;
    q.first = w0 + static_cast<std::size_t>(r0) * kWave;
    q.n = nruns;
    q.rows = r1 - r0;
    q.split = (smask & lanemask_lt(r1) & ~below0) != 0;
}

// Folds the apply pass's pending batch (fold_apply_runs when it holds a
// split step; kGiven: page-register hits from `hits`) and empties it.
template <bool kR, bool kGiven>
__device__ __forceinline__ void fold_batch(const KArgs& a, const std::uint64_t* xp,
                                           LinBatchT<kR>& q, int lane, std::uint64_t* p_busy,
                                           std::uint64_t* c_busy, std::uint32_t* p_tag,
                                           std::uint64_t* completion, std::uint8_t* status,
                                           ApplySums& t, std::uint64_t* mt_p, std::uint64_t* mt_c,
                                           const std::uint8_t* hits)
{
    if constexpr (kR) {
        if (q.any_split()) {
            fold_apply_runs<kGiven>(a, xp, q, lane, p_busy, c_busy, p_tag, completion, status, t,
                                    mt_p, mt_c, hits);
            q.clear();
            return;
        }
    }
    fold_apply<kR, kGiven>(a, xp, q, lane, p_busy, c_busy, p_tag, completion, status, t, mt_p,
                           mt_c, hits);
    q.clear();
}

// The apply pass over one tile.  kSplit: the tile holds split steps (packed
// records; the summary pass says so per tile), which its batches take as
// runs; without it the body is the whole-step one, whose folds and stores
// then keep every register the pass has (the split-capable body needs more:
// compiled into the same code path it would make the whole-step folds spill).
template <bool kRefresh, bool kHits, bool kStaged, bool kPacked, bool kSplit, bool kWide = false>
__device__ __forceinline__ void apply_tile(
    const KArgs& a, const void* rec, std::size_t n, std::uint64_t base_ps,
    const PlaneCarry* pcarry, const MaskWord* tmask, const std::uint64_t* ccarry,
    const std::uint64_t* tile_seq, std::uint64_t* completion, std::uint8_t* status,
    DevReport* tile_rep, const std::uint8_t* hits, const StepDesc* desc, std::uint64_t* sm,
    std::uint64_t* xp)
{
    RangeView fence(sm);
    std::uint64_t* p_busy = sm + a.r_nfence;
    std::uint64_t* c_busy = p_busy + a.Rp;
    std::uint32_t* p_tag = reinterpret_cast<std::uint32_t*>(c_busy + a.Rc);
    const int lane = threadIdx.x;
    const std::size_t tile = blockIdx.x;
    // set-up loads in flight together: the fences, then the carry-ins, which
    // exist for the planes the tile touches (the only ones it reads)
    const std::size_t begin = tile * a.tile;
    const std::size_t end = begin + a.tile < n ? begin + a.tile : n;
    // kStaged: the launch found descriptors and a tile of at most kStageSteps
    // steps (a template parameter: as a run-time flag it costs registers)
    constexpr bool stage = kStaged;
    StepDesc* sdesc = reinterpret_cast<StepDesc*>(reinterpret_cast<unsigned char*>(sm) +
                                                  apply_desc_offset(a));
    std::uint64_t* mt_p = a.match_lds ? reinterpret_cast<std::uint64_t*>(
                                            reinterpret_cast<unsigned char*>(sm) +
                                            apply_match_offset(a))
                                      : nullptr;
    std::uint64_t* mt_c = a.match_lds ? mt_p + a.Rp : nullptr;
    const std::size_t tsteps = (end - begin + kWave - 1) / kWave;
    const FenceRegs fr = fetch_fences(a, lane);
    const RangeRegs rr = fetch_ranges(a, lane);
    const std::uint64_t xv = fetch_xfer(a, lane);
    constexpr int kDescPerLane = static_cast<int>(kStageSteps) / kWave;
    StepDesc dv[kDescPerLane];
#pragma unroll
    for (int k = 0; k < kDescPerLane; ++k) {
        const std::size_t j = static_cast<std::size_t>(k * kWave + lane);
        dv[k] = StepDesc{0, 0, 0};
        if (stage && j < tsteps) {
            dv[k] = desc[begin / kWave + j];
        }
    }
    load_plane_carry(a, tmask, pcarry, tile, p_busy, p_tag, lane);
    load_chan_carry(a, ccarry, tile, c_busy, lane);
    store_fences(a, fr, sm, lane);
    store_ranges(a, rr, reinterpret_cast<unsigned char*>(sm) + apply_range_offset(a), fence, lane);
    store_xfer(xp, xv, lane);
    if (a.match_lds) {
        for (std::uint32_t r = lane; r < a.Rp + a.Rc; r += kWave) {
            mt_p[r] = 0;
        }
    }
    std::uint32_t* stab = nullptr;
    if (a.stripe_lds) {
        stab = reinterpret_cast<std::uint32_t*>(reinterpret_cast<unsigned char*>(sm) +
                                                apply_stripe_offset(a));
        fill_stripe_table(a, stab, lane);
    }
    if (stage) {
#pragma unroll
        for (int k = 0; k < kDescPerLane; ++k) {
            const std::size_t j = static_cast<std::size_t>(k * kWave + lane);
            if (j < tsteps) {
                sdesc[j] = dv[k];
            }
        }
    }
    __syncthreads();
    // the batch folds' accumulators, and the ones only the general path adds to
    ApplySums t{0, 0, 0, 0, 0, 0, 0, 0, 0, tile_seq[tile], 0};
    std::uint64_t n_byp = 0, n_uns = 0, n_wr = 0, n_prog = 0;
    RangeCache rc = empty_cache();
    RangeCache rcu = empty_cache();  // wave-uniform copy for linear steps
    LinBatchT<kSplit> q = empty_batch<kSplit>();
    constexpr int kFull = kSplit ? kWave - 1 : kWave;  // room for a split step's runs
    std::uint32_t lin_miss = 0;  // steps in a row that were not linear (wave-uniform)
    // Windows of 64 steps.  A window whose steps the summary pass found all
    // linear is replayed from their descriptors alone, without reading its
    // records; any other window streams its records through the pipeline.
    for (std::size_t w0 = begin; w0 < end; w0 += kWave * kWave) {
        const std::size_t wend = w0 + kWave * kWave < end ? w0 + kWave * kWave : end;
        if (desc != nullptr) {
            const int nst = static_cast<int>((wend - w0 + kWave - 1) / kWave);
            StepDesc sd{0, 0, 0};
            if (lane < nst) {
                if (stage) {
                    sd = sdesc[(w0 - begin) / kWave + lane];
                } else {
                    sd = desc[w0 / kWave + lane];
                }
            }
            const std::uint64_t all = nst == kWave ? ~0ull : ((1ull << nst) - 1);
            // (a split step's descriptor in a tile not marked split: the
            // window is streamed, where such a step takes the general path)
            const bool ok = sd.bytes != 0 && (kSplit || (sd.bytes & kSplitFlag) == 0);
            if (__ballot(lane < nst && ok) == all) {
                const std::uint32_t rid =
                    a.desc_rid != nullptr && lane < nst ? a.desc_rid[w0 / kWave + lane] : 0u;
                const std::uint64_t smask =
                    kSplit ? __ballot(lane < nst && (sd.bytes & kSplitFlag) != 0) : 0ull;
                // split steps have their second runs in the side array; the
                // window's runs fold in one batch, or in two when they exceed 64
                SplitDesc sp{0, 0, 0, 0};
                if (kSplit && ((smask >> lane) & 1ull) != 0) {
                    sp = a.desc_split[w0 / kWave + lane];
                }
                if constexpr (!kSplit) {
                    q.page1 = sd.page1;
                    q.bytes = sd.bytes;
                    q.issue = sd.issue;
                    q.rid = rid;
                    q.first = w0;
                    q.n = nst;
                    q.rows = nst;
                    fold_batch<kSplit, kHits>(a, xp, q, lane, p_busy, c_busy, p_tag, completion,
                               status, t, mt_p, mt_c, hits);
                } else {
                    const int runs = nst + __popcll(smask);
                    const int half = runs <= kWave ? nst : nst / 2;
                    for (int r0 = 0; r0 < nst;) {
                        const int r1 = r0 == 0 ? half : nst;
                        if (smask != 0) {
                            expand_rows(q, sd, sp, rid, smask, r0, r1, w0, lane);
                        } else {
                            q.page1 = sd.page1;
                            q.bytes = sd.bytes;
                            q.issue = sd.issue;
                            q.rid = rid;
                            q.m = kWave;
                            q.lo = 0;
                            q.first = w0;
                            q.n = nst;
                            q.rows = nst;
                        }
                        fold_batch<kSplit, kHits>(a, xp, q, lane, p_busy, c_busy, p_tag, completion,
                                   status, t, mt_p, mt_c, hits);
                        r0 = r1;
                    }
                }
                continue;
            }
        }
        // (the four-wave form keeps two steps in flight)
        constexpr int kDepth = kPacked && kWide ? 2 : kPipe;
        constexpr std::size_t kSpan = static_cast<std::size_t>(kDepth) * kWave;
        using Pipe = std::conditional_t<kPacked, PackedPipeT<kDepth>, RecordPipe>;
        static_assert(kPacked || kDepth == kPipe, "32-byte records keep kPipe steps");
        Pipe pipe;
        pipe.issue(rec, w0, wend, lane);
        for (std::size_t g = w0; g < wend; g += kSpan) {
            pipe.advance(rec, g + kSpan, wend, lane);
            const std::size_t gend = g + kSpan < wend ? g + kSpan : wend;
            for (std::size_t s = g; s < gend; s += kWave) {
                typename Pipe::Step sr;
                pipe.take(sr);
                const std::size_t i = s + lane;
                const bool valid = i < end;
                if ((kHits || a.slots == 1) && a.lead == nullptr) {
                    // batched as in the summary pass
                    LinStep ls;
                    bool lin = false;
                    if (lin_miss < kLinGiveUp || (s / kWave) % kLinProbe == 0) {
                        lin = detect_step<kRefresh, kSplit>(a, fence, rcu, sr, base_ps,
                                                            s + kWave <= end, lane, ls);
                        lin_miss = lin ? 0u : lin_miss + 1u;
                    }
                    if (lin) {
                        if (ls.k == 0) {
                            q.push(ls.page1, ls.issue, ls.bytes, s, ls.rid);
                        } else {
                            q.push_split(ls.page1, ls.page1b, ls.k, ls.issue, ls.bytes, s,
                                         ls.rid, ls.ridb);
                        }
                    }
                    if (q.n != 0 && (!lin || q.n >= kFull || s + kWave >= wend)) {
                        fold_batch<kSplit, kHits>(a, xp, q, lane, p_busy, c_busy, p_tag, completion,
                               status, t, mt_p, mt_c, hits);
                    }
                    if (lin) {
                        continue;
                    }
                }
                uint4 x, y;
                step_records(sr, lane, x, y);
                Dec d = valid ? decode<kRefresh>(a, fence, rc, x, y, base_ps, stab)
                              : invalid_dec();
                if (!kPacked && a.lead != nullptr && valid && a.lead[i] != 0) {
                    d.cls = kClsFollower;  // timed by k_follow from its group's request
                }
                const bool m = valid && d.cls == kClsModeled;
                const bool hbit = kHits && valid && hits[i] != 0;
                const std::uint64_t active = __ballot(m);
                std::uint8_t st = static_cast<std::uint8_t>(d.cls);
                std::uint64_t done = 0;
                if (!kHits && active != 0 && run_step(a, d, active, lane)) {
                    bool same_x;
                    const std::uint64_t xfer = lane_xfer(a, xp, d, m, active, same_x);
                    const std::uint64_t W = run_channel_max(d, xfer, lane);
                    const std::uint32_t page1 = static_cast<std::uint32_t>(d.page1);
                    const std::uint32_t pkey = d.plane;
                    const std::uint32_t ckey = d.chan;
                    const std::uint32_t tag = p_tag[pkey];
                    const std::uint64_t pbusy = p_busy[pkey];
                    const std::uint64_t cbusy = c_busy[ckey];
                    const std::uint64_t i0 = readlane64(d.issue, 0);
                    const bool lhit = tag == page1;
                    const std::uint64_t ls = lhit ? 0ull : a.read_ps;
                    const std::uint64_t lead = a.contention ? umax64(pbusy, i0) + ls : i0 + ls;
                    std::uint64_t pd;
                    if (lane == 0) {
                        pd = lead;
                    } else {
                        pd = a.contention ? umax64(lead, d.issue) : d.issue;
                    }
                    const std::uint64_t k1 = static_cast<std::uint64_t>(lane + 1);
                    const std::uint64_t back = static_cast<std::uint64_t>(62 - lane);
                    const std::uint64_t cd =
                        umax64(cbusy + xfer * k1, lane == 63 ? W + xfer : W - xfer * back);
                    if (lane == 63) {
                        if (a.contention) {
                            p_busy[pkey] = pd;
                        }
                        p_tag[pkey] = page1;
                        c_busy[ckey] = cd;
                    }
                    done = umax64(pd, cd);
                    const bool hit = lane == 0 ? lhit : true;
                    const std::uint64_t svc = lane == 0 ? ls : 0ull;
                    if (a.hybrid) {
                        const std::uint64_t qn = t.seq + static_cast<std::uint64_t>(lane);
                        const std::uint64_t key = ((d.page1 - 1) << a.page_shift) ^
                                                  (static_cast<std::uint64_t>(d.range_id) << 32);
                        if (qn < a.hybrid_warmup ||
                            (a.hybrid_threshold != 0 && mix64(qn ^ key) <= a.hybrid_threshold)) {
                            st |= 8u;
                            ++t.n_hyb;
                        }
                    }
                    ++t.n_mod;
                    ++t.n_rd;
                    if (hit) {
                        st |= 4u;
                        ++t.n_hit;
                    }
                    t.mk = umax64(t.mk, done);
                    const std::uint64_t lat = done - d.issue;
                    add128(t.lat_lo, t.lat_hi, lat);
                    t.lat_max = umax64(t.lat_max, lat);
                    t.svc_sum += umax64(svc, xfer);
                    t.seq += 64;
                } else if (active != 0) {
                    bool same_x = false;
                    const std::uint64_t xfer = lane_xfer(a, xp, d, m, active, same_x);
                    const std::uint32_t page1 = static_cast<std::uint32_t>(d.page1);
                    const std::uint32_t pkey = m ? d.plane : 0u;
                    const std::uint32_t ckey = m ? d.chan : 0u;
                    const Group gp = group_by(pkey, a.pbits, m, active, lane, mt_p);
                    const Group gc = group_by(ckey, a.cbits, m, active, lane, mt_c);
                    // state reads come before this step's writes
                    const std::uint32_t tag = m ? p_tag[pkey] : 0u;
                    const std::uint64_t pbusy = m ? p_busy[pkey] : 0ull;
                    const std::uint64_t cbusy = m ? c_busy[ckey] : 0ull;
                    std::uint32_t prev1 = static_cast<std::uint32_t>(
                        __shfl(static_cast<int>(page1), gp.pred < 0 ? lane : gp.pred));
                    if (gp.pred < 0) {
                        prev1 = tag;
                    }
                    const bool hit = kHits ? (m && hbit) : (a.slots != 0 && m && prev1 == page1);
                    const std::uint64_t svc = plane_service(a, d.bits, hit);
                    std::uint64_t pd, cd;
                    const StepCounts sc = count_services(m, d.bits, hit);
                    const std::uint64_t origin = readlane64(
                        d.issue, __ffsll(static_cast<long long>(active)) - 1);
                    const std::uint64_t most =
                        static_cast<std::uint64_t>(static_cast<std::uint32_t>(
                            __popcll(sc.miss))) * a.read_ps +
                        static_cast<std::uint64_t>(static_cast<std::uint32_t>(
                            __popcll(sc.prog))) * a.program_ps;
                    const bool small =
                        !kRefresh && same_x && most < (1ull << 30) && xfer < (1ull << 24) &&
                        __ballot(m && d.issue - origin >= (1ull << 30)) == 0;
                    if (small) {
                        // lane i of a group completes at max(busy, max over
                        // k <= i of (issue_k - E_k)) + E_i + its service, with
                        // E the service of the group's lanes before: where no
                        // lane's issue time passes busy + E the maximum is busy,
                        // else it is a prefix maximum of issue - E, in 32 bits
                        // from the step's first issue time
                        const std::uint64_t below = lanemask_lt(lane);
                        const std::uint32_t Ep = static_cast<std::uint32_t>(
                            count_service(a, sc, gp.peers & below));
                        const std::uint32_t x32 = static_cast<std::uint32_t>(xfer);
                        const std::uint32_t Ec =
                            x32 * static_cast<std::uint32_t>(__popcll(gc.peers & below));
                        const bool wp = a.contention != 0 &&
                                        __ballot(m && d.issue > pbusy + Ep) != 0;
                        const bool wc = __ballot(m && d.issue > cbusy + Ec) != 0;
                        std::uint64_t tp = pbusy, tc = cbusy;
                        if (wp || wc) {
                            const std::uint32_t rel =
                                m ? static_cast<std::uint32_t>(d.issue - origin) : 0u;
                            const std::uint32_t most32 = static_cast<std::uint32_t>(most);
                            const std::uint32_t c64 = x32 * 64u;
                            std::uint32_t vp = rel + most32 - Ep, vc = rel + c64 - Ec;
                            group_prefix_max(vp, wp ? gp.pred : -1, vc, wc ? gc.pred : -1, lane);
                            // (origin - most can only pass below zero where the
                            // maximum is another lane's: compare before taking off)
                            if (wp) {
                                tp = origin + vp > pbusy + most32 ? origin + vp - most32 : pbusy;
                            }
                            if (wc) {
                                tc = origin + vc > cbusy + c64 ? origin + vc - c64 : cbusy;
                            }
                        }
                        pd = a.contention ? (m ? tp + Ep + svc : 0ull) : d.issue + svc;
                        cd = m ? tc + Ec + xfer : 0ull;
                    } else {
                        std::uint64_t Ap = m ? svc : 0ull;
                        std::uint64_t Bp = m ? d.issue + svc : 0ull;
                        std::uint64_t Ac = m ? xfer : 0ull;
                        std::uint64_t Bc = m ? d.issue + xfer : 0ull;
                        if (a.contention) {
                            scan_pair(gp, Ap, Bp, gc, Ac, Bc, d, m, active, svc, xfer, lane);
                        } else {
                            scan_group(gc, Ac, Bc, lane);
                        }
                        pd = a.contention ? (m ? umax64(pbusy + Ap, Bp) : 0ull) : d.issue + svc;
                        cd = m ? umax64(cbusy + Ac, Bc) : 0ull;
                    }
                    if (m && lane == gp.last) {
                        if (a.contention) {
                            p_busy[pkey] = pd;
                        }
                        p_tag[pkey] = page1;
                    }
                    if (m && lane == gc.last) {
                        c_busy[ckey] = cd;
                    }
                    if (m) {
                        done = umax64(pd, cd);
                        const std::uint64_t rank = __popcll(active & lanemask_lt(lane));
                        const std::uint64_t qn = t.seq + rank;
                        if (a.hybrid) {
                            const std::uint64_t key =
                                ((d.page1 - 1) << a.page_shift) ^
                                (static_cast<std::uint64_t>(d.range_id) << 32) ^ dec_op(d.bits);
                            const bool sampled =
                                qn < a.hybrid_warmup ||
                                (a.hybrid_threshold != 0 && mix64(qn ^ key) <= a.hybrid_threshold);
                            if (sampled) {
                                st |= 8u;
                                ++t.n_hyb;
                            }
                        }
                        ++t.n_mod;
                        if ((d.bits & 1u) == 0) {
                            ++t.n_rd;
                            if (hit) {
                                st |= 4u;
                                ++t.n_hit;
                            }
                        } else {
                            n_wr += (d.bits & 4u) ? 0u : 1u;
                            if (svc != 0) {
                                st |= 16u;
                                ++n_prog;
                            }
                        }
                        t.mk = umax64(t.mk, done);
                        const std::uint64_t lat = done - d.issue;
                        add128(t.lat_lo, t.lat_hi, lat);
                        t.lat_max = umax64(t.lat_max, lat);
                        t.svc_sum += umax64(svc, xfer);
                    }
                    t.seq += __popcll(active);
                }
                if (valid) {
                    ++t.n_rec;
                    if (d.cls == kClsBypass) {
                        done = d.issue;
                        ++n_byp;
                    } else if (d.cls == kClsUnsupported) {
                        done = ~0ull;
                        ++n_uns;
                    }
                    put_done(&completion[i], done);
                    if (status != nullptr) {
                        status[i] = st;
                    }
                }
            }
        }
    }
    // 128-bit latency sum: reduce the high words, then the low words with
    // their carries.
    std::uint64_t hi = wave_sum(t.lat_hi);
    std::uint64_t carry = 0;
    std::uint64_t v = t.lat_lo;
    for (int o = 32; o > 0; o >>= 1) {
        const std::uint64_t other = shfl64(v, threadIdx.x ^ o);
        const std::uint64_t oc = shfl64(carry, threadIdx.x ^ o);
        const std::uint64_t sum = v + other;
        carry = carry + oc + (sum < v ? 1u : 0u);
        v = sum;
    }
    hi += carry;
    const std::uint64_t vals[14] = {
        wave_sum(t.n_rec), wave_sum(t.n_mod), wave_sum(n_byp), wave_sum(n_uns), wave_sum(t.n_rd),
        wave_sum(n_wr),  wave_sum(t.n_hit), wave_sum(n_prog), wave_sum(t.n_hyb), wave_max(t.mk),
        v,               hi,              wave_max(t.lat_max), wave_sum(t.svc_sum)};
    if (lane < 14) {
        unsigned long long out = 0;
#pragma unroll
        for (int k = 0; k < 14; ++k) {
            out = lane == k ? vals[k] : out;
        }
        tile_rep[tile].v[lane] = out;
    }
}

// Packed records: three waves per SIMD (at most 168 registers), since the
// general steps' chains of ballots, shuffles and LDS updates need the
// latency hiding and the streamed linear steps lose nothing.  32-byte
// records hold twice the bytes per step in registers and would spill.
// kWide: four waves per SIMD with two steps in flight, for large streams of
// general steps (k_apply 4.15 -> 3.59 ms at 2^28 random records); on streams
// of linear steps its spilled registers cost 7-15% of the pass.
template <bool kRefresh, bool kHits, bool kStaged = false, bool kPacked = false,
          bool kWide = false>
__global__ __launch_bounds__(64) __attribute__((amdgpu_waves_per_eu(kWide ? 4 : (kPacked ? 3 : 1)))) void k_apply(
    KArgs a, const void* rec, std::size_t n, std::uint64_t base_ps, const PlaneCarry* pcarry,
    const MaskWord* tmask, const std::uint64_t* ccarry, const std::uint64_t* tile_seq,
    std::uint64_t* completion, std::uint8_t* status, DevReport* tile_rep,
    const std::uint8_t* hits, const StepDesc* desc)
{
    extern __shared__ std::uint64_t sm[];
    __shared__ std::uint64_t xp[33];
    if (a.mixed == 0) {
        stamp_start(a, 2);
    }
    // a stream that went back in time is timed again from a sorted copy:
    // nothing of this run is kept (8.4M records: 190 us not spent here)
    if (a.disorder != nullptr && *a.disorder != 0u) {
        return;
    }
    const std::uint8_t kind = a.tile_split != nullptr ? a.tile_split[blockIdx.x] : 0;
    if (kind == kTilePlain) {
        return;  // k_plain_apply took it
    }
    if constexpr (!kRefresh) {
        if (kind != 0) {
            apply_tile<kRefresh, kHits, kStaged, kPacked, true, kWide>(
                a, rec, n, base_ps, pcarry, tmask, ccarry, tile_seq, completion, status, tile_rep,
                hits, desc, sm, xp);
            return;
        }
    }
    apply_tile<kRefresh, kHits, kStaged, kPacked, false, kWide>(a, rec, n, base_ps, pcarry, tmask,
                                                                ccarry, tile_seq, completion,
                                                                status, tile_rep, hits, desc, sm,
                                                                xp);
}

// ---- scattered records -----------------------------------------------------
//
// k_summary and k_apply are built around runs of linear steps; what they hold
// for those costs a step of scattered records registers, spilled scalars and
// occupancy.  Streams over geometries of power-of-two axes whose range table
// fits LDS (plain_run) have two kernels of their own with the same inputs
// and outputs and none of that: k_plain_summary takes the tiles that do not
// look like runs of lines and leaves the others to k_summary, and
// k_plain_apply replays those it took.
//
// What bounds them is the number of instructions a step issues (k_summary: 515
// vector, 256 scalar and 86 branches on records spread over 37 ranges), so a
// step is decoded without divergence in 32-bit page arithmetic, its groups
// come from a 32-slot LDS table and a ballot per further key bit, and sums over
// a group are population counts of its mask (count_services).
constexpr std::uint32_t kMatchSlots = 32;

// LDS of both kernels, in this order: the range table (bases, lengths), the
// per-plane and per-channel 64-bit words, the match table, then 32-bit words.
struct PlainLds {
    std::uint64_t* fence;
    std::uint64_t* len;
    std::uint64_t* w64;       // kernel's own 64-bit state
    std::uint64_t* tab;       // [kMatchSlots], zero between uses
    std::uint32_t* page0;
    std::uint32_t* w32;       // kernel's own 32-bit state
};

__host__ __device__ __forceinline__ std::size_t plain_lds_bytes(const KArgs& a, std::size_t w64,
                                                                std::size_t w32)
{
    return 8ull * (2ull * a.r_count + w64 + kMatchSlots) + 4ull * (a.r_count + w32);
}

__host__ __device__ __forceinline__ std::size_t plain_summary_lds(const KArgs& a)
{
    const std::size_t rp = plane_slots(a);
    return plain_lds_bytes(a, rp + 2ull * a.Rc, 2 * rp) + 2 * rp;
}

__host__ __device__ __forceinline__ std::size_t plain_apply_lds(const KArgs& a)
{
    return plain_lds_bytes(a, static_cast<std::size_t>(a.Rp) + a.Rc, a.Rp);
}

__device__ __forceinline__ PlainLds plain_layout(const KArgs& a, std::uint64_t* sm,
                                                 std::size_t w64)
{
    PlainLds l;
    l.fence = sm;
    l.len = l.fence + a.r_count;
    l.w64 = l.len + a.r_count;
    l.tab = l.w64 + w64;
    l.page0 = reinterpret_cast<std::uint32_t*>(l.tab + kMatchSlots);
    l.w32 = l.page0 + a.r_count;
    return l;
}

__device__ __forceinline__ void plain_load(const KArgs& a, const PlainLds& l, int lane)
{
#pragma unroll
    for (int k = 0; k < kRangesPerLane; ++k) {
        const std::uint32_t j = static_cast<std::uint32_t>(k * kWave + lane);
        if (j < a.r_count) {
            l.fence[j] = a.r_base[j];
            const std::uint32_t meta = a.r_meta[j];
            l.len[j] = a.r_length[j] | (static_cast<std::uint64_t>((meta >> 8) & 0xfu) << 60);
            l.page0[j] = static_cast<std::uint32_t>(a.r_file_offset[j] >> a.page_shift);
        }
    }
    if (lane < static_cast<int>(kMatchSlots)) {
        l.tab[lane] = 0;
    }
}

// One record (x: address, bytes; y: issue time, flags), classified as decode()
// does for reads and writes.
struct PlainRec {
    std::uint64_t issue;
    std::uint32_t cls, bits, page1, plane, chan, bytes;
};

__device__ __forceinline__ PlainRec plain_record(const KArgs& a, const PlainLds& l,
                                                 const uint4& x, const uint4& y, bool valid,
                                                 std::uint64_t base_ps)
{
    const std::uint64_t addr = x.x | (static_cast<std::uint64_t>(x.y) << 32);
    const std::uint32_t bytes = x.z;
    const bool huge = x.w != 0;  // 2^32 bytes or more
    const std::uint32_t op = y.z & 0xffu;
    PlainRec d;
    d.issue = base_ps + (y.x | (static_cast<std::uint64_t>(y.y) << 32));
    d.bytes = bytes;
    std::uint32_t lo = 0;  // ranges whose base is at most addr
    for (std::uint32_t step = a.r_top; step != 0; step >>= 1) {
        const std::uint32_t mid = lo + step;
        const std::uint32_t at = (mid < a.r_count ? mid : a.r_count) - 1;
        lo = l.fence[at] <= addr && mid <= a.r_count ? mid : lo;
    }
    const std::uint32_t idx = lo == 0 ? 0u : lo - 1;
    const std::uint64_t off = addr - l.fence[idx];
    const std::uint64_t lm = l.len[idx];
    const std::uint64_t len = lm & kRangeLenMask;
    const std::uint32_t page_bytes = 1u << a.page_shift;
    const std::uint32_t in_page = static_cast<std::uint32_t>(off) & (page_bytes - 1);
    const bool inside = lo != 0 && off < len;
    // access_supported and media_descriptor (hbf_device.cuh:843-860): inside
    // one page and the range, permitted
    const bool ok = inside && !huge && bytes != 0 && op <= 1 && bytes <= page_bytes - in_page &&
                    bytes <= len - off &&
                    ((static_cast<std::uint32_t>(lm >> 60) >> (op & 1u)) & 1u) != 0;
    d.cls = ok ? kClsModeled : (inside || huge ? kClsUnsupported : kClsBypass);
    if (__ballot(valid && !inside) != 0 && !inside && lo < a.r_count) {
        // outside every range: unsupported when the span reaches the next one
        if (overlaps(l.fence[lo], l.len[lo] & kRangeLenMask, addr, bytes)) {
            d.cls = kClsUnsupported;
        }
    }
    d.cls = valid ? d.cls : kClsInvalid;
    const std::uint32_t page = l.page0[idx] + static_cast<std::uint32_t>(off >> a.page_shift);
    d.page1 = page + 1;
    d.bits = op;
    if (op == 1 && (a.every_write != 0 || in_page + bytes == page_bytes)) {
        d.bits = 3u;
    }
    d.plane = 0;
    d.chan = 0;
    if (!a.flat) {
        std::uint32_t c[4];
#pragma unroll
        for (int ax = 0; ax < 4; ++ax) {
            c[ax] = (page >> a.axis_shift[ax]) & (a.axis_size[ax] - 1);
        }
        d.chan = c[0];
        d.plane = ((c[0] * a.W + c[1]) * a.D + c[2]) * a.P + c[3];
    }
    return d;
}

// Lanes of `active` with this lane's key (m: this lane is one of them): the
// low five key bits through the LDS table, the others by ballots.
__device__ __forceinline__ std::uint64_t plain_match(const PlainLds& l, std::uint32_t key,
                                                     std::uint32_t bits, bool m, int lane)
{
    std::uint64_t peers = match_lds(l.tab, key & (kMatchSlots - 1), m, lane);
    for (std::uint32_t b = 5; b < bits; ++b) {
        const bool bit = ((key >> b) & 1u) != 0;
        const std::uint64_t ones = __ballot(bit);
        peers &= bit ? ones : ~ones;
    }
    return peers;
}

// Every lane's transfer time; `same` (wave-uniform): the modeled lanes move
// the same byte count, whose time is kept from step to step (x_bytes, x_ps).
__device__ __forceinline__ std::uint64_t plain_xfer(const KArgs& a, const PlainRec& d, bool m,
                                                    std::uint64_t active, std::uint32_t& x_bytes,
                                                    std::uint64_t& x_ps, bool& same)
{
    if (a.transfer_page != 0) {
        same = true;
        if (x_bytes == 0) {
            x_bytes = 1;
            x_ps = xfer_ps(a, 1ull << a.page_shift);
        }
        return x_ps;
    }
    const std::uint32_t b0 = static_cast<std::uint32_t>(__builtin_amdgcn_readlane(
        static_cast<int>(d.bytes), __ffsll(static_cast<long long>(active)) - 1));
    same = __ballot(m && d.bytes != b0) == 0;
    if (same) {
        if (b0 != x_bytes) {
            x_bytes = b0;
            x_ps = xfer_ps(a, b0);
        }
        return x_ps;
    }
    return m ? a.xfer_q * ((static_cast<std::uint64_t>(d.bytes) * a.xfer_num + a.xfer_den - 1) /
                           a.xfer_den)
             : 0ull;
}

// A step's lanes that continue their neighbour's line at its issue time: what
// weight and KV streams are made of (k_summary batches them).
__device__ __forceinline__ std::uint32_t plain_continues(const uint4& x, const uint4& y)
{
    const std::uint32_t pa = dpp32<0x138, 0xF>(x.x), pt = dpp32<0x138, 0xF>(y.x);
    return static_cast<std::uint32_t>(__popcll(__ballot(pa + x.z == x.x && pt == y.x)));
}

// Steps of mostly continuing lines that make a tile k_summary's: the pass
// stops at the second one it meets.
constexpr std::uint32_t kStreamLanes = 32;
constexpr int kStreamSteps = 2;
// steps in flight: 4 KiB a wave in either form
template <bool kPacked>
constexpr int kPlainPipe = kPacked ? 4 : 2;

// The summary pass of scattered records: one wave per tile, the outputs of
// k_summary (without step descriptors, which only k_apply reads).  kAll: every
// tile is taken (short runs, where one launch counts more than a tile's steps).
template <bool kPacked, bool kAll>
__global__ __launch_bounds__(64) __attribute__((amdgpu_waves_per_eu(6)))
void k_plain_summary(KArgs a, const void* rec, std::size_t n, std::uint64_t base_ps,
                     PlaneSum* psum, MaskWord* tmask, ChanSum* csum, std::uint64_t* tile_count)
{
    extern __shared__ std::uint64_t sm[];
    const int lane = threadIdx.x;
    const std::size_t tile = blockIdx.x;
    const std::size_t begin = tile * a.tile;
    const std::size_t end = begin + a.tile < n ? begin + a.tile : n;
    stamp_start(a, 0);
    using Pipe = std::conditional_t<kPacked, PackedPipeT<kPlainPipe<kPacked>>,
                                    RecordPipeT<kPlainPipe<kPacked>>>;
    Pipe pipe;
    pipe.issue(rec, begin, end, lane);
    std::uint64_t last_issue = base_ps;
    if (begin > 0) {
        last_issue = base_ps + (kPacked ? (static_cast<const hbf_record16*>(rec)[begin - 1].issue_op &
                                           ((1ull << 56) - 1))
                                        : static_cast<const hbf_record32*>(rec)[begin - 1].issue_ps);
    }
    const std::uint32_t rpp = plane_slots(a);
    const PlainLds l = plain_layout(a, sm, rpp + 2ull * a.Rc);
    // Per plane 18 bytes: the map's B; its A as counts (senses, programs in
    // the high half); the last page; and 1 + the tile's first record there, read
    // again at the end for its page and issue time.  (33 bytes, as k_summary
    // keeps them, left nine waves per CU at 512 planes instead of fifteen.)
    std::uint64_t* p_rB = l.w64;
    std::uint64_t* c_A = p_rB + rpp;
    std::uint64_t* c_B = c_A + a.Rc;
    std::uint32_t* p_n = l.w32;
    std::uint32_t* p_l1 = p_n + rpp;
    std::uint16_t* p_f = reinterpret_cast<std::uint16_t*>(p_l1 + rpp);
    plain_load(a, l, lane);
    for (std::uint32_t r = lane; r < rpp; r += kWave) {
        p_rB[r] = 0;
        p_n[r] = 0;
        p_l1[r] = 0;
        p_f[r] = 0;
    }
    for (std::uint32_t r = lane; r < a.Rc; r += kWave) {
        c_A[r] = 0;
        c_B[r] = 0;
    }
    __syncthreads();
    const std::uint64_t lt = lanemask_lt(lane);
    std::uint64_t modeled = 0, x_ps = 0;
    std::uint32_t x_bytes = 0;
    bool disorder = false;
    int streams = 0;
    constexpr std::size_t kSpan = static_cast<std::size_t>(kPlainPipe<kPacked>) * kWave;
    for (std::size_t g = begin; g < end; g += kSpan) {
        pipe.advance(rec, g + kSpan, end, lane);
        const std::size_t gend = g + kSpan < end ? g + kSpan : end;
        for (std::size_t s = g; s < gend; s += kWave) {
            typename Pipe::Step st;
            pipe.take(st);
            uint4 x, y;
            step_records(st, lane, x, y);
            const bool valid = s + lane < end;
            if (!kAll) {
                streams += plain_continues(x, y) >= kStreamLanes ? 1 : 0;
                if (streams >= kStreamSteps) {
                    if (lane == 0) {
                        a.tile_split[tile] = 0;
                    }
                    return;  // k_summary takes the tile
                }
            }
            const PlainRec d = plain_record(a, l, x, y, valid, base_ps);
            {
                const std::uint64_t prev = prev_lane64(d.issue);
                const bool back = valid && d.issue < (lane == 0 ? last_issue : prev);
                disorder = disorder || __ballot(back) != 0;
                const std::uint64_t vmask = __ballot(valid);  // lanes 0 .. k
                last_issue = readlane64(d.issue, 63 - __clzll(static_cast<long long>(vmask)));
            }
            const bool m = d.cls == kClsModeled;
            const std::uint64_t active = __ballot(m);
            if (active == 0) {
                continue;
            }
            modeled += __popcll(active);
            bool same = false;
            const std::uint64_t xfer = plain_xfer(a, d, m, active, x_bytes, x_ps, same);
            const std::uint64_t pp = plain_match(l, d.plane, a.pbits, m, lane);
            const std::uint64_t pc = plain_match(l, d.chan, a.cbits, m, lane);
            const std::uint32_t pk = pslot(d.plane);
            const std::uint32_t f1 = m ? p_f[pk] : 0u;
            const std::uint64_t below = pp & lt;
            std::uint32_t prev1 = static_cast<std::uint32_t>(__shfl(
                static_cast<int>(d.page1),
                m && below != 0 ? 63 - __clzll(static_cast<long long>(below)) : lane));
            const bool lead = m && below == 0;
            if (lead) {
                prev1 = p_l1[pk];
            }
            const bool tfirst = lead && f1 == 0;
            const bool hit = a.slots != 0 && prev1 == d.page1;
            const StepCounts sc = count_services(m && !tfirst, d.bits, hit);
            // Per group of lanes on one plane, (A, B) becomes (A + S, max(B +
            // S, issue_k + S_k) over its lanes k), with S the service of all
            // of them and S_k that of lane k and later: the group's last lane
            // adds S, then every lane joins its own term (a wave's LDS
            // operations complete in issue order).  The tile's first record on
            // a plane is kept apart, its hit not known yet.
            const std::uint64_t from = count_service(a, sc, pp & ~lt);
            if (tfirst) {
                p_f[pk] = static_cast<std::uint16_t>(s + lane - begin + 1);
            }
            if (m && (pp >> lane) == 1ull) {
                const std::uint32_t senses = static_cast<std::uint32_t>(__popcll(pp & sc.miss));
                const std::uint32_t programs = static_cast<std::uint32_t>(__popcll(pp & sc.prog));
                (void)__hip_atomic_fetch_add(&p_n[pk], senses | (programs << 16), __ATOMIC_RELAXED,
                                             __HIP_MEMORY_SCOPE_WORKGROUP);
                lds_add(&p_rB[pk], senses * a.read_ps + programs * a.program_ps);
                p_l1[pk] = d.page1;
            }
            if (m && !tfirst) {
                lds_max(&p_rB[pk], d.issue + from);
            }
            // channels likewise
            std::uint64_t Sc, after;
            if (same) {
                const auto times = [&](std::uint64_t lanes) {
                    return static_cast<std::uint64_t>(
                               static_cast<std::uint32_t>(__popcll(lanes))) * xfer;
                };
                Sc = times(pc);
                after = times(pc & ~lt);
            } else {
                // different byte counts: sums along the group by pointer jumping
                Sc = m ? xfer : 0ull;
                std::uint64_t unused = 0;
                group_scan(Sc, unused, m && (pc & lt) != 0
                                           ? 63 - __clzll(static_cast<long long>(pc & lt))
                                           : -1, lane);
                const std::uint64_t upto = Sc;
                Sc = shfl64(Sc, m ? 63 - __clzll(static_cast<long long>(pc)) : lane);
                after = Sc - upto + xfer;
            }
            if (m && (pc >> lane) == 1ull) {
                lds_add(&c_A[d.chan], Sc);
                lds_add(&c_B[d.chan], Sc);
            }
            if (m) {
                lds_max(&c_B[d.chan], d.issue + after);
            }
        }
    }
    if (lane == 0) {
        if (disorder && a.disorder != nullptr) {
            *a.disorder = 1u;
        }
        a.tile_split[tile] = kTilePlain;
        tile_count[tile] = modeled;
    }
    __syncthreads();
    // the touched planes' summaries, packed in plane order, as k_summary's
    PlaneSum* ps = psum + tile * a.Rp;
    MaskWord* tm = tmask + tile * mask_words(a);
    std::uint32_t count = 0;
    for (std::uint32_t r0 = 0; r0 < a.Rp; r0 += kWave) {
        const std::uint32_t r = r0 + lane;
        const std::uint32_t k = pslot(r);
        const std::uint32_t f = r < a.Rp ? p_f[k] : 0u;
        const bool touched = f != 0;
        const std::uint64_t bits = __ballot(touched);
        if (lane == 0) {
            tm[r0 / kWave] = MaskWord{bits, count, 0};
        }
        uint4 x = make_uint4(0, 0, 0, 0), y = x;
        if (touched) {
            const std::size_t i = begin + f - 1;
            if constexpr (kPacked) {
                unpack16(static_cast<const uint4*>(rec)[i], x, y);
            } else {
                load_record(static_cast<const hbf_record32*>(rec), i, x, y);
            }
        }
        const PlainRec d = plain_record(a, l, x, y, touched, base_ps);
        if (touched) {
            PlaneSum v;
            v.fpage1 = d.page1;
            v.fissue = d.issue;
            v.rA = (p_n[k] & 0xffffu) * a.read_ps + (p_n[k] >> 16) * a.program_ps;
            v.rB = p_rB[k];
            v.lpage1 = p_l1[k];
            v.fcls = d.bits;
            v.pad = 0;
            ps[count + __popcll(bits & lt)] = v;
        }
        count += static_cast<std::uint32_t>(__popcll(bits));
    }
    ChanSum* cs = csum + tile * a.Rc;
    for (std::uint32_t r = lane; r < a.Rc; r += kWave) {
        cs[r] = ChanSum{c_A[r], c_B[r]};
    }
}

// The apply pass over the tiles k_plain_summary took.
template <bool kPacked, bool kAll>
__global__ __launch_bounds__(64) __attribute__((amdgpu_waves_per_eu(4)))
void k_plain_apply(KArgs a, const void* rec, std::size_t n, std::uint64_t base_ps,
                   const PlaneCarry* pcarry, const MaskWord* tmask, const std::uint64_t* ccarry,
                   std::uint64_t* completion, std::uint8_t* status, DevReport* tile_rep)
{
    extern __shared__ std::uint64_t sm[];
    stamp_start(a, 2);
    if ((a.disorder != nullptr && *a.disorder != 0u) ||
        (!kAll && a.tile_split[blockIdx.x] != kTilePlain)) {
        return;
    }
    const int lane = threadIdx.x;
    const std::size_t tile = blockIdx.x;
    const std::size_t begin = tile * a.tile;
    const std::size_t end = begin + a.tile < n ? begin + a.tile : n;
    using Pipe = std::conditional_t<kPacked, PackedPipeT<kPlainPipe<kPacked>>,
                                    RecordPipeT<kPlainPipe<kPacked>>>;
    Pipe pipe;
    pipe.issue(rec, begin, end, lane);
    const PlainLds l = plain_layout(a, sm, static_cast<std::size_t>(a.Rp) + a.Rc);
    std::uint64_t* p_busy = l.w64;
    std::uint64_t* c_busy = p_busy + a.Rp;
    std::uint32_t* p_tag = l.w32;
    load_plane_carry<4>(a, tmask, pcarry, tile, p_busy, p_tag, lane);
    load_chan_carry(a, ccarry, tile, c_busy, lane);
    plain_load(a, l, lane);
    __syncthreads();
    const std::uint64_t lt = lanemask_lt(lane);
    std::uint64_t x_ps = 0, mk = 0, lat_lo = 0, lat_hi = 0, lat_max = 0, svc_sum = 0;
    std::uint32_t x_bytes = 0;
    // wave-uniform counts
    std::uint32_t n_mod = 0, n_byp = 0, n_uns = 0, n_rd = 0, n_hit = 0, n_prog = 0;
    constexpr std::size_t kSpan = static_cast<std::size_t>(kPlainPipe<kPacked>) * kWave;
    for (std::size_t g = begin; g < end; g += kSpan) {
        pipe.advance(rec, g + kSpan, end, lane);
        const std::size_t gend = g + kSpan < end ? g + kSpan : end;
        for (std::size_t s = g; s < gend; s += kWave) {
            typename Pipe::Step sr;
            pipe.take(sr);
            uint4 x, y;
            step_records(sr, lane, x, y);
            const std::size_t i = s + lane;
            const bool valid = i < end;
            const PlainRec d = plain_record(a, l, x, y, valid, base_ps);
            const bool m = d.cls == kClsModeled;
            const std::uint64_t active = __ballot(m);
            std::uint32_t st = d.cls;
            std::uint64_t done = d.cls == kClsBypass ? d.issue : ~0ull;
            if (active != 0) {
                bool same = false;
                const std::uint64_t xfer = plain_xfer(a, d, m, active, x_bytes, x_ps, same);
                const std::uint64_t pp = plain_match(l, d.plane, a.pbits, m, lane);
                const std::uint64_t pc = plain_match(l, d.chan, a.cbits, m, lane);
                const std::uint64_t below = pp & lt, cbelow = pc & lt;
                const int ppred =
                    m && below != 0 ? 63 - __clzll(static_cast<long long>(below)) : -1;
                const int cpred =
                    m && cbelow != 0 ? 63 - __clzll(static_cast<long long>(cbelow)) : -1;
                const std::uint64_t pbusy = m ? p_busy[d.plane] : 0ull;
                const std::uint64_t cbusy = m ? c_busy[d.chan] : 0ull;
                std::uint32_t prev1 = static_cast<std::uint32_t>(
                    __shfl(static_cast<int>(d.page1), ppred < 0 ? lane : ppred));
                if (m && ppred < 0) {
                    prev1 = p_tag[d.plane];
                }
                const bool hit = a.slots != 0 && m && prev1 == d.page1;
                const StepCounts sc = count_services(m, d.bits, hit);
                const std::uint64_t svc = count_service(a, sc, 1ull << lane);
                const std::uint64_t origin =
                    readlane64(d.issue, __ffsll(static_cast<long long>(active)) - 1);
                const std::uint64_t most =
                    static_cast<std::uint64_t>(static_cast<std::uint32_t>(
                        __popcll(sc.miss))) * a.read_ps +
                    static_cast<std::uint64_t>(static_cast<std::uint32_t>(
                        __popcll(sc.prog))) * a.program_ps;
                std::uint64_t pd, cd;
                if (same && most < (1ull << 30) && xfer < (1ull << 24) &&
                    __ballot(m && d.issue - origin >= (1ull << 30)) == 0) {
                    // lane i of a group completes at max(busy, max over k <= i
                    // of (issue_k - E_k)) + E_i + its service, with E the
                    // service of the group's lanes before: where no lane's
                    // issue time passes busy + E the maximum is busy, else it
                    // is a prefix maximum of issue - E, in 32 bits from the
                    // step's first issue time
                    const std::uint32_t Ep =
                        static_cast<std::uint32_t>(count_service(a, sc, below));
                    const std::uint32_t x32 = static_cast<std::uint32_t>(xfer);
                    const std::uint32_t Ec = x32 * static_cast<std::uint32_t>(__popcll(cbelow));
                    const bool wp = a.contention != 0 &&
                                    __ballot(m && d.issue > pbusy + Ep) != 0;
                    const bool wc = __ballot(m && d.issue > cbusy + Ec) != 0;
                    std::uint64_t tp = pbusy, tc = cbusy;
                    if (wp || wc) {
                        const std::uint32_t rel =
                            m ? static_cast<std::uint32_t>(d.issue - origin) : 0u;
                        const std::uint32_t most32 = static_cast<std::uint32_t>(most);
                        const std::uint32_t c64 = x32 * 64u;
                        std::uint32_t vp = rel + most32 - Ep, vc = rel + c64 - Ec;
                        group_prefix_max(vp, wp ? ppred : -1, vc, wc ? cpred : -1, lane);
                        // (issue - E may lie below zero where busy is the
                        // maximum: compared before the offset is taken off)
                        if (wp) {
                            tp = origin + vp > pbusy + most32 ? origin + vp - most32 : pbusy;
                        }
                        if (wc) {
                            tc = origin + vc > cbusy + c64 ? origin + vc - c64 : cbusy;
                        }
                    }
                    pd = a.contention != 0 ? tp + Ep + svc : d.issue + svc;
                    cd = tc + Ec + xfer;
                } else {
                    std::uint64_t Ap = m ? svc : 0ull, Bp = m ? d.issue + svc : 0ull;
                    std::uint64_t Ac = m ? xfer : 0ull, Bc = m ? d.issue + xfer : 0ull;
                    if (a.contention != 0) {
                        group_scan(Ap, Bp, ppred, lane);
                    }
                    group_scan(Ac, Bc, cpred, lane);
                    pd = a.contention != 0 ? umax64(pbusy + Ap, Bp) : d.issue + svc;
                    cd = umax64(cbusy + Ac, Bc);
                }
                if (m && (pp >> lane) == 1ull) {
                    if (a.contention != 0) {
                        p_busy[d.plane] = pd;
                    }
                    p_tag[d.plane] = d.page1;
                }
                if (m && (pc >> lane) == 1ull) {
                    c_busy[d.chan] = cd;
                }
                const bool write = (d.bits & 1u) != 0;
                n_mod += static_cast<std::uint32_t>(__popcll(active));
                n_rd += static_cast<std::uint32_t>(__popcll(__ballot(m && !write)));
                n_hit += static_cast<std::uint32_t>(__popcll(__ballot(hit && !write)));
                n_prog += static_cast<std::uint32_t>(__popcll(__ballot(m && write && svc != 0)));
                if (m) {
                    done = umax64(pd, cd);
                    st |= write ? (svc != 0 ? 16u : 0u) : (hit ? 4u : 0u);
                    mk = umax64(mk, done);
                    const std::uint64_t lat = done - d.issue;
                    add128(lat_lo, lat_hi, lat);
                    lat_max = umax64(lat_max, lat);
                    svc_sum += umax64(svc, xfer);
                }
            }
            const std::uint64_t byp = __ballot(d.cls == kClsBypass);
            const std::uint64_t uns = __ballot(d.cls == kClsUnsupported);
            n_byp += static_cast<std::uint32_t>(__popcll(byp));
            n_uns += static_cast<std::uint32_t>(__popcll(uns));
            if (valid) {
                put_done(&completion[i], done);
                if (status != nullptr) {
                    status[i] = static_cast<std::uint8_t>(st);
                }
            }
        }
    }
    // 128-bit latency sum: the high words, then the low words with carries
    std::uint64_t hi = wave_sum(lat_hi), carry = 0, lo = lat_lo;
    for (int o = 32; o > 0; o >>= 1) {
        const std::uint64_t other = shfl64(lo, lane ^ o);
        const std::uint64_t oc = shfl64(carry, lane ^ o);
        const std::uint64_t sum = lo + other;
        carry = carry + oc + (sum < lo ? 1u : 0u);
        lo = sum;
    }
    hi += carry;
    const std::uint64_t vals[14] = {end - begin, n_mod, n_byp, n_uns, n_rd,
                                    n_mod - n_rd, n_hit, n_prog, 0ull, wave_max(mk),
                                    lo, hi, wave_max(lat_max), wave_sum(svc_sum)};
    if (lane < 14) {
        unsigned long long out = 0;
#pragma unroll
        for (int k = 0; k < 14; ++k) {
            out = lane == k ? vals[k] : out;
        }
        tile_rep[tile].v[lane] = out;
    }
}

// Report reduction: each block folds a run of tile reports; the last block to
// finish folds their partials and writes the result to pinned host memory
// (two launches and a copy took 8-16 us).  A block's 256 threads are 16
// streams x 16 words (the 14 report words, the carry out of the 128-bit
// latency sum, padding); sums and maxima are exact in any order.
constexpr int kRepWords = 16;
constexpr int kRepCarry = 14;
constexpr int kRepParts = 256;
constexpr std::size_t kRepRun = 128;  // tile reports per block at least: one round of loads

// The burst state before a tile of the empirical model, and the modeled
// records before it.
struct alignas(16) EmpState {
    std::uint64_t key;
    std::uint64_t seq;
    std::uint32_t run, valid;
    std::uint32_t pad[2];
};

// What a run leaves for the host, in pinned memory: the last kernel writes it
// there (a copy command behind the kernels took another 4 us).
struct HostOut {
    DevReport rep;
    std::uint64_t back;      // some record's issue time went back
    std::uint64_t stamp[4];  // starts of the passes, and of the report
    EmpState fin;            // the empirical model's burst state after the run
};

__device__ __forceinline__ void rep_join(int f, std::uint64_t& acc, std::uint64_t& carry,
                                         std::uint64_t v, std::uint64_t vcarry)
{
    if (f == R_MAKESPAN || f == R_LAT_MAX) {
        acc = umax64(acc, v);
    } else if (f == R_LAT_LO) {
        const std::uint64_t s2 = acc + v;
        carry += vcarry + (s2 < acc ? 1u : 0u);
        acc = s2;
    } else {
        acc += v;
    }
}

// Folds entries [lo, hi) of kIn words (14: tile reports, kRepWords: partials)
// into acc_sh[0] and carry_sh[0].  kShared: the entries were written by other
// blocks of this launch.
template <int kIn, bool kShared>
__device__ __forceinline__ void rep_fold(const std::uint64_t* in, std::size_t lo, std::size_t hi,
                                         std::uint64_t (*acc_sh)[kRepWords],
                                         std::uint64_t* carry_sh)
{
    const int f = threadIdx.x % kRepWords;
    const int stream = threadIdx.x / kRepWords;
    const auto load = [&](std::size_t w) {
        if constexpr (kShared) {
            return __hip_atomic_load(&in[w], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        } else {
            return in[w];
        }
    };
    std::uint64_t acc = 0, carry = 0;
    // kBatch entries per stream are loaded before any is joined (one memory
    // round trip per batch, not per entry); entries past `hi` read as 0,
    // which every field's join leaves unchanged
    constexpr int kBatch = 8;
    for (std::size_t i0 = lo + stream; i0 < hi; i0 += 16 * kBatch) {
        std::uint64_t v[kBatch], vc[kBatch];
#pragma unroll
        for (int k = 0; k < kBatch; ++k) {
            const std::size_t i = i0 + 16 * static_cast<std::size_t>(k);
            v[k] = i < hi && f < kIn ? load(i * kIn + f) : 0ull;
            // a partial's carry word travels with its latency word
            vc[k] = i < hi && kIn == kRepWords && f == R_LAT_LO ? load(i * kIn + kRepCarry) : 0ull;
        }
#pragma unroll
        for (int k = 0; k < kBatch; ++k) {
            rep_join(f, acc, carry, f == kRepCarry ? 0ull : v[k], vc[k]);
        }
    }
    __syncthreads();
    acc_sh[stream][f] = acc;
    if (f == R_LAT_LO) {
        carry_sh[stream] = carry;
    }
    __syncthreads();
    for (int half = 8; half > 0; half >>= 1) {
        if (stream < half) {
            std::uint64_t a0 = acc_sh[stream][f];
            std::uint64_t c0 = f == R_LAT_LO ? carry_sh[stream] : 0ull;
            rep_join(f, a0, c0, acc_sh[stream + half][f],
                     f == R_LAT_LO ? carry_sh[stream + half] : 0ull);
            acc_sh[stream][f] = a0;
            if (f == R_LAT_LO) {
                carry_sh[stream] = c0;
            }
        }
        __syncthreads();
    }
}

// Block b folds tile reports [b * per, (b + 1) * per); `done` counts the
// blocks that have (0 between launches).  The disorder flag travels with the
// report and is cleared for the next run.
__global__ __launch_bounds__(256) void k_report(const DevReport* tile_rep, std::size_t count,
                                                std::size_t per, std::uint64_t* parts,
                                                std::uint32_t* done, std::uint32_t* disorder,
                                                const std::uint64_t* stamp, HostOut* out)
{
    __shared__ std::uint64_t acc_sh[16][kRepWords];
    __shared__ std::uint64_t carry_sh[16];
    __shared__ std::uint32_t last;
    const std::uint64_t start = static_cast<std::uint64_t>(wall_clock64());
    const int t = threadIdx.x;
    const std::size_t lo = static_cast<std::size_t>(blockIdx.x) * per;
    const std::size_t hi = lo + per < count ? lo + per : count;
    rep_fold<14, false>(reinterpret_cast<const std::uint64_t*>(tile_rep), lo, hi, acc_sh,
                        carry_sh);
    if (gridDim.x > 1) {
        if (t < kRepWords) {
            parts[static_cast<std::size_t>(blockIdx.x) * kRepWords + t] =
                t == kRepCarry ? carry_sh[0] : acc_sh[0][t];
            __threadfence();
        }
        __syncthreads();
        if (t == 0) {
            last = atomicAdd(done, 1u) + 1 == gridDim.x ? 1u : 0u;
        }
        __syncthreads();
        if (last == 0) {
            return;
        }
        __threadfence();
        rep_fold<kRepWords, true>(parts, 0, gridDim.x, acc_sh, carry_sh);
        if (t == 0) {
            *done = 0;
        }
    }
    if (t < 14) {
        out->rep.v[t] = t == R_LAT_HI ? acc_sh[0][t] + carry_sh[0] : acc_sh[0][t];
    } else if (t == 14) {
        out->back = disorder != nullptr ? *disorder : 0u;
        if (disorder != nullptr) {
            *disorder = 0u;
        }
    } else if (t < 18) {
        out->stamp[t - 15] = stamp[t - 15];
    } else if (t == 18) {
        out->stamp[3] = start;
    }
}

// ---- warp grouping (hbf_device.cu:1223-1231) ----------------------------
//
// The lanes of one warp instruction are consecutive records with one nonzero
// group id (flags bits 32-63); among them, modeled records with the same
// (range, media page) share the media request of the first.  k_lead marks
// every other such record with how far back that first record is; the
// summary and apply passes then time only the requests, and k_follow gives
// each marked record its request's completion.

constexpr std::size_t kLeadSpan = 1024;  // records per wave of k_lead
constexpr unsigned kFollowBlocks = 8192;

// One wave per kLeadSpan records; the 64 records before them are decoded
// too, as history.  Two windows of 64 records live in LDS: record i in slot
// ((i >> 6) & 1) * 64 + (i & 63).  A group of more than 64 records or with
// two issue times sets *err (the run is refused before anything is timed).
__global__ __launch_bounds__(64) void k_lead(KArgs a, const hbf_record32* rec, std::size_t n,
                                             std::uint8_t* lead, std::uint32_t* err)
{
    extern __shared__ std::uint64_t sm[];
    std::uint64_t* fence = sm;
    __shared__ std::uint64_t s_issue[2 * kWave];
    __shared__ std::uint64_t s_page1[2 * kWave];  // media page + 1; 0: not modeled
    __shared__ std::uint32_t s_group[2 * kWave];
    __shared__ std::uint32_t s_range[2 * kWave];
    const int lane = threadIdx.x;
    const std::size_t begin = static_cast<std::size_t>(blockIdx.x) * kLeadSpan;
    const std::size_t end = begin + kLeadSpan < n ? begin + kLeadSpan : n;
    load_fences(a, fence, lane);
    __syncthreads();
    RangeCache rc = empty_cache();
    std::uint32_t bad = 0;
    for (std::size_t s = begin >= kWave ? begin - kWave : begin; s < end; s += kWave) {
        const std::size_t i = s + lane;
        const int slot = static_cast<int>(((i >> 6) & 1u) * kWave + (i & 63u));
        std::uint32_t g = 0, rid = 0;
        std::uint64_t issue = 0, page1 = 0;
        if (i < end) {
            uint4 x, y;
            load_record(rec, i, x, y);
            g = y.w;
            issue = y.x | (static_cast<std::uint64_t>(y.y) << 32);
            if (g != 0) {
                const Dec d = decode<false>(a, fence, rc, x, y, 0);
                if (d.cls == kClsModeled) {
                    page1 = d.page1;
                    rid = d.range_id;
                }
            }
        }
        s_group[slot] = g;
        s_issue[slot] = issue;
        s_page1[slot] = page1;
        s_range[slot] = rid;
        __syncthreads();
        if (s >= begin && i < end) {
            std::uint32_t back = 0;
            if (g != 0) {
                // the group's earlier records: at most 63, all in the two windows
                for (std::size_t t = 1; t <= kWave && t <= i; ++t) {
                    const std::size_t j = i - t;
                    const int sj = static_cast<int>(((j >> 6) & 1u) * kWave + (j & 63u));
                    if (s_group[sj] != g) {
                        break;
                    }
                    if (t == kWave || s_issue[sj] != issue) {
                        bad = 1;
                        break;
                    }
                    if (page1 != 0 && s_page1[sj] == page1 && s_range[sj] == rid) {
                        back = static_cast<std::uint32_t>(t);
                    }
                }
            }
            lead[i] = static_cast<std::uint8_t>(back);
        }
        __syncthreads();
    }
    if (__ballot(bad != 0) != 0 && lane == 0) {
        atomicMax(err, 1u);
    }
}

// Each marked record takes its request's completion (final once k_apply
// has run: a request is never itself marked) and status kStGrouped, and is
// counted into frep: records that joined, reads, writes, makespan, latency
// sum (low, high words), latency maximum.
__global__ __launch_bounds__(256) void k_follow(const hbf_record32* rec, std::size_t n,
                                                std::uint64_t base_ps, const std::uint8_t* lead,
                                                std::uint64_t* comp, std::uint8_t* status,
                                                unsigned long long* frep)
{
    std::uint64_t cnt = 0, rd = 0, wr = 0, mk = 0, lo = 0, hi = 0, mx = 0;
    const std::size_t stride = static_cast<std::size_t>(gridDim.x) * blockDim.x;
    for (std::size_t i = static_cast<std::size_t>(blockIdx.x) * blockDim.x + threadIdx.x; i < n;
         i += stride) {
        const std::uint32_t back = lead[i];
        if (back == 0) {
            continue;
        }
        const std::uint64_t done = comp[i - back];
        comp[i] = done;
        if (status != nullptr) {
            status[i] = kStGrouped;
        }
        const uint4 y = reinterpret_cast<const uint4*>(rec + i)[1];
        const std::uint64_t issue = base_ps + (y.x | (static_cast<std::uint64_t>(y.y) << 32));
        const std::uint32_t op = y.z & 0xffu;
        ++cnt;
        rd += op == 0 ? 1u : 0u;
        wr += op == 1 ? 1u : 0u;
        mk = umax64(mk, done);
        const std::uint64_t lat = done - issue;
        const std::uint64_t l2 = lo + lat;
        hi += l2 < lo ? 1u : 0u;
        lo = l2;
        mx = umax64(mx, lat);
    }
    const std::uint64_t total = wave_sum(cnt);
    if (total == 0) {
        return;  // wave-uniform
    }
    // 128-bit latency sum across the wave: high words, then low words with
    // their carries
    hi = wave_sum(hi);
    std::uint64_t carry = 0;
    for (int o = 32; o > 0; o >>= 1) {
        const std::uint64_t other = shfl64(lo, threadIdx.x ^ o);
        const std::uint64_t oc = shfl64(carry, threadIdx.x ^ o);
        const std::uint64_t sum = lo + other;
        carry = carry + oc + (sum < lo ? 1u : 0u);
        lo = sum;
    }
    hi += carry;
    rd = wave_sum(rd);
    wr = wave_sum(wr);
    mk = wave_max(mk);
    mx = wave_max(mx);
    if ((threadIdx.x & 63u) == 0) {
        atomicAdd(&frep[0], static_cast<unsigned long long>(total));
        atomicAdd(&frep[1], static_cast<unsigned long long>(rd));
        atomicAdd(&frep[2], static_cast<unsigned long long>(wr));
        atomicMax(&frep[3], static_cast<unsigned long long>(mk));
        const unsigned long long old = atomicAdd(&frep[4], static_cast<unsigned long long>(lo));
        hi += old + lo < old ? 1u : 0u;
        atomicAdd(&frep[5], static_cast<unsigned long long>(hi));
        atomicMax(&frep[6], static_cast<unsigned long long>(mx));
    }
}

// Folds `ntiles` (at least 1) tile reports into *out; parts: kRepParts *
// kRepWords words, done: a zero word.  disorder may be null.
void launch_report(hipStream_t stream, const DevReport* tile_rep, std::size_t ntiles,
                   std::uint64_t* parts, std::uint32_t* done, std::uint32_t* disorder,
                   const std::uint64_t* stamp, HostOut* out)
{
    const std::size_t per = std::max(kRepRun, (ntiles + kRepParts - 1) / kRepParts);
    hipLaunchKernelGGL(k_report, dim3(static_cast<unsigned>((ntiles + per - 1) / per)), dim3(256),
                       0, stream, tile_rep, ntiles, per, parts, done, disorder, stamp, out);
}

}  // namespace

// ------------------------------------------------------------------------
// Scratch of the entry point that allocates nothing
// (hbfsim_amd_run_device_packed_noalloc): one array per device, part of the
// code object, so the entry point never calls an allocator.  Host code uses
// only the device address hipGetSymbolAddress returns for it (kept per device
// in noalloc_scratch below), never the array's name.  Every call on a device
// shares it; calls that overlap on one device race.  Nothing in it needs to
// start at zero: each kernel of a run writes every scratch word it reads
// before reading it, as with the engine's own reused scratch.

}  // namespace hbfamd

static __device__ __align__(256) unsigned char scratch[hbfamd::kNoAllocScratchBytes];

namespace hbfamd {

namespace {

constexpr int kMaxDevices = 64;
std::mutex g_noalloc_mu;
void* g_noalloc_ptr[kMaxDevices] = {};

// Looks the array's device address up once per device; `device` must be
// current.  Returns nullptr when the lookup fails.
void* noalloc_scratch(int device)
{
    if (device < 0 || device >= kMaxDevices) {
        return nullptr;
    }
    std::lock_guard<std::mutex> lock(g_noalloc_mu);
    if (g_noalloc_ptr[device] == nullptr) {
        void* ptr = nullptr;
        if (hipGetSymbolAddress(&ptr, HIP_SYMBOL(scratch)) == hipSuccess) {
            g_noalloc_ptr[device] = ptr;
        }
    }
    return g_noalloc_ptr[device];
}

}  // namespace

// ------------------------------------------------------------------------
// host side

struct engine {
    engine_config cfg;
    int device{0};
    KArgs args{};
    // ranges
    std::vector<range_rec> ranges;
    bool ranges_dirty{true};
    bool ranges_pack{false};  // the range table fits its packed form in LDS
    // The arrays of one purpose lie in one allocation (an engine's first run
    // spent most of its time in some thirty small ones).
    unsigned char* range_block{nullptr};
    unsigned char* state_block{nullptr};
    std::size_t state_bytes{0};  // of state_block, that a reset clears
    unsigned char* tile_block{nullptr};
    unsigned char* desc_block{nullptr};
    std::uint64_t* d_r_base{nullptr};
    std::uint64_t* d_r_length{nullptr};
    std::uint64_t* d_r_offset{nullptr};
    std::uint32_t* d_r_meta{nullptr};
    std::uint32_t* d_r_id{nullptr};
    std::size_t range_cap{0};
    // persistent state
    std::uint64_t* d_pbusy{nullptr};
    std::uint64_t* d_ptag{nullptr};
    std::uint64_t* d_cbusy{nullptr};
    std::uint64_t* d_ptot{nullptr};
    std::uint64_t* d_ctot{nullptr};
    std::uint64_t* d_seq{nullptr};
    HostOut* h_out{nullptr};    // pinned; written by a run's last kernel
    std::uint32_t* d_done{nullptr};   // blocks of the report reduction that are done
    std::uint64_t* d_stamp{nullptr};  // the passes' start times (KArgs::stamp)
    double ms_per_tick{0};
    std::uint64_t* d_rep_parts{nullptr};  // report partials
    std::uint32_t* d_disorder{nullptr};  // a run's records went back in time
    // scratch
    std::size_t tile_cap{0};
    PlaneSum* d_psum{nullptr};
    MaskWord* d_tmask{nullptr};  // touched planes per tile
    ChanSum* d_csum{nullptr};
    PlaneCarry* d_pcarry{nullptr};
    std::uint64_t* d_ccarry{nullptr};
    std::uint64_t* d_tcount{nullptr};
    std::uint64_t* d_tseq{nullptr};
    PlaneSum* d_gpsum{nullptr};
    ChanSum* d_gcsum{nullptr};
    PlaneCarry* d_gpcarry{nullptr};
    std::uint64_t* d_gccarry{nullptr};
    std::uint64_t* d_gcount{nullptr};
    std::uint64_t* d_gseq{nullptr};
    DevReport* d_tile_rep{nullptr};
    std::uint8_t* d_tsplit{nullptr};  // per tile: holds a split step
    StepDesc* d_desc{nullptr};  // per-step descriptors (records / 64)
    std::uint32_t* d_desc_rid{nullptr};  // and their range ids (hybrid runs)
    SplitDesc* d_desc_split{nullptr};    // and split steps' second runs
    std::size_t desc_cap{0};
    float last_ms[3]{0, 0, 0};
    std::uint64_t burst{0};
    std::uint64_t* d_emp_svc{nullptr};  // the empirical model's services by run
    // the last completed run's modeled records and page-register hits: a
    // large stream with few hits is mostly general steps, and its next run
    // takes the four-wave apply pass (results are the same either way)
    std::uint64_t last_modeled{0};
    std::uint64_t last_hits{0};
    int last_apply_waves{0};  // waves per SIMD the last run's apply pass was built for
    // the last run's tiles, and which passes were launched over them (with both,
    // d_tsplit says which took a tile; a run that reuses d_tsplit sets these too)
    enum class Passes { none, batched, scattered, both } last_passes{Passes::none};
    std::size_t last_tiles{0};
};

// Where one run of the main pipeline keeps its per-tile and per-group
// summaries, carries, tile reports and step descriptors.
struct RunScratch {
    PlaneSum* psum;
    MaskWord* tmask;
    ChanSum* csum;
    PlaneCarry* pcarry;
    std::uint64_t* ccarry;
    std::uint64_t* tcount;
    std::uint64_t* tseq;
    PlaneSum* gpsum;
    ChanSum* gcsum;
    PlaneCarry* gpcarry;
    std::uint64_t* gccarry;
    std::uint64_t* gcount;
    std::uint64_t* gseq;
    DevReport* tile_rep;
    StepDesc* desc;
    std::uint8_t* tsplit;
};

namespace {

// Lays a run's scratch out in one buffer from `base`, each piece 256-byte
// aligned: per tile the plane summaries and carries (64 B per plane), the
// mask words (16 B per 64 planes), the channel summaries and carries (24 B
// per channel), two counters, a tile report (128 B) and a split flag (1 B);
// per group of kGroup
// tiles the same summaries and carries; and 16 B of step descriptor per 64
// records.  Returns the bytes needed; with base == nullptr it only counts.
std::size_t carve_scratch(const KArgs& a, std::size_t ntiles, std::size_t nsteps,
                          unsigned char* base, RunScratch* s)
{
    std::size_t off = 0;
    auto take = [&](auto*& ptr, std::size_t count) {
        using T = std::remove_reference_t<decltype(*ptr)>;
        off = (off + 255) & ~static_cast<std::size_t>(255);
        ptr = base != nullptr ? reinterpret_cast<T*>(base + off) : nullptr;
        off += sizeof(T) * (count == 0 ? 1 : count);
    };
    RunScratch t{};
    const std::size_t rp = a.Rp, rc = a.Rc;
    const std::size_t groups = (ntiles + kGroup - 1) / kGroup;
    take(t.psum, ntiles * rp);
    take(t.tmask, ntiles * mask_words(a));
    take(t.csum, ntiles * rc);
    take(t.pcarry, ntiles * rp);
    take(t.ccarry, ntiles * rc);
    take(t.tcount, ntiles);
    take(t.tseq, ntiles);
    take(t.gpsum, groups * rp);
    take(t.gcsum, groups * rc);
    take(t.gpcarry, groups * rp);
    take(t.gccarry, groups * rc);
    take(t.gcount, groups);
    take(t.gseq, groups);
    take(t.tile_rep, ntiles);
    take(t.desc, nsteps);
    take(t.tsplit, ntiles);
    if (s != nullptr) {
        *s = t;
    }
    return off;
}

}  // namespace

namespace {

int hip_status(hipError_t e) { return e == hipSuccess ? HBFSIM_OK : HBFSIM_CUDA_ERROR; }

template <typename T>
void hfree(T*& p)
{
    if (p != nullptr) {
        (void)hipFree(p);
        p = nullptr;
    }
}

template <typename T>
hipError_t halloc(T*& p, std::size_t count)
{
    const std::size_t bytes = sizeof(T) * (count == 0 ? 1 : count);
    hipError_t err = hipMalloc(reinterpret_cast<void**>(&p), bytes);
    if (err != hipSuccess) {
        (void)hipGetLastError();
        scratch_trim();  // idle scratch goes first
        err = hipMalloc(reinterpret_cast<void**>(&p), bytes);
    }
    return err;
}

// An array of a block laid out by a ScratchPlan.
template <typename T>
void place(T*& p, unsigned char* block, std::size_t at)
{
    p = reinterpret_cast<T*>(block + at);
}

std::uint32_t bits_for(std::uint32_t n)
{
    std::uint32_t b = 0;
    while ((1u << b) < n) {
        ++b;
    }
    return b;
}

bool is_pow2(std::uint64_t v) { return v != 0 && (v & (v - 1)) == 0; }

std::uint32_t log2u(std::uint64_t v)
{
    std::uint32_t b = 0;
    while ((1ull << b) < v) {
        ++b;
    }
    return b;
}

void free_scratch(engine* e)
{
    hfree(e->tile_block);
    hfree(e->desc_block);
    e->desc_cap = 0;
    e->tile_cap = 0;
}

int ensure_scratch(engine* e, std::size_t ntiles)
{
    if (ntiles <= e->tile_cap) {
        return HBFSIM_OK;
    }
    free_scratch(e);
    // an eighth of headroom, so that batches a little larger than the last
    // do not reallocate (freeing device memory synchronises the device)
    const std::size_t cap = std::max<std::size_t>(ntiles + ntiles / 8, 16);
    const std::size_t rp = e->args.Rp, rc = e->args.Rc;
    const std::size_t gcap = (cap + kGroup - 1) / kGroup;
    ScratchPlan plan;
    const std::size_t psum = plan.add<PlaneSum>(cap * rp);
    const std::size_t tmask = plan.add<MaskWord>(cap * mask_words(e->args));
    const std::size_t csum = plan.add<ChanSum>(cap * rc);
    const std::size_t pcarry = plan.add<PlaneCarry>(cap * rp);
    const std::size_t ccarry = plan.add<std::uint64_t>(cap * rc);
    const std::size_t tcount = plan.add<std::uint64_t>(cap);
    const std::size_t tseq = plan.add<std::uint64_t>(cap);
    const std::size_t gpsum = plan.add<PlaneSum>(gcap * rp);
    const std::size_t gcsum = plan.add<ChanSum>(gcap * rc);
    const std::size_t gpcarry = plan.add<PlaneCarry>(gcap * rp);
    const std::size_t gccarry = plan.add<std::uint64_t>(gcap * rc);
    const std::size_t gcount = plan.add<std::uint64_t>(gcap);
    const std::size_t gseq = plan.add<std::uint64_t>(gcap);
    const std::size_t tile_rep = plan.add<DevReport>(cap);
    const std::size_t tsplit = plan.add<std::uint8_t>(cap);
    if (halloc(e->tile_block, plan.bytes) != hipSuccess) {
        free_scratch(e);
        return HBFSIM_CUDA_ERROR;
    }
    place(e->d_psum, e->tile_block, psum);
    place(e->d_tmask, e->tile_block, tmask);
    place(e->d_csum, e->tile_block, csum);
    place(e->d_pcarry, e->tile_block, pcarry);
    place(e->d_ccarry, e->tile_block, ccarry);
    place(e->d_tcount, e->tile_block, tcount);
    place(e->d_tseq, e->tile_block, tseq);
    place(e->d_gpsum, e->tile_block, gpsum);
    place(e->d_gcsum, e->tile_block, gcsum);
    place(e->d_gpcarry, e->tile_block, gpcarry);
    place(e->d_gccarry, e->tile_block, gccarry);
    place(e->d_gcount, e->tile_block, gcount);
    place(e->d_gseq, e->tile_block, gseq);
    place(e->d_tile_rep, e->tile_block, tile_rep);
    place(e->d_tsplit, e->tile_block, tsplit);
    e->tile_cap = cap;
    return HBFSIM_OK;
}

int upload_ranges(engine* e, hipStream_t stream)
{
    const std::size_t count = e->ranges.size();
    if (count > e->range_cap || e->range_block == nullptr) {
        hfree(e->range_block);
        const std::size_t cap = std::max<std::size_t>(count, 64);
        ScratchPlan plan;
        const std::size_t rbase = plan.add<std::uint64_t>(cap);
        const std::size_t rlength = plan.add<std::uint64_t>(cap);
        const std::size_t roffset = plan.add<std::uint64_t>(cap);
        const std::size_t rmeta = plan.add<std::uint32_t>(cap);
        const std::size_t rid = plan.add<std::uint32_t>(cap);
        if (halloc(e->range_block, plan.bytes) != hipSuccess) {
            return HBFSIM_CUDA_ERROR;
        }
        place(e->d_r_base, e->range_block, rbase);
        place(e->d_r_length, e->range_block, rlength);
        place(e->d_r_offset, e->range_block, roffset);
        place(e->d_r_meta, e->range_block, rmeta);
        place(e->d_r_id, e->range_block, rid);
        e->range_cap = cap;
    }
    std::vector<std::uint64_t> base(count), length(count), offset(count);
    std::vector<std::uint32_t> meta(count), id(count);
    for (std::size_t i = 0; i < count; ++i) {
        base[i] = e->ranges[i].base;
        length[i] = e->ranges[i].length;
        offset[i] = e->ranges[i].file_offset;
        meta[i] = (e->ranges[i].mode & 0xffu) | (e->ranges[i].permissions << 8);
        id[i] = e->ranges[i].range_id;
    }
    if (count != 0) {
        hipError_t err = hipMemcpyAsync(e->d_r_base, base.data(), count * 8,
                                        hipMemcpyHostToDevice, stream);
        if (err == hipSuccess)
            err = hipMemcpyAsync(e->d_r_length, length.data(), count * 8, hipMemcpyHostToDevice,
                                 stream);
        if (err == hipSuccess)
            err = hipMemcpyAsync(e->d_r_offset, offset.data(), count * 8, hipMemcpyHostToDevice,
                                 stream);
        if (err == hipSuccess)
            err = hipMemcpyAsync(e->d_r_meta, meta.data(), count * 4, hipMemcpyHostToDevice,
                                 stream);
        if (err == hipSuccess)
            err = hipMemcpyAsync(e->d_r_id, id.data(), count * 4, hipMemcpyHostToDevice, stream);
        if (err == hipSuccess) err = hipStreamSynchronize(stream);
        if (err != hipSuccess) {
            return HBFSIM_CUDA_ERROR;
        }
    }
    KArgs& a = e->args;
    a.r_base = e->d_r_base;
    a.r_length = e->d_r_length;
    a.r_file_offset = e->d_r_offset;
    a.r_meta = e->d_r_meta;
    a.r_id = e->d_r_id;
    a.r_count = static_cast<std::uint32_t>(count);
    a.r_stride = count <= kMaxFences ? 1u
                                     : static_cast<std::uint32_t>((count + kMaxFences - 1) /
                                                                  kMaxFences);
    a.r_nfence = count == 0 ? 0u
                            : static_cast<std::uint32_t>((count + a.r_stride - 1) / a.r_stride);
    // the packed form of the table in LDS (store_ranges)
    e->ranges_pack = count != 0 && count <= kLdsRanges;
    for (std::size_t i = 0; i < count; ++i) {
        e->ranges_pack = e->ranges_pack && length[i] <= kRangeLenMask &&
                         (offset[i] >> a.page_shift) <= 0xffffffffull &&
                         (offset[i] & ((1ull << a.page_shift) - 1)) == 0 &&
                         (e->ranges[i].mode == 1 || e->ranges[i].mode == 2) &&
                         e->ranges[i].permissions <= 0xfu;
    }
    e->ranges_dirty = false;
    return HBFSIM_OK;
}

// Modeled records per (window of issue time, die), for the thermal power
// map.  Each block histograms a chunk in LDS over the windows it spans and
// flushes the non-zero bins with global atomics.
constexpr std::uint32_t kCountChunk = 4096;
constexpr std::uint32_t kCountBins = 4096;

__global__ __launch_bounds__(256) void k_window_counts(KArgs a, const hbf_record32* rec,
                                                       std::size_t n, std::uint64_t window_ps,
                                                       std::uint64_t windows,
                                                       std::uint32_t ndie,
                                                       std::uint32_t* counts)
{
    extern __shared__ std::uint64_t sm[];
    std::uint64_t* fence = sm;
    std::uint32_t* hist = reinterpret_cast<std::uint32_t*>(fence + a.r_nfence);
    const int tid = threadIdx.x;
    for (std::uint32_t j = tid; j < a.r_nfence; j += blockDim.x) {
        fence[j] = a.r_base[static_cast<std::size_t>(j) * a.r_stride];
    }
    for (std::uint32_t j = tid; j < kCountBins; j += blockDim.x) {
        hist[j] = 0;
    }
    __syncthreads();
    const std::size_t begin = static_cast<std::size_t>(blockIdx.x) * kCountChunk;
    const std::size_t end = begin + kCountChunk < n ? begin + kCountChunk : n;
    const std::uint64_t w0 = rec[begin].issue_ps / window_ps;
    RangeCache rc = empty_cache();
    for (std::size_t i = begin + tid; i < end; i += blockDim.x) {
        uint4 x, y;
        load_record(rec, i, x, y);
        const Dec d = decode<false>(a, fence, rc, x, y, 0);
        if (d.cls != kClsModeled) {
            continue;
        }
        const std::uint64_t w = d.issue / window_ps;
        if (w >= windows) {
            continue;
        }
        const std::uint32_t die = d.plane / a.P;
        const std::uint64_t bin = (w - w0) * ndie + die;
        if (w >= w0 && bin < kCountBins) {
            atomicAdd(&hist[bin], 1u);
        } else {
            atomicAdd(&counts[w * ndie + die], 1u);
        }
    }
    __syncthreads();
    for (std::uint32_t j = tid; j < kCountBins; j += blockDim.x) {
        if (hist[j] != 0) {
            atomicAdd(&counts[w0 * ndie + j], hist[j]);
        }
    }
}

// ---- empirical single-tail model (hbf_device.cu:796-881) -----------------
// One busy-until tail; a read's service is the cumulative curve's increment
// at its burst run (streak of consecutive ascending pages with one
// operation, capped at 1023, hbf_device.cuh:1031-1080), a write's is tPROG.
//
//   k_emp_tile<false>  per tile of 2,048 records: where its streaks start,
//                      and the tail's (max,+) map of the records after the
//                      first streak (whose runs do not depend on what came
//                      before the tile);
//   k_emp_chain        the burst state and sequence before every tile;
//   k_emp_lead         per tile, the map of the first streak from that
//                      state, joined to the rest: only those records are
//                      read again (24 of 2,048 at a mean streak of 24);
//   k_emp_tail         the tail before every tile, and the engine state;
//   k_emp_tile<true>   completions, status and the tile report.
//
// A page and its operation are one number, key = page << 1 | op, so that a
// record continues the streak when its key is the last one plus two.  Both
// tile passes load record-per-lane, decode once and hand the records to the
// threads eight in a row through LDS: a thread walks its records serially
// (a wave scan per 64 records would spend six rounds of 64-bit moves on
// each), and runs follow from two 32-bit scans over the threads (records so
// far, and where the current streak started).  6M records: 104 us for the two
// tile passes (43 + 61 us, 4.5 and 4.0 TB/s of records and results), against
// 545 us for three when every pass gathered 16 records per thread at a
// 512-byte stride, decoded them up to three times and folded the tile report
// in one thread.
constexpr int kEmpThreads = 256;
constexpr int kEmpWaves = kEmpThreads / kWave;
constexpr int kEmpPer = 8;
constexpr std::uint32_t kEmpTile = kEmpThreads * kEmpPer;
constexpr std::uint64_t kRunCap = 1023;
// LDS slot of a tile's record: one pad per eight, so that threads reading
// their eight in a row spread over the banks.
constexpr std::uint32_t kEmpSlots = kEmpTile + kEmpTile / kEmpPer;
__device__ __forceinline__ std::uint32_t emp_slot(std::uint32_t i) { return i + i / kEmpPer; }

struct alignas(16) TailMap {
    std::uint64_t A, B;  // b -> max(b + A, B)
};

// A tile's streaks.
struct alignas(16) EmpTile {
    std::uint64_t fkey, lkey;  // first and last modeled record
    std::uint32_t count;       // modeled records (0: the rest is unset)
    std::uint32_t tail;        // length of the last streak, at most kRunCap
    std::uint32_t all;         // 1: one streak
    std::uint32_t lead_end;    // records up to the first streak's last one
};

__device__ __forceinline__ TailMap tail_compose(const TailMap& f, const TailMap& s)
{
    return TailMap{f.A + s.A, umax64(f.B + s.A, s.B)};
}

__device__ __forceinline__ std::uint32_t wave_prefix_add32(std::uint32_t v)
{
    v += dpp32<0x111, 0xF>(v);
    v += dpp32<0x112, 0xF>(v);
    v += dpp32<0x114, 0xF>(v);
    v += dpp32<0x118, 0xF>(v);
    v += dpp32<0x142, 0xA>(v);
    v += dpp32<0x143, 0xC>(v);
    return v;
}

__device__ __forceinline__ std::uint64_t emp_service(std::uint64_t key, std::uint64_t run,
                                                     const std::uint64_t* svc_ps,
                                                     std::uint64_t program_ps)
{
    return (key & 1u) != 0 ? program_ps : svc_ps[run < kRunCap ? run : kRunCap];
}

// Media pages are below 2^52 here (4-KiB pages), far below the reference's
// limit on burst pages (hbf_device.cuh:1031-1080), so every modeled record
// takes part in streaks and key, operation and class share one word.
template <bool kApply>
__global__ __launch_bounds__(kEmpThreads) __attribute__((amdgpu_waves_per_eu(4)))
void k_emp_tile(KArgs a, const hbf_record32* rec, std::size_t n, std::uint64_t base_ps,
                const std::uint64_t* svc_ps, std::uint64_t program_ps, EmpTile* tiles,
                TailMap* maps, const EmpState* tile_in, const std::uint64_t* tile_tail,
                std::uint64_t* completion, std::uint8_t* status, DevReport* tile_rep)
{
    stamp_start(a, kApply ? 2 : 0);
    extern __shared__ std::uint64_t fence[];
    __shared__ ulonglong2 sh[kEmpSlots];  // issue (then completion), key << 2 | class
    __shared__ std::uint32_t w_count[kEmpWaves], w_start[kEmpWaves], w_lead[kEmpWaves];
    __shared__ std::uint64_t w_last[kEmpWaves];
    __shared__ TailMap w_map[kEmpWaves];
    // hybrid runs: the records' range ids (the sampler's key)
    std::uint32_t* rid = reinterpret_cast<std::uint32_t*>(fence + a.r_nfence);
    const int tid = threadIdx.x, lane = tid & (kWave - 1), wave = tid / kWave;
    const std::size_t begin = static_cast<std::size_t>(blockIdx.x) * kEmpTile;
    uint4 x[kEmpPer], y[kEmpPer];
#pragma unroll
    for (int k = 0; k < kEmpPer; ++k) {
        const std::size_t i = begin + static_cast<std::size_t>(k) * kEmpThreads + tid;
        load_record(rec, i < n ? i : n - 1, x[k], y[k]);
    }
    std::uint64_t before = base_ps;  // the issue time of the record before the tile
    if (!kApply && a.disorder != nullptr && tid == 0 && begin != 0) {
        before = base_ps + rec[begin - 1].issue_ps;
    }
    for (std::uint32_t j = tid; j < a.r_nfence; j += kEmpThreads) {
        fence[j] = a.r_base[static_cast<std::size_t>(j) * a.r_stride];
    }
    __syncthreads();
    RangeCache rc = empty_cache();
#pragma unroll
    for (int k = 0; k < kEmpPer; ++k) {
        const std::uint32_t at = k * kEmpThreads + tid;
        const Dec d = decode<false>(a, fence, rc, x[k], y[k], base_ps);
        const std::uint32_t cls = begin + at < n ? d.cls : kClsInvalid;
        const std::uint64_t key =
            cls == kClsModeled ? ((d.page1 - 1) << 1) | dec_op(d.bits) : 0ull;
        sh[emp_slot(at)] = make_ulonglong2(d.issue, (key << 2) | cls);
        if (kApply && a.hybrid) {
            rid[emp_slot(at)] = d.range_id;
        }
    }
    __syncthreads();
    // this thread's eight records: modeled ones, first and last key, and the
    // place (among them) where the last streak that starts inside starts
    const std::uint32_t own = tid * kEmpPer;
    std::uint64_t issue[kEmpPer], key[kEmpPer];
    std::uint32_t cls[kEmpPer];
#pragma unroll
    for (int k = 0; k < kEmpPer; ++k) {
        const ulonglong2 v = sh[emp_slot(own + k)];
        issue[k] = v.x;
        key[k] = v.y >> 2;
        cls[k] = static_cast<std::uint32_t>(v.y) & 3u;
    }
    if (!kApply && a.disorder != nullptr) {
        std::uint64_t prev = tid == 0 ? before : sh[emp_slot(own - 1)].x;
        bool back = false;
#pragma unroll
        for (int k = 0; k < kEmpPer; ++k) {
            back = back || (cls[k] != kClsInvalid && issue[k] - base_ps < prev - base_ps);
            prev = issue[k];
        }
        if (__ballot(back) != 0 && lane == 0) {
            *a.disorder = 1u;
        }
    }
    std::uint32_t mine = 0, brk = 0;  // brk: 1 + the last inner start, 0: none
    std::uint64_t first = 0, last = 0;
#pragma unroll
    for (int k = 0; k < kEmpPer; ++k) {
        if (cls[k] == kClsModeled) {
            if (mine == 0) {
                first = key[k];
            } else if (key[k] != last + 2) {
                brk = mine + 1;
            }
            last = key[k];
            ++mine;
        }
    }
    const std::uint32_t incl = wave_prefix_add32(mine);
    const std::uint64_t has = __ballot(mine != 0);
    if (lane == kWave - 1) {
        w_count[wave] = incl;
    }
    if (has != 0 && lane == 63 - __clzll(static_cast<long long>(has))) {
        w_last[wave] = last;
    }
    __syncthreads();
    // records before this thread, and the key before its first one
    std::uint32_t c = incl - mine;
    std::uint64_t prev_key = 0;
#pragma unroll
    for (int w = 0; w < kEmpWaves; ++w) {
        if (w < wave) {
            c += w_count[w];
            prev_key = w_count[w] != 0 ? w_last[w] : prev_key;
        }
    }
    {
        const std::uint64_t lower = has & lanemask_lt(lane);
        const std::uint64_t pk =
            shfl64(last, lower != 0 ? 63 - __clzll(static_cast<long long>(lower)) : lane);
        prev_key = lower != 0 ? pk : prev_key;
    }
    // where the streak starts that reaches this thread's end: 1 + the place
    // among the tile's modeled records (1: the tile's first streak)
    const bool cont = c != 0 && mine != 0 && first == prev_key + 2;
    std::uint32_t start = 0;
    if (mine != 0) {
        start = brk != 0 ? c + brk : (cont ? 0u : c + 1);
    }
    const std::uint32_t smax = wave_prefix_max32(start);
    if (lane == kWave - 1) {
        w_start[wave] = smax;
    }
    __syncthreads();
    std::uint32_t s_in = static_cast<std::uint32_t>(__shfl_up(static_cast<int>(smax), 1));
    s_in = lane == 0 ? 0u : s_in;
    std::uint32_t s_all = 0, total = 0;
#pragma unroll
    for (int w = 0; w < kEmpWaves; ++w) {
        if (w < wave && w_start[w] > s_in) {
            s_in = w_start[w];
        }
        s_all = w_start[w] > s_all ? w_start[w] : s_all;
        total += w_count[w];
    }
    // services and this thread's map
    EmpState in{};
    std::uint64_t r0 = 0;  // the first streak's run before the tile
    if (kApply) {
        in = tile_in[blockIdx.x];
        if (c == 0 && mine != 0) {
            // the tile's first modeled record decides
            r0 = in.valid != 0 && first == in.key + 2 ? in.run : 0;
            w_lead[0] = static_cast<std::uint32_t>(r0);
        }
        __syncthreads();
        r0 = total != 0 ? w_lead[0] : 0;
    }
    std::uint64_t svc[kEmpPer];
    TailMap m{0, 0};
    std::uint32_t lead_end = 0;
    {
        std::uint32_t at = c, s = s_in;
        std::uint64_t pk = prev_key;
#pragma unroll
        for (int k = 0; k < kEmpPer; ++k) {
            svc[k] = 0;
            if (cls[k] != kClsModeled) {
                continue;
            }
            if (at == 0 || key[k] != pk + 2) {
                s = at + 1;
            }
            pk = key[k];
            ++at;
            const std::uint64_t run = at - s + 1 + (s == 1 ? r0 : 0);
            if (!kApply && s == 1) {
                lead_end = own + k + 1;  // left to k_emp_lead
                continue;
            }
            svc[k] = emp_service(key[k], run, svc_ps, program_ps);
            m = tail_compose(m, TailMap{svc[k], issue[k] + svc[k]});
        }
    }
    TailMap scan = m;
    wave_scan(scan.A, scan.B);
    if (lane == kWave - 1) {
        w_map[wave] = scan;
    }
    if (!kApply) {
        lead_end = wave_prefix_max32(lead_end);
        if (lane == kWave - 1) {
            w_lead[wave] = lead_end;
        }
        __syncthreads();
        if (tid == kEmpThreads - 1) {
            TailMap all = w_map[0];
            std::uint32_t le = w_lead[0];
#pragma unroll
            for (int w = 1; w < kEmpWaves; ++w) {
                all = tail_compose(all, w_map[w]);
                le = w_lead[w] > le ? w_lead[w] : le;
            }
            maps[blockIdx.x] = all;
            EmpTile& t = tiles[blockIdx.x];
            t.lkey = mine != 0 ? last : prev_key;
            t.count = total;
            const std::uint32_t len = total != 0 ? total - s_all + 1 : 0u;
            t.tail = len < kRunCap ? len : static_cast<std::uint32_t>(kRunCap);
            t.all = s_all == 1 ? 1u : 0u;
            t.lead_end = le;
        }
        if (c == 0 && mine != 0) {
            tiles[blockIdx.x].fkey = first;
        }
        return;
    }
    __syncthreads();
    // the tail before this thread's records
    TailMap ex;
    ex.A = shfl64(scan.A, lane == 0 ? 0 : lane - 1);
    ex.B = shfl64(scan.B, lane == 0 ? 0 : lane - 1);
    ex = lane == 0 ? TailMap{0, 0} : ex;
    std::uint64_t tail = tile_tail[blockIdx.x];
#pragma unroll
    for (int w = 0; w < kEmpWaves; ++w) {
        if (w < wave) {
            tail = umax64(tail + w_map[w].A, w_map[w].B);
        }
    }
    tail = umax64(tail + ex.A, ex.B);
    // counts of at most 2,048 a tile, 12 bits each: modeled, bypass,
    // unsupported, reads, sampled
    std::uint64_t counts = 0, makespan = 0, lat_lo = 0, lat_hi = 0, lat_max = 0, service = 0;
    std::uint64_t seq = in.seq + c;
#pragma unroll
    for (int k = 0; k < kEmpPer; ++k) {
        std::uint32_t sb = cls[k];
        std::uint64_t done = issue[k];
        if (cls[k] == kClsBypass) {
            counts += 1ull << 12;
        } else if (cls[k] == kClsUnsupported) {
            done = ~0ull;
            counts += 1ull << 24;
        } else if (cls[k] == kClsModeled) {
            const std::uint32_t op = static_cast<std::uint32_t>(key[k]) & 1u;
            if (a.hybrid) {
                const std::uint64_t h =
                    ((key[k] >> 1) << a.page_shift) ^
                    (static_cast<std::uint64_t>(rid[emp_slot(own + k)]) << 32) ^ op;
                if (seq < a.hybrid_warmup ||
                    (a.hybrid_threshold != 0 && mix64(seq ^ h) <= a.hybrid_threshold)) {
                    sb |= 8u;
                    counts += 1ull << 48;
                }
            }
            ++seq;
            done = umax64(tail, issue[k]) + svc[k];
            tail = done;
            counts += 1ull + (op == 0 ? 1ull << 36 : 0ull);
            makespan = umax64(makespan, done);
            const std::uint64_t lat = done - issue[k];
            lat_lo += lat;
            lat_hi += lat_lo < lat ? 1u : 0u;
            lat_max = umax64(lat_max, lat);
            service += svc[k];
        }
        sh[emp_slot(own + k)] = make_ulonglong2(done, sb);
    }
    __syncthreads();
#pragma unroll
    for (int k = 0; k < kEmpPer; ++k) {
        const std::uint32_t at = k * kEmpThreads + tid;
        const std::size_t i = begin + at;
        if (i < n) {
            const ulonglong2 v = sh[emp_slot(at)];
            put_done(&completion[i], v.x);
            if (status != nullptr) {
                status[i] = static_cast<std::uint8_t>(v.y);
            }
        }
    }
    // tile report: wave reductions, then the four waves by one thread
#pragma unroll
    for (int o = kWave / 2; o > 0; o >>= 1) {
        counts += shfl64(counts, lane ^ o);
        makespan = umax64(makespan, shfl64(makespan, lane ^ o));
        lat_max = umax64(lat_max, shfl64(lat_max, lane ^ o));
        service += shfl64(service, lane ^ o);
        const std::uint64_t lo = shfl64(lat_lo, lane ^ o);
        lat_hi += shfl64(lat_hi, lane ^ o);
        lat_lo += lo;
        lat_hi += lat_lo < lo ? 1u : 0u;
    }
    __shared__ std::uint64_t part[kEmpWaves][6];
    if (lane == 0) {
        part[wave][0] = counts;
        part[wave][1] = makespan;
        part[wave][2] = lat_max;
        part[wave][3] = service;
        part[wave][4] = lat_lo;
        part[wave][5] = lat_hi;
    }
    __syncthreads();
    if (tid == 0) {
        for (int w = 1; w < kEmpWaves; ++w) {
            counts += part[w][0];
            makespan = umax64(makespan, part[w][1]);
            lat_max = umax64(lat_max, part[w][2]);
            service += part[w][3];
            lat_lo += part[w][4];
            lat_hi += part[w][5] + (lat_lo < part[w][4] ? 1u : 0u);
        }
        const auto count = [&](int k) { return (counts >> (12 * k)) & 0xfffull; };
        DevReport out{};
        out.v[R_RECORDS] = n - begin < kEmpTile ? n - begin : kEmpTile;
        out.v[R_MODELED] = count(0);
        out.v[R_BYPASS] = count(1);
        out.v[R_UNSUPPORTED] = count(2);
        out.v[R_READS] = count(3);
        out.v[R_WRITES] = count(0) - count(3);
        out.v[R_HYBRID] = count(4);
        out.v[R_MAKESPAN] = makespan;
        out.v[R_LAT_LO] = lat_lo;
        out.v[R_LAT_HI] = lat_hi;
        out.v[R_LAT_MAX] = lat_max;
        out.v[R_SERVICE] = service;
        tile_rep[blockIdx.x] = out;
    }
}

// Streaks of a range of tiles, for the chain's scan.
struct EmpSpan {
    std::uint64_t fkey, lkey, count;
    std::uint32_t tail, all;
};

// a then b
__device__ __forceinline__ EmpSpan span_join(const EmpSpan& a, const EmpSpan& b)
{
    if (b.count == 0) {
        return a;
    }
    if (a.count == 0) {
        return b;
    }
    const bool cont = b.fkey == a.lkey + 2;
    const std::uint32_t sum = a.tail + b.tail;
    EmpSpan r;
    r.fkey = a.fkey;
    r.lkey = b.lkey;
    r.count = a.count + b.count;
    r.tail = !(b.all && cont) ? b.tail
                              : (sum < kRunCap ? sum : static_cast<std::uint32_t>(kRunCap));
    r.all = a.all && b.all && cont ? 1u : 0u;
    return r;
}

__device__ __forceinline__ EmpState span_apply(const EmpState& st, const EmpSpan& s)
{
    if (s.count == 0) {
        return st;
    }
    const bool cont = st.valid != 0 && s.fkey == st.key + 2;
    const std::uint32_t sum = st.run + s.tail;
    EmpState r{};
    r.key = s.lkey;
    r.valid = 1;
    r.run = !(s.all && cont) ? s.tail
                             : (sum < kRunCap ? sum : static_cast<std::uint32_t>(kRunCap));
    r.seq = st.seq + s.count;
    return r;
}

__device__ __forceinline__ EmpSpan span_of(const EmpTile& t)
{
    EmpSpan s;
    s.count = t.count;
    s.fkey = t.fkey;
    s.lkey = t.lkey;
    s.tail = t.tail;
    s.all = t.all;
    return s;
}

constexpr int kEmpChain = 1024;

// One block, a run of tiles per thread: the burst state and sequence before
// every tile, and after the last (`fin`).
__global__ __launch_bounds__(kEmpChain) void k_emp_chain(KArgs a, const EmpTile* tiles, std::size_t ntiles,
                                                         EmpState init, const std::uint64_t* seq0,
                                                         EmpState* tile_in,
                                                         std::uint64_t* fin_seq, EmpState* fin)
{
    __shared__ EmpSpan w_span[kEmpChain / kWave];
    stamp_start(a, 1);
    const int lane = threadIdx.x & (kWave - 1), wave = threadIdx.x / kWave;
    const std::size_t per = (ntiles + kEmpChain - 1) / kEmpChain;
    const std::size_t b = threadIdx.x * per;
    const std::size_t e = b + per < ntiles ? b + per : ntiles;
    EmpSpan s{};
    for (std::size_t t = b; t < e; ++t) {
        s = span_join(s, span_of(tiles[t]));
    }
    for (int o = 1; o < kWave; o <<= 1) {
        const int src = lane >= o ? lane - o : lane;
        EmpSpan p;
        p.fkey = shfl64(s.fkey, src);
        p.lkey = shfl64(s.lkey, src);
        p.count = shfl64(s.count, src);
        p.tail = static_cast<std::uint32_t>(__shfl(static_cast<int>(s.tail), src));
        p.all = static_cast<std::uint32_t>(__shfl(static_cast<int>(s.all), src));
        s = lane >= o ? span_join(p, s) : s;
    }
    if (lane == kWave - 1) {
        w_span[wave] = s;
    }
    const int src = lane == 0 ? 0 : lane - 1;
    EmpSpan ex;
    ex.fkey = shfl64(s.fkey, src);
    ex.lkey = shfl64(s.lkey, src);
    ex.count = shfl64(s.count, src);
    ex.tail = static_cast<std::uint32_t>(__shfl(static_cast<int>(s.tail), src));
    ex.all = static_cast<std::uint32_t>(__shfl(static_cast<int>(s.all), src));
    ex.count = lane == 0 ? 0ull : ex.count;
    __syncthreads();
    init.seq = *seq0;
    EmpState st = init;
    for (int w = 0; w < wave; ++w) {
        st = span_apply(st, w_span[w]);
    }
    st = span_apply(st, ex);
    for (std::size_t t = b; t < e; ++t) {
        tile_in[t] = st;
        st = span_apply(st, span_of(tiles[t]));
    }
    if (e == ntiles && b < e) {
        *fin = st;
        *fin_seq = st.seq;
    }
}

// One wave per tile: the map of the tile's first streak from its incoming
// state, joined to the map of the rest.
__global__ __launch_bounds__(kEmpThreads) void k_emp_lead(KArgs a, const hbf_record32* rec,
                                                          std::size_t n, std::size_t ntiles,
                                                          std::uint64_t base_ps,
                                                          const std::uint64_t* svc_ps,
                                                          std::uint64_t program_ps,
                                                          const EmpTile* tiles,
                                                          const EmpState* tile_in, TailMap* maps)
{
    extern __shared__ std::uint64_t fence[];
    const int lane = threadIdx.x & (kWave - 1);
    for (std::uint32_t j = threadIdx.x; j < a.r_nfence; j += kEmpThreads) {
        fence[j] = a.r_base[static_cast<std::size_t>(j) * a.r_stride];
    }
    __syncthreads();
    const std::size_t t = static_cast<std::size_t>(blockIdx.x) * kEmpWaves + threadIdx.x / kWave;
    if (t >= ntiles) {
        return;
    }
    const EmpTile et = tiles[t];
    if (et.count == 0) {
        return;  // nothing modeled: the rest's map is the identity already
    }
    const EmpState in = tile_in[t];
    std::uint64_t run = in.valid != 0 && et.fkey == in.key + 2 ? in.run : 0;
    const std::size_t begin = t * kEmpTile;
    RangeCache rc = empty_cache();
    TailMap m{0, 0};
    for (std::uint32_t s = 0; s < et.lead_end; s += kWave) {
        TailMap one{0, 0};
        bool modeled = false;
        Dec d = invalid_dec();
        if (s + lane < et.lead_end) {
            uint4 x, y;
            load_record(rec, begin + s + lane, x, y);
            d = decode<false>(a, fence, rc, x, y, base_ps);
            modeled = d.cls == kClsModeled;
        }
        const std::uint64_t mask = __ballot(modeled);
        if (modeled) {
            const std::uint64_t key = ((d.page1 - 1) << 1) | dec_op(d.bits);
            const std::uint64_t svc = emp_service(
                key, run + 1 + __popcll(mask & lanemask_lt(lane)), svc_ps, program_ps);
            one = TailMap{svc, d.issue + svc};
        }
        run += __popcll(mask);
        wave_scan(one.A, one.B);
        m = tail_compose(m, TailMap{readlane64(one.A, 63), readlane64(one.B, 63)});
    }
    if (lane == 0) {
        maps[t] = tail_compose(m, maps[t]);
    }
}

// One block: the tail before every tile.  Unless the stream went back in
// time, also the engine state after the run: tail, sequence and the service
// charged (the maps' sums).
__global__ __launch_bounds__(kEmpChain) void k_emp_tail(const TailMap* maps, std::size_t ntiles,
                                                        const std::uint64_t* fin_seq,
                                                        const std::uint32_t* disorder,
                                                        std::uint64_t* tile_tail,
                                                        std::uint64_t* cursor, std::uint64_t* seq,
                                                        std::uint64_t* total)
{
    __shared__ TailMap w_map[kEmpChain / kWave];
    const int lane = threadIdx.x & (kWave - 1), wave = threadIdx.x / kWave;
    const std::size_t per = (ntiles + kEmpChain - 1) / kEmpChain;
    const std::size_t b = threadIdx.x * per;
    const std::size_t e = b + per < ntiles ? b + per : ntiles;
    const std::uint64_t tail0 = *cursor;
    TailMap m{0, 0};
    for (std::size_t t = b; t < e; ++t) {
        m = tail_compose(m, maps[t]);
    }
    wave_scan(m.A, m.B);
    if (lane == kWave - 1) {
        w_map[wave] = m;
    }
    TailMap ex;
    ex.A = shfl64(m.A, lane == 0 ? 0 : lane - 1);
    ex.B = shfl64(m.B, lane == 0 ? 0 : lane - 1);
    ex = lane == 0 ? TailMap{0, 0} : ex;
    __syncthreads();  // (every thread has read the cursor)
    std::uint64_t g = tail0;
    for (int w = 0; w < wave; ++w) {
        g = umax64(g + w_map[w].A, w_map[w].B);
    }
    g = umax64(g + ex.A, ex.B);
    for (std::size_t t = b; t < e; ++t) {
        tile_tail[t] = g;
        g = umax64(g + maps[t].A, maps[t].B);
    }
    if (threadIdx.x == 0 && (disorder == nullptr || *disorder == 0)) {
        TailMap all{0, 0};
        for (int w = 0; w < kEmpChain / kWave; ++w) {
            all = tail_compose(all, w_map[w]);
        }
        *cursor = umax64(tail0 + all.A, all.B);
        *seq = *fin_seq;
        *total += all.A;
    }
}

// ---- two page registers per plane (device_coalescer.cpp:134-168) ---------
// A miss fills the first empty slot, else slot 0.  Slot 1 is therefore
// written once and then kept, and from then on a read hits when its page is
// slot 1's or the last page other than slot 1's seen on the plane.  Hits do
// not depend on timing, so they come from their own scans and the timing
// pipeline consumes them (kHits):
//   k_k2_first   per plane, the first record (optionally: whose page differs
//                from a given one) -- the fill events before both slots hold
//                a page; only run while some plane has an empty slot;
//   k_k2_hits    one hit byte per record, and per tile and plane the first and
//                the last record on a page other than slot 1's;
//   k_k2_up/mid/down  the carry of that page across tiles; the last level
//                settles each first record's hit, which needs the carry.
struct K2Plane {
    std::uint64_t start3;  // first record index with both slots held
    std::uint64_t miss1, miss2;  // fill events before that (or ~0)
    std::uint32_t t1;      // slot 1's page + 1 from start3 on (0: never)
    std::uint32_t l_init;  // last page other than t1 before the run
};

constexpr std::uint32_t kK2Chunk = 16384;

__global__ __launch_bounds__(256) void k_k2_first(KArgs a, const hbf_record32* rec,
                                                  std::size_t n, std::uint64_t base_ps,
                                                  const std::uint32_t* want,
                                                  const std::uint32_t* differ,
                                                  unsigned long long* first)
{
    extern __shared__ std::uint64_t sm[];
    std::uint64_t* fence = sm;
    unsigned long long* lmin = reinterpret_cast<unsigned long long*>(fence + a.r_nfence);
    for (std::uint32_t j = threadIdx.x; j < a.r_nfence; j += blockDim.x) {
        fence[j] = a.r_base[static_cast<std::size_t>(j) * a.r_stride];
    }
    for (std::uint32_t r = threadIdx.x; r < a.Rp; r += blockDim.x) {
        lmin[r] = ~0ull;
    }
    __syncthreads();
    const std::size_t begin = static_cast<std::size_t>(blockIdx.x) * kK2Chunk;
    const std::size_t end = begin + kK2Chunk < n ? begin + kK2Chunk : n;
    RangeCache rc = empty_cache();
    for (std::size_t i = begin + threadIdx.x; i < end; i += blockDim.x) {
        uint4 x, y;
        load_record(rec, i, x, y);
        const Dec d = decode<false>(a, fence, rc, x, y, base_ps);
        if (d.cls != kClsModeled || !want[d.plane]) {
            continue;
        }
        const std::uint32_t page1 = static_cast<std::uint32_t>(d.page1);
        if (differ[d.plane] != 0 && page1 == differ[d.plane]) {
            continue;
        }
        atomicMin(&lmin[d.plane], static_cast<unsigned long long>(i));
    }
    __syncthreads();
    for (std::uint32_t r = threadIdx.x; r < a.Rp; r += blockDim.x) {
        if (lmin[r] != ~0ull) {
            atomicMin(&first[r], lmin[r]);
        }
    }
}

// Page + 1 of record idx[r] for every plane r (0 when none).
__global__ __launch_bounds__(256) void k_k2_page(KArgs a, const hbf_record32* rec, std::size_t n,
                                                 std::uint64_t base_ps,
                                                 const unsigned long long* idx,
                                                 std::uint32_t* page1)
{
    extern __shared__ std::uint64_t fence[];
    for (std::uint32_t j = threadIdx.x; j < a.r_nfence; j += blockDim.x) {
        fence[j] = a.r_base[static_cast<std::size_t>(j) * a.r_stride];
    }
    __syncthreads();
    for (std::uint32_t r = threadIdx.x; r < a.Rp; r += blockDim.x) {
        std::uint32_t v = 0;
        if (idx[r] < n) {
            RangeCache rc = empty_cache();
            uint4 x, y;
            load_record(rec, idx[r], x, y);
            v = static_cast<std::uint32_t>(decode<false>(a, fence, rc, x, y, base_ps).page1);
        }
        page1[r] = v;
    }
}

// A tile's first record on a plane whose page is not slot 1's: its hit byte is
// settled by k_k2_down.  Valid where tile_last is nonzero.
struct K2First {
    std::uint32_t page1;
    std::uint32_t at;  // index in the tile
};

// The wave of a tile walks its records once.  Only a tile's first record off
// slot 1's page on a plane depends on earlier tiles, so all other hits are
// written here, and the records are read and decoded once instead of by one
// pass for the carry and one for the hits.  Records arrive through the
// pipeline of the timing passes (four steps in flight), and steps of one or
// two linear runs are classified by run: every record of a run after its first
// hits the page the first one left in a register.
// The paged-KV step of 73M records with two registers: 2981 -> 2369 us, of
// which this pass takes 776 (3.1 TB/s).
__global__ __launch_bounds__(64) void k_k2_hits(KArgs a, const hbf_record32* rec, std::size_t n,
                                                std::uint64_t base_ps, const K2Plane* kp,
                                                std::uint32_t* tile_last, K2First* tile_first,
                                                std::uint8_t* hits)
{
    extern __shared__ std::uint64_t sm[];
    std::uint64_t* fence = sm;
    // per 64 planes, those that still fill a slot at or after this tile's start
    std::uint64_t* late = fence + a.r_nfence;
    const std::uint32_t words = (a.Rp + kWave - 1) / kWave;
    std::uint32_t* t1 = reinterpret_cast<std::uint32_t*>(late + words);
    std::uint32_t* last = t1 + a.Rp;
    const int lane = threadIdx.x;
    const std::size_t tile = blockIdx.x;
    const std::size_t begin = tile * a.tile;
    const std::size_t end = begin + a.tile < n ? begin + a.tile : n;
    RecordPipe pipe;
    pipe.issue(rec, begin, end, lane);
    load_fences(a, fence, lane);
    for (std::uint32_t w = 0; w < words; ++w) {
        const std::uint32_t r = w * kWave + static_cast<std::uint32_t>(lane);
        bool l = false;
        if (r < a.Rp) {
            t1[r] = kp[r].t1;
            last[r] = 0;
            l = kp[r].start3 > begin;
        }
        const std::uint64_t m = __ballot(l);
        if (lane == 0) {
            late[w] = m;
        }
    }
    __syncthreads();
    // the hit of a modeled record before both of its plane's slots hold a page
    const auto filling = [&](std::uint32_t plane, std::size_t i, bool hit) {
        if (((late[plane / kWave] >> (plane % kWave)) & 1u) != 0) {
            const K2Plane& k = kp[plane];
            if (i < k.start3) {
                hit = i != k.miss1 && i != k.miss2;
            }
        }
        return hit;
    };
    RangeCache rc = empty_cache();
    RangeCache rcu = empty_cache();  // wave-uniform copy for linear steps
    std::uint32_t lin_miss = 0;
    constexpr std::size_t kSpan = static_cast<std::size_t>(kPipe) * kWave;
    for (std::size_t g = begin; g < end; g += kSpan) {
        pipe.advance(rec, g + kSpan, end, lane);
        const std::size_t gend = g + kSpan < end ? g + kSpan : end;
        for (std::size_t s = g; s < gend; s += kWave) {
            Step32 st;
            pipe.take(st);
            const std::size_t i = s + lane;
            if (lin_miss < kLinGiveUp || (s / kWave) % kLinProbe == 0) {
                LinStep ls;
                const bool lin = detect_step<false, true>(a, fence, rcu, st, base_ps,
                                                          s + kWave <= end, lane, ls);
                lin_miss = lin ? 0u : lin_miss + 1u;
                if (lin) {
                    bool hit = true;
                    std::uint32_t plane = 0;
                    for (std::uint32_t part = 0; part < (ls.k != 0 ? 2u : 1u); ++part) {
                        const std::uint32_t page1 = part == 0 ? ls.page1 : ls.page1b;
                        const std::uint32_t lo = part == 0 ? 0u : ls.k;
                        Dec d;
                        d.plane = 0;
                        d.chan = 0;
                        stripe(a, page1 - 1u, d);
                        if (static_cast<std::uint32_t>(lane) >= lo) {
                            plane = d.plane;
                        }
                        if (page1 == t1[d.plane]) {
                            continue;  // slot 1's page
                        }
                        const std::uint32_t prev1 = last[d.plane];
                        __syncthreads();  // read before it changes
                        if (static_cast<std::uint32_t>(lane) == lo) {
                            hit = prev1 == page1;
                            last[d.plane] = page1;
                            if (prev1 == 0) {
                                tile_first[tile * a.Rp + d.plane] =
                                    K2First{page1, static_cast<std::uint32_t>(i - begin)};
                            }
                        }
                        __syncthreads();
                    }
                    hits[i] = filling(plane, i, hit) ? 1u : 0u;
                    continue;
                }
            }
            const bool valid = i < end;
            uint4 x, y;
            step_records(st, lane, x, y);
            Dec d = invalid_dec();
            if (valid) {
                d = decode<false>(a, fence, rc, x, y, base_ps);
            }
            const bool m = valid && d.cls == kClsModeled;
            const std::uint32_t page1 = static_cast<std::uint32_t>(d.page1);
            const bool nt = m && page1 != t1[d.plane];
            const std::uint64_t active = __ballot(nt);
            bool hit = m && !nt;  // slot 1's page
            if (active != 0) {
                const Group gr = group_by(nt ? d.plane : 0u, a.pbits, nt, active, lane);
                std::uint32_t prev1 = static_cast<std::uint32_t>(
                    __shfl(static_cast<int>(page1), gr.pred < 0 ? lane : gr.pred));
                if (gr.pred < 0) {
                    prev1 = nt ? last[d.plane] : 0u;
                }
                __syncthreads();  // every lane has read `last` before it changes
                if (nt) {
                    hit = prev1 == page1;
                    if (prev1 == 0) {
                        tile_first[tile * a.Rp + d.plane] =
                            K2First{page1, static_cast<std::uint32_t>(i - begin)};
                    }
                    if (lane == gr.last) {
                        last[d.plane] = page1;
                    }
                }
                __syncthreads();
            }
            if (valid) {
                hits[i] = (m ? filling(d.plane, i, hit) : false) ? 1u : 0u;
            }
        }
    }
    __syncthreads();
    for (std::uint32_t r = lane; r < a.Rp; r += kWave) {
        tile_last[tile * a.Rp + r] = last[r];
    }
}

// Level 1: the last nonzero page of each (group of kGroup tiles, plane).
__global__ __launch_bounds__(256) void k_k2_up(KArgs a, std::size_t ntiles, std::size_t ngroups,
                                               const std::uint32_t* tile_last,
                                               std::uint32_t* group_last)
{
    const std::size_t t = blockIdx.x * static_cast<std::size_t>(blockDim.x) + threadIdx.x;
    if (t >= ngroups * a.Rp) {
        return;
    }
    const std::size_t g = t / a.Rp, r = t % a.Rp;
    std::uint32_t v = 0;
    const std::size_t e = (g + 1) * kGroup < ntiles ? (g + 1) * kGroup : ntiles;
    for (std::size_t k = g * kGroup; k < e; ++k) {
        const std::uint32_t x = tile_last[k * a.Rp + r];
        v = x != 0 ? x : v;
    }
    group_last[g * a.Rp + r] = v;
}

// Level 2: per plane, the page before each group, and after the last.
__global__ __launch_bounds__(256) void k_k2_mid(KArgs a, std::size_t ngroups, const K2Plane* kp,
                                                const std::uint32_t* group_last,
                                                std::uint32_t* group_in, std::uint32_t* final_last)
{
    const std::uint32_t r = blockIdx.x * blockDim.x + threadIdx.x;
    if (r >= a.Rp) {
        return;
    }
    std::uint32_t v = kp[r].l_init;
    // sixteen groups' loads in flight together (one at a time the walk of 280
    // groups took 72 us, 22 now)
    constexpr int kAhead = 16;
    for (std::size_t g = 0; g < ngroups; g += kAhead) {
        std::uint32_t x[kAhead];
#pragma unroll
        for (int j = 0; j < kAhead; ++j) {
            x[j] = g + j < ngroups ? group_last[(g + j) * a.Rp + r] : 0u;
        }
#pragma unroll
        for (int j = 0; j < kAhead; ++j) {
            if (g + j < ngroups) {
                group_in[(g + j) * a.Rp + r] = v;
            }
            v = x[j] != 0 ? x[j] : v;
        }
    }
    final_last[r] = v;
}

// Level 3: the page before each tile, which settles the hit of the tile's first
// record on a page other than slot 1's (once both slots hold a page).
__global__ __launch_bounds__(256) void k_k2_down(KArgs a, std::size_t ntiles, std::size_t ngroups,
                                                 const K2Plane* kp,
                                                 const std::uint32_t* tile_last,
                                                 const K2First* tile_first,
                                                 const std::uint32_t* group_in,
                                                 std::uint8_t* hits)
{
    const std::size_t t = blockIdx.x * static_cast<std::size_t>(blockDim.x) + threadIdx.x;
    if (t >= ngroups * a.Rp) {
        return;
    }
    const std::size_t g = t / a.Rp, r = t % a.Rp;
    std::uint32_t v = group_in[g * a.Rp + r];
    const std::uint64_t start3 = kp[r].start3;
    const std::size_t e = (g + 1) * kGroup < ntiles ? (g + 1) * kGroup : ntiles;
    for (std::size_t k = g * kGroup; k < e; ++k) {
        const std::uint32_t x = tile_last[k * a.Rp + r];
        if (x != 0) {
            const K2First f = tile_first[k * a.Rp + r];
            const std::size_t i = k * a.tile + f.at;
            if (i >= start3) {
                hits[i] = f.page1 == v ? 1u : 0u;
            }
            v = x;
        }
    }
}

std::size_t lds_summary(const KArgs& a) { return summary_range_offset(a) + range_lds_bytes(a); }

std::size_t lds_apply(const KArgs& a) { return apply_range_offset(a) + range_lds_bytes(a); }

// The lane-matching tables go where they cost neither per-record pass any
// waves per CU (gfx950: 160 KB of LDS per CU, four SIMDs; both passes run at
// most four waves per SIMD).
constexpr std::size_t kLdsPerCuBytes = 160 * 1024;  // gfx950
constexpr std::size_t kSimdsPerCu = 4;
// the four-wave apply pass is considered from this many records
constexpr std::size_t kWideApplyRecords = std::size_t{1} << 24;
// A workgroup may hold all of it; beyond 64 KB of dynamic LDS a kernel has
// to be allowed the size first (allow_lds).
constexpr std::size_t kLdsPerBlockBytes = 160 * 1024;

// Raises a kernel's dynamic-LDS limit where a launch needs more than the
// default 64 KB (geometries of more than about 1,900 planes).
template <typename F>
hipError_t allow_lds(F* kernel, std::size_t bytes)
{
    if (bytes <= 65536) {
        return hipSuccess;
    }
    return hipFuncSetAttribute(reinterpret_cast<const void*>(kernel),
                               hipFuncAttributeMaxDynamicSharedMemorySize,
                               static_cast<int>(bytes));
}

// Whether the scattered-record passes can take a packed run: power-of-two axes
// (or one plane), the range table in its packed form, no hybrid sampling,
// tiles whose counts fit 16 bits, and their LDS within what a workgroup gets by
// default.
bool plain_run(const KArgs& a, bool ranges_pack)
{
    return ranges_pack && a.hybrid == 0 && (a.flat != 0 || a.pow2 != 0) && a.tile < 65536 &&
           plain_summary_lds(a) <= 65536 && plain_apply_lds(a) <= 65536;
}

// Runs of up to this many records in tiles of at most four steps take the
// scattered-record passes alone, whatever their steps look like: what a run of
// lines costs there is less than the two launches the mixed form adds.
constexpr std::size_t kPlainAlone = std::size_t{1} << 18;

// Whether the scattered-record passes, where they can take a run, take all its
// tiles: short runs, and runs without page registers, whose lines the batched
// passes would take record by record as well (they batch what hits a
// register), at more instructions a step: 67M 32-byte lines 2,512 us with the
// tiles of lines left to them, 2,415 alone (2,466 before there were two pairs
// of passes), packed 2,321 and 2,115.  Flat geometry has one plane: group_by
// sees at once that a step has one group, where the match table takes its 64
// lanes in turn, so tiles of lines stay with the batched passes (packed 1,422
// us with them, 1,875 without).
bool plain_takes_all(const KArgs& a, std::size_t n)
{
    return (n <= kPlainAlone && a.tile <= 256) || (a.slots == 0 && a.flat == 0);
}

void choose_match(KArgs& a, bool ranges_pack)
{
    constexpr std::size_t kLdsPerCu = kLdsPerCuBytes;
    constexpr std::size_t kMaxWaves = 4 * kSimdsPerCu;
    const auto waves = [&](std::size_t bytes) {
        const std::size_t w = bytes == 0 ? kMaxWaves : kLdsPerCu / bytes;
        return w < kMaxWaves ? w : kMaxWaves;
    };
    a.match_lds = 0;
    a.stripe_lds = 0;
    a.r_lds = 0;
    if (ranges_pack) {
        const std::size_t s0 = lds_summary(a), p0 = lds_apply(a);
        a.r_lds = 1;
        if (waves(lds_summary(a)) < waves(s0) || waves(lds_apply(a)) < waves(p0)) {
            a.r_lds = 0;
        }
    }
    const std::size_t s0 = lds_summary(a), p0 = lds_apply(a);
    a.match_lds = 1;
    if (waves(lds_summary(a)) < waves(s0) || waves(lds_apply(a)) < waves(p0)) {
        a.match_lds = 0;
    }
    // the stripe table likewise, for power-of-two axes (plane ids below
    // 2^20 and channel ids below 2^12 pack into one word)
    if (!a.flat && a.pow2 && a.Rp <= (1u << 20) && a.Rc <= (1u << 12)) {
        const std::size_t s1 = lds_summary(a), p1 = lds_apply(a);
        a.stripe_lds = 1;
        if (waves(lds_summary(a)) < waves(s1) || waves(lds_apply(a)) < waves(p1)) {
            a.stripe_lds = 0;
        }
    }
}

// Records per tile when the configuration leaves it open: the largest power
// of two up to 16384 that gives every CU sixteen tiles, down to 1024 records;
// below that, the largest that gives every CU eight tiles, at least 256.
// (Mid-sized runs of 2^22 to 2^25 records take twice the tiles they would at
// eight per CU: more waves to cover the per-record passes' latency, at the
// price of a carry chain of twice the tiles.)  Runs of fewer than 1,024 such
// tiles (up to 2^18 records) leave most of the chip idle and take as long as
// one tile's steps in a row: their tiles go down to 64 records, one step each
// (4,096 records 87 -> 72 us, 2^16 92 -> 81; at 2^18 records 64-record tiles
// cost the carry chain more than they save, 105 -> 116).
std::uint32_t auto_tile(std::size_t n)
{
    std::uint32_t t = 16384;
    while (t > 1024 && (n + t - 1) / t < 4096) {
        t >>= 1;
    }
    while (t > 256 && (n + t - 1) / t < 2048) {
        t >>= 1;
    }
    while (t > 64 && (n + t - 1) / t < 1024) {
        t >>= 1;
    }
    return t;
}

// Empirical curve on the host (hbf_device.cuh:959-1029), for the per-run
// service table.
std::uint64_t sat_mul(std::uint64_t a, std::uint32_t b)
{
    return b != 0 && a > ~0ull / b ? ~0ull : a * b;
}

std::uint64_t sat_add_host(std::uint64_t a, std::uint64_t b)
{
    return b > ~0ull - a ? ~0ull : a + b;
}

std::uint64_t ceiling_scaled_delta(std::uint64_t delta, std::uint32_t offset, std::uint32_t span)
{
    if (delta == 0 || offset == 0) {
        return 0;
    }
    if (span == 0) {
        return ~0ull;
    }
    const std::uint64_t q = delta / span, r = delta % span;
    return sat_add_host(sat_mul(q, offset), (r * offset + span - 1) / span);
}

std::uint64_t emp_cumulative(const engine_config& c, std::uint32_t run)
{
    if (run == 0) {
        return 0;
    }
    const std::uint32_t count = 6;
    std::uint32_t right = 0;
    while (right < count && run > c.emp_pages[right]) {
        ++right;
    }
    if (right == count) {
        right = count - 1;
    }
    std::uint32_t left_pages = 0;
    std::uint64_t left_ns = 0;
    if (right != 0) {
        left_pages = c.emp_pages[right - 1];
        left_ns = c.emp_cum_ns[right - 1];
    }
    if (run > c.emp_pages[right]) {
        left_pages = c.emp_pages[count - 2];
        left_ns = c.emp_cum_ns[count - 2];
        right = count - 1;
    }
    if (c.emp_pages[right] <= left_pages || c.emp_cum_ns[right] < left_ns || run < left_pages) {
        return ~0ull;
    }
    return sat_add_host(left_ns, ceiling_scaled_delta(c.emp_cum_ns[right] - left_ns,
                                                      run - left_pages,
                                                      c.emp_pages[right] - left_pages));
}

bool emp_control_valid(const engine_config& c)
{
    if (c.emp_program_ns == 0) {
        return false;
    }
    for (int i = 0; i < 6; ++i) {
        if (c.emp_pages[i] == 0 || c.emp_cum_ns[i] == 0 ||
            (i != 0 && (c.emp_pages[i] <= c.emp_pages[i - 1] ||
                        c.emp_cum_ns[i] <= c.emp_cum_ns[i - 1]))) {
            return false;
        }
    }
    return c.emp_pages[5] <= kRunCap;
}

// Service (ps) of a read at burst run 0..1023; products wrap like the CPU
// restatement's.
std::vector<std::uint64_t> emp_service_table(const engine_config& c)
{
    std::vector<std::uint64_t> t(kRunCap + 1, 0);
    for (std::uint32_t run = 1; run <= kRunCap; ++run) {
        const std::uint64_t cur = emp_cumulative(c, run), prev = emp_cumulative(c, run - 1);
        const std::uint64_t ns = cur < prev ? ~0ull : cur - prev;
        t[run] = ns * 1000ull;
    }
    return t;
}

// The passes' times over the run that has just completed, from their stamps.
void note_times(engine* e)
{
    for (int k = 0; k < 3; ++k) {
        const std::uint64_t from = e->h_out->stamp[k], to = e->h_out->stamp[k + 1];
        e->last_ms[k] = to > from ? static_cast<float>((to - from) * e->ms_per_tick) : 0.0f;
    }
}

int run_empirical(engine* e, const hbf_record32* d_rec, std::size_t n, std::uint64_t* d_comp,
                  std::uint8_t* d_status, std::uint64_t base_ps, hipStream_t stream,
                  hbfsim_amd_report* out, bool in_order)
{
    const engine_config& c = e->cfg;
    if (c.page_shift != 12 || !emp_control_valid(c)) {
        return HBFSIM_UNSUPPORTED;
    }
    KArgs a = e->args;
    a.disorder = in_order ? nullptr : e->d_disorder;
    const std::size_t ntiles = (n + kEmpTile - 1) / kEmpTile;
    if (ntiles > 0x7fffffffull) {
        return HBFSIM_UNSUPPORTED;
    }
    if (e->d_emp_svc == nullptr) {
        // (the profile's; made by the engine's first run)
        const std::vector<std::uint64_t> table = emp_service_table(c);
        if (halloc(e->d_emp_svc, table.size()) != hipSuccess) {
            return HBFSIM_CUDA_ERROR;
        }
        if (hipMemcpy(e->d_emp_svc, table.data(), table.size() * 8, hipMemcpyHostToDevice) !=
            hipSuccess) {
            hfree(e->d_emp_svc);
            return HBFSIM_CUDA_ERROR;
        }
    }
    const std::uint64_t* d_svc = e->d_emp_svc;
    ScratchPlan plan;
    const std::size_t o_tiles = plan.add<EmpTile>(ntiles);
    const std::size_t o_in = plan.add<EmpState>(ntiles);
    const std::size_t o_maps = plan.add<TailMap>(ntiles);
    const std::size_t o_tail = plan.add<std::uint64_t>(ntiles);
    const std::size_t o_rep = plan.add<DevReport>(ntiles);
    const std::size_t o_fseq = plan.add<std::uint64_t>(1);
    ScratchLease lease(plan.bytes, stream);
    if (!lease.ok()) {
        return HBFSIM_CUDA_ERROR;
    }
    auto* d_tiles = lease.at<EmpTile>(o_tiles);
    auto* d_in = lease.at<EmpState>(o_in);
    auto* d_maps = lease.at<TailMap>(o_maps);
    auto* d_tail = lease.at<std::uint64_t>(o_tail);
    auto* d_trep = lease.at<DevReport>(o_rep);
    auto* d_fseq = lease.at<std::uint64_t>(o_fseq);  // the sequence after the run
    EmpState init{};
    {
        const std::uint64_t packed = e->burst;
        const std::uint64_t p1 = packed >> 11;
        init.valid = (packed != 0 && (packed & kRunCap) != 0 && p1 != 0) ? 1u : 0u;
        init.key = ((p1 == 0 ? 0 : p1 - 1) << 1) | ((packed >> 10) & 1u);
        init.run = static_cast<std::uint32_t>(packed & kRunCap);
    }
    const std::size_t lds = 8ull * a.r_nfence;
    const std::size_t lds_apply = lds + (a.hybrid ? 4ull * kEmpSlots : 0ull);
    const std::uint64_t program_ps = c.emp_program_ns * 1000ull;
    const dim3 grid(static_cast<unsigned>(ntiles));
    hipLaunchKernelGGL(k_emp_tile<false>, grid, dim3(kEmpThreads), lds, stream, a, d_rec, n,
                       base_ps, d_svc, program_ps, d_tiles, d_maps,
                       static_cast<const EmpState*>(nullptr),
                       static_cast<const std::uint64_t*>(nullptr),
                       static_cast<std::uint64_t*>(nullptr), static_cast<std::uint8_t*>(nullptr),
                       static_cast<DevReport*>(nullptr));
    hipLaunchKernelGGL(k_emp_chain, dim3(1), dim3(kEmpChain), 0, stream, a, d_tiles, ntiles, init,
                       e->d_seq, d_in, d_fseq, &e->h_out->fin);
    hipLaunchKernelGGL(k_emp_lead, dim3(static_cast<unsigned>((ntiles + kEmpWaves - 1) / kEmpWaves)),
                       dim3(kEmpThreads), lds, stream, a, d_rec, n, ntiles, base_ps, d_svc,
                       program_ps, d_tiles, d_in, d_maps);
    hipLaunchKernelGGL(k_emp_tail, dim3(1), dim3(kEmpChain), 0, stream, d_maps, ntiles, d_fseq,
                       a.disorder, d_tail, e->d_cbusy, e->d_seq, e->d_ctot);
    hipLaunchKernelGGL(k_emp_tile<true>, grid, dim3(kEmpThreads), lds_apply, stream, a, d_rec, n,
                       base_ps, d_svc, program_ps, static_cast<EmpTile*>(nullptr),
                       static_cast<TailMap*>(nullptr), d_in, d_tail, d_comp, d_status, d_trep);
    launch_report(stream, d_trep, ntiles, e->d_rep_parts, e->d_done, a.disorder, e->d_stamp,
                  e->h_out);
    hipError_t err = hipGetLastError();
    if (err == hipSuccess) err = hipStreamSynchronize(stream);
    if (err != hipSuccess) {
        return HBFSIM_CUDA_ERROR;
    }
    lease.synced(err);
    if (e->h_out->back != 0) {
        // a record's issue time goes back: served in (issue, position) order;
        // the engine state is as the run found it
        lease.release();
        return run_in_issue_order(
            d_rec, false, n, d_comp, d_status, stream,
            [&](const void* sorted, std::uint64_t* comp, std::uint8_t* status) {
                return run_empirical(e, static_cast<const hbf_record32*>(sorted), n, comp, status,
                                     base_ps, stream, out, true);
            });
    }
    const EmpState& fin = e->h_out->fin;
    if (fin.valid) {
        e->burst = (((fin.key >> 1) + 1) << 11) | ((fin.key & 1u) << 10) | fin.run;
    }
    note_times(e);
    if (out != nullptr) {
        std::memcpy(out, &e->h_out->rep, sizeof(DevReport));
    }
    return HBFSIM_OK;
}

// Per-record page-buffer hits for two registers per plane, and the tags the
// run leaves behind (host array [2 * planes]).  d_hits: n bytes.
int k2_hits(engine* e, KArgs a, const hbf_record32* d_rec, std::size_t n,
            std::uint64_t base_ps, std::size_t ntiles, hipStream_t stream, std::uint8_t* d_hits,
            std::vector<std::uint64_t>& tags_out)
{
    a.r_lds = 0;  // these passes look ranges up through the fences
    const std::uint32_t rp = a.Rp;
    std::vector<std::uint64_t> tags(2ull * rp);
    hipError_t err = hipMemcpyAsync(tags.data(), e->d_ptag, tags.size() * 8,
                                    hipMemcpyDeviceToHost, stream);
    if (err == hipSuccess) err = hipStreamSynchronize(stream);
    if (err != hipSuccess) {
        return HBFSIM_CUDA_ERROR;
    }
    std::vector<K2Plane> kp(rp);
    std::vector<std::uint32_t> want(rp, 0), differ(rp, 0);
    std::vector<unsigned long long> idx_a(rp, ~0ull), idx_b(rp, ~0ull);
    std::vector<std::uint32_t> page_a(rp, 0), page_b(rp, 0);
    bool need_a = false;
    for (std::uint32_t r = 0; r < rp; ++r) {
        const std::uint64_t t0 = tags[2 * r], t1 = tags[2 * r + 1];
        need_a = need_a || (t0 == 0 && t1 == 0);
    }
    const std::size_t ngroups = (ntiles + kGroup - 1) / kGroup;
    ScratchPlan plan;
    const std::size_t o_want = plan.add<std::uint32_t>(rp);
    const std::size_t o_differ = plan.add<std::uint32_t>(rp);
    const std::size_t o_first = plan.add<unsigned long long>(rp);
    const std::size_t o_page = plan.add<std::uint32_t>(rp);
    const std::size_t o_kp = plan.add<K2Plane>(rp);
    const std::size_t o_tlast = plan.add<std::uint32_t>(ntiles * rp);
    const std::size_t o_tfirst = plan.add<K2First>(ntiles * rp);
    const std::size_t o_glast = plan.add<std::uint32_t>(ngroups * rp);
    const std::size_t o_gin = plan.add<std::uint32_t>(ngroups * rp);
    const std::size_t o_final = plan.add<std::uint32_t>(rp);
    ScratchLease lease(plan.bytes, stream);
    if (!lease.ok()) {
        return HBFSIM_CUDA_ERROR;
    }
    auto* d_want = lease.at<std::uint32_t>(o_want);
    auto* d_differ = lease.at<std::uint32_t>(o_differ);
    auto* d_first = lease.at<unsigned long long>(o_first);
    auto* d_page = lease.at<std::uint32_t>(o_page);
    auto* d_kp = lease.at<K2Plane>(o_kp);
    auto* d_tlast = lease.at<std::uint32_t>(o_tlast);
    auto* d_tfirst = lease.at<K2First>(o_tfirst);
    auto* d_glast = lease.at<std::uint32_t>(o_glast);
    auto* d_gin = lease.at<std::uint32_t>(o_gin);
    auto* d_final = lease.at<std::uint32_t>(o_final);
    const unsigned first_blocks = static_cast<unsigned>((n + kK2Chunk - 1) / kK2Chunk);
    const std::size_t lds_first = 8ull * a.r_nfence + 8ull * rp;
    // pass A: the first record of every plane with both slots empty
    auto first_pass = [&](std::vector<unsigned long long>& idx,
                          std::vector<std::uint32_t>& page) -> hipError_t {
        std::vector<unsigned long long> init(rp, ~0ull);
        hipError_t e2 = hipMemcpyAsync(d_want, want.data(), rp * 4, hipMemcpyHostToDevice, stream);
        if (e2 == hipSuccess)
            e2 = hipMemcpyAsync(d_differ, differ.data(), rp * 4, hipMemcpyHostToDevice, stream);
        if (e2 == hipSuccess)
            e2 = hipMemcpyAsync(d_first, init.data(), rp * 8, hipMemcpyHostToDevice, stream);
        if (e2 != hipSuccess) return e2;
        hipLaunchKernelGGL(k_k2_first, dim3(first_blocks), dim3(256), lds_first, stream, a, d_rec,
                           n, base_ps, static_cast<const std::uint32_t*>(d_want),
                           static_cast<const std::uint32_t*>(d_differ), d_first);
        hipLaunchKernelGGL(k_k2_page, dim3(1), dim3(256), 8ull * a.r_nfence, stream, a, d_rec, n,
                           base_ps, static_cast<const unsigned long long*>(d_first), d_page);
        e2 = hipGetLastError();
        if (e2 == hipSuccess)
            e2 = hipMemcpyAsync(idx.data(), d_first, rp * 8, hipMemcpyDeviceToHost, stream);
        if (e2 == hipSuccess)
            e2 = hipMemcpyAsync(page.data(), d_page, rp * 4, hipMemcpyDeviceToHost, stream);
        if (e2 == hipSuccess) e2 = hipStreamSynchronize(stream);
        return e2;
    };
    if (need_a) {
        for (std::uint32_t r = 0; r < rp; ++r) {
            want[r] = tags[2 * r] == 0 && tags[2 * r + 1] == 0;
            differ[r] = 0;
        }
        err = first_pass(idx_a, page_a);
    }
    // pass B: the first record whose page differs from the one slot held
    if (err == hipSuccess) {
        bool any = false;
        for (std::uint32_t r = 0; r < rp; ++r) {
            const std::uint64_t t0 = tags[2 * r], t1 = tags[2 * r + 1];
            want[r] = 0;
            differ[r] = 0;
            if (t0 != 0 && t1 == 0) {
                want[r] = 1;
                differ[r] = static_cast<std::uint32_t>(t0);
            } else if (t0 == 0 && t1 != 0) {
                want[r] = 1;
                differ[r] = static_cast<std::uint32_t>(t1);
            } else if (t0 == 0 && t1 == 0 && idx_a[r] < n) {
                want[r] = 1;
                differ[r] = page_a[r];
            }
            any = any || want[r];
        }
        if (any) {
            err = first_pass(idx_b, page_b);
        }
    }
    if (err != hipSuccess) {
        return HBFSIM_CUDA_ERROR;
    }
    for (std::uint32_t r = 0; r < rp; ++r) {
        const std::uint64_t t0 = tags[2 * r], t1 = tags[2 * r + 1];
        K2Plane& k = kp[r];
        k.start3 = ~0ull;
        k.miss1 = k.miss2 = ~0ull;
        k.t1 = 0;
        k.l_init = 0;
        const bool b = idx_b[r] < n;
        if (t0 != 0 && t1 != 0) {
            k.start3 = 0;
            k.t1 = static_cast<std::uint32_t>(t1);
            k.l_init = static_cast<std::uint32_t>(t0);
        } else if (t0 != 0) {
            k.l_init = static_cast<std::uint32_t>(t0);
            if (b) {
                k.miss2 = idx_b[r];
                k.start3 = idx_b[r] + 1;
                k.t1 = page_b[r];
            }
        } else if (t1 != 0) {
            k.t1 = static_cast<std::uint32_t>(t1);
            if (b) {
                k.miss1 = idx_b[r];
                k.start3 = idx_b[r] + 1;
            }
        } else if (idx_a[r] < n) {
            k.miss1 = idx_a[r];
            if (b) {
                k.miss2 = idx_b[r];
                k.start3 = idx_b[r] + 1;
                k.t1 = page_b[r];
            }
        }
    }
    err = hipMemcpyAsync(d_kp, kp.data(), rp * sizeof(K2Plane), hipMemcpyHostToDevice, stream);
    if (err != hipSuccess) {
        return HBFSIM_CUDA_ERROR;
    }
    const std::size_t lds = 8ull * (a.r_nfence + (rp + kWave - 1) / kWave) + 8ull * rp;
    const unsigned wide = static_cast<unsigned>((ngroups * rp + 255) / 256);
    hipLaunchKernelGGL(k_k2_hits, dim3(static_cast<unsigned>(ntiles)), dim3(kWave), lds, stream, a,
                       d_rec, n, base_ps, static_cast<const K2Plane*>(d_kp), d_tlast, d_tfirst,
                       d_hits);
    hipLaunchKernelGGL(k_k2_up, dim3(wide), dim3(256), 0, stream, a, ntiles, ngroups,
                       static_cast<const std::uint32_t*>(d_tlast), d_glast);
    hipLaunchKernelGGL(k_k2_mid, dim3((rp + 255) / 256), dim3(256), 0, stream, a, ngroups,
                       static_cast<const K2Plane*>(d_kp), static_cast<const std::uint32_t*>(d_glast),
                       d_gin, d_final);
    hipLaunchKernelGGL(k_k2_down, dim3(wide), dim3(256), 0, stream, a, ntiles, ngroups,
                       static_cast<const K2Plane*>(d_kp), static_cast<const std::uint32_t*>(d_tlast),
                       static_cast<const K2First*>(d_tfirst),
                       static_cast<const std::uint32_t*>(d_gin), d_hits);
    std::vector<std::uint32_t> fin(rp);
    err = hipGetLastError();
    if (err == hipSuccess)
        err = hipMemcpyAsync(fin.data(), d_final, rp * 4, hipMemcpyDeviceToHost, stream);
    if (err == hipSuccess) err = hipStreamSynchronize(stream);
    lease.synced(err);
    if (err != hipSuccess) {
        return HBFSIM_CUDA_ERROR;
    }
    tags_out.assign(2ull * rp, 0);
    for (std::uint32_t r = 0; r < rp; ++r) {
        tags_out[2 * r] = fin[r];
        tags_out[2 * r + 1] = kp[r].t1;
    }
    return HBFSIM_OK;
}

}  // namespace

int engine_create(const engine_config& c, engine** out)
{
    *out = nullptr;
    const std::uint32_t rp = c.n_planes(), rc = c.n_channels();
    if (c.channels == 0 || c.ways == 0 || c.dies == 0 || c.planes == 0 || c.page_shift < 9 ||
        c.page_shift > 31 || c.slots > 2 || c.xfer_den == 0 || c.xfer_quantum == 0 ||
        c.tile % kWave != 0) {
        return HBFSIM_INVALID_ARGUMENT;
    }
    if (rp > kMaxPlanes || rc > kMaxChannels) {
        return HBFSIM_UNSUPPORTED;
    }
    // bytes * num must fit 64 bits for every transfer size up to a page.
    const unsigned __int128 worst =
        static_cast<unsigned __int128>(1ull << c.page_shift) * c.xfer_num + c.xfer_den;
    if (worst > ~0ull) {
        return HBFSIM_UNSUPPORTED;
    }
    auto* e = new (std::nothrow) engine;
    if (e == nullptr) {
        return HBFSIM_IO_ERROR;
    }
    e->cfg = c;
    scratch_hold();
    if (hipGetDevice(&e->device) != hipSuccess) {
        scratch_drop();
        delete e;
        return HBFSIM_CUDA_ERROR;
    }
    KArgs& a = e->args;
    std::memset(&a, 0, sizeof(a));
    a.Rp = rp;
    a.Rc = rc;
    a.W = c.ways;
    a.D = c.dies;
    a.P = c.planes;
    a.pbits = bits_for(rp);
    a.cbits = bits_for(rc);
    a.flat = (rp == 1 && rc == 1) ? 1u : 0u;
    const std::uint32_t size[4] = {c.channels, c.ways, c.dies, c.planes};
    std::uint64_t div = 1;
    bool pow2 = true;
    for (int i = 0; i < 4; ++i) {
        const std::uint32_t ax = c.order[i];
        a.axis_size[ax] = size[ax];
        a.axis_div[ax] = div;
        pow2 = pow2 && is_pow2(size[ax]);
        div *= size[ax];
    }
    for (int ax = 0; ax < 4; ++ax) {
        a.axis_shift[ax] = log2u(a.axis_div[ax]);
    }
    a.pow2 = pow2 ? 1u : 0u;
    a.page_shift = c.page_shift;
    a.slots = c.slots;
    a.contention = c.contention;
    a.transfer_page = c.transfer_page;
    a.every_write = c.every_write;
    a.hybrid = c.hybrid;
    a.hybrid_warmup = c.hybrid_warmup;
    a.hybrid_threshold = c.hybrid_threshold;
    a.read_ps = c.read_ps;
    a.program_ps = c.program_ps;
    a.xfer_num = c.xfer_num;
    a.xfer_den = c.xfer_den;
    a.xfer_q = c.xfer_quantum;
    for (int k = 0; k <= 32; ++k) {
        const unsigned __int128 prod = static_cast<unsigned __int128>(1ull << k) * c.xfer_num;
        a.xfer_pow2[k] = c.xfer_quantum *
                         static_cast<std::uint64_t>((prod + c.xfer_den - 1) / c.xfer_den);
    }
    a.tile = c.tile;
    a.media_pages = c.media_pages;
    ScratchPlan plan;
    const std::size_t pbusy = plan.add<std::uint64_t>(rp);
    const std::size_t ptag = plan.add<std::uint64_t>(2ull * rp);
    const std::size_t cbusy = plan.add<std::uint64_t>(rc);
    const std::size_t ptot = plan.add<std::uint64_t>(rp);
    const std::size_t ctot = plan.add<std::uint64_t>(rc);
    const std::size_t seq = plan.add<std::uint64_t>(1);
    const std::size_t done = plan.add<std::uint32_t>(1);
    const std::size_t disorder = plan.add<std::uint32_t>(1);
    e->state_bytes = plan.bytes;
    const std::size_t stamp = plan.add<std::uint64_t>(4);
    const std::size_t rep_parts = plan.add<std::uint64_t>(kRepParts * kRepWords);
    hipError_t err = halloc(e->state_block, plan.bytes);
    if (err == hipSuccess) {
        place(e->d_pbusy, e->state_block, pbusy);
        place(e->d_ptag, e->state_block, ptag);
        place(e->d_cbusy, e->state_block, cbusy);
        place(e->d_ptot, e->state_block, ptot);
        place(e->d_ctot, e->state_block, ctot);
        place(e->d_seq, e->state_block, seq);
        place(e->d_done, e->state_block, done);
        place(e->d_stamp, e->state_block, stamp);
        place(e->d_rep_parts, e->state_block, rep_parts);
        place(e->d_disorder, e->state_block, disorder);
    }
    if (err == hipSuccess)
        err = hipHostMalloc(reinterpret_cast<void**>(&e->h_out), sizeof(HostOut));
    int khz = 0;
    if (err == hipSuccess)
        err = hipDeviceGetAttribute(&khz, hipDeviceAttributeWallClockRate, e->device);
    e->ms_per_tick = khz > 0 ? 1.0 / khz : 0.0;
    a.stamp = e->d_stamp;
    if (err != hipSuccess) {
        engine_destroy(e);
        return HBFSIM_CUDA_ERROR;
    }
    const int rs = engine_reset(e);
    if (rs != HBFSIM_OK) {
        engine_destroy(e);
        return rs;
    }
    // set-up of the no-allocation entry point on this device (once per
    // device; a failed lookup only disables that entry point)
    (void)noalloc_scratch(e->device);
    *out = e;
    return HBFSIM_OK;
}

void engine_destroy(engine* e)
{
    if (e == nullptr) {
        return;
    }
    (void)hipSetDevice(e->device);
    (void)hipDeviceSynchronize();
    free_scratch(e);
    hfree(e->range_block);
    hfree(e->state_block);
    hfree(e->d_emp_svc);
    if (e->h_out != nullptr) {
        (void)hipHostFree(e->h_out);
    }
    delete e;
    scratch_drop();
}

const engine_config& engine_get_config(const engine* e) { return e->cfg; }

int engine_set_ranges(engine* e, const std::vector<range_rec>& ranges)
{
    e->ranges = ranges;
    e->ranges_dirty = true;
    return HBFSIM_OK;
}

int engine_reset(engine* e)
{
    hipError_t err = hipMemset(e->state_block, 0, e->state_bytes);
    if (err == hipSuccess) err = hipDeviceSynchronize();
    e->burst = 0;
    return hip_status(err);
}

int engine_synchronize(engine* e)
{
    (void)e;
    return hip_status(hipDeviceSynchronize());
}

// in_order: the records are known to be in issue order (a sorted copy), so
// the summary pass does not watch for records that go back in time.
int engine_run_any(engine* e, const void* d_rec, bool packed, std::size_t n,
                   std::uint64_t* d_comp, std::uint8_t* d_status, std::uint64_t base_ps,
                   void* stream_ptr, hbfsim_amd_report* out, bool refresh_records,
                   unsigned char* ext_scratch = nullptr, bool in_order = false);

int engine_run(engine* e, const hbf_record32* d_rec, std::size_t n, std::uint64_t* d_comp,
               std::uint8_t* d_status, std::uint64_t base_ps, void* stream_ptr,
               hbfsim_amd_report* out, bool refresh_records)
{
    return engine_run_any(e, d_rec, false, n, d_comp, d_status, base_ps, stream_ptr, out,
                          refresh_records);
}

int engine_run_packed(engine* e, const hbf_record16* d_rec, std::size_t n,
                      std::uint64_t* d_comp, std::uint8_t* d_status, std::uint64_t base_ps,
                      void* stream_ptr, hbfsim_amd_report* out)
{
    return engine_run_any(e, d_rec, true, n, d_comp, d_status, base_ps, stream_ptr, out, false);
}

int engine_run_packed_noalloc(engine* e, const hbf_record16* d_rec, std::size_t n,
                              std::uint64_t* d_comp, std::uint8_t* d_status,
                              std::uint64_t base_ps, void* stream_ptr, hbfsim_amd_report* out)
{
    if (hipSetDevice(e->device) != hipSuccess) {
        return HBFSIM_CUDA_ERROR;
    }
    void* ptr = noalloc_scratch(e->device);
    if (ptr == nullptr) {
        return HBFSIM_UNSUPPORTED;  // the static scratch's address lookup failed
    }
    if (e->ranges_dirty) {
        return HBFSIM_UNSUPPORTED;  // uploading a changed range table allocates
    }
    return engine_run_any(e, d_rec, true, n, d_comp, d_status, base_ps, stream_ptr, out, false,
                          static_cast<unsigned char*>(ptr));
}

// Tile size of a run whose scratch comes from a fixed buffer: the engine's
// configured tile, else the automatic one doubled (up to 16,384 records)
// until the scratch fits; 0 when it never does.
std::uint32_t fitting_tile(const engine* e, std::size_t n, std::size_t capacity)
{
    KArgs a = e->args;
    std::uint32_t tile = e->cfg.tile != 0 ? e->cfg.tile : auto_tile(n);
    const std::size_t nsteps = (n + kWave - 1) / kWave;
    for (;;) {
        const std::size_t ntiles = (n + tile - 1) / tile;
        a.tile = tile;
        if (carve_scratch(a, ntiles, nsteps, nullptr, nullptr) <= capacity) {
            return tile;
        }
        if (e->cfg.tile != 0 || tile >= 16384) {
            return 0;
        }
        tile *= 2;
    }
}

int engine_run_any(engine* e, const void* d_rec, bool packed, std::size_t n,
                   std::uint64_t* d_comp, std::uint8_t* d_status, std::uint64_t base_ps,
                   void* stream_ptr, hbfsim_amd_report* out, bool refresh_records,
                   unsigned char* ext_scratch, bool in_order)
{
    if (out != nullptr) {
        std::memset(out, 0, sizeof(*out));
    }
    if (n == 0) {
        // a run of no records still uploads a changed range table, so that
        // it can prepare a context for the entry point that allocates nothing
        if (ext_scratch == nullptr && e->ranges_dirty) {
            if (hipSetDevice(e->device) != hipSuccess) {
                return HBFSIM_CUDA_ERROR;
            }
            return upload_ranges(e, static_cast<hipStream_t>(stream_ptr));
        }
        return HBFSIM_OK;
    }
    if (d_rec == nullptr || d_comp == nullptr ||
        (reinterpret_cast<std::uintptr_t>(d_rec) & 15u) != 0 ||
        (reinterpret_cast<std::uintptr_t>(d_comp) & 7u) != 0) {
        return HBFSIM_INVALID_ARGUMENT;
    }
    // packed records take the main pipeline only: at most one page register,
    // the HBF model (no refresh records: they need flags); hybrid sampling
    // needs the linear steps' range ids beside their descriptors, for which
    // the run without allocation has no room
    if (packed && (e->cfg.model != HBFSIM_AMD_MODEL_HBF || e->cfg.slots > 1 ||
                   (e->cfg.hybrid != 0 && ext_scratch != nullptr))) {
        return HBFSIM_UNSUPPORTED;
    }
    if (e->cfg.model != HBFSIM_AMD_MODEL_HBF && e->cfg.model != HBFSIM_AMD_MODEL_EMPIRICAL) {
        return HBFSIM_UNSUPPORTED;
    }
    if (e->cfg.model == HBFSIM_AMD_MODEL_HBF && e->cfg.slots == 2 && refresh_records) {
        return HBFSIM_UNSUPPORTED;
    }
    // warp grouping reads group ids from 32-byte records (packed records
    // carry none); it runs on the main pipeline with at most one page
    // register and no merged refresh records
    const bool grouping = e->cfg.grouping != 0 && !packed;
    if (grouping && (e->cfg.model != HBFSIM_AMD_MODEL_HBF || e->cfg.slots == 2 ||
                     refresh_records || ext_scratch != nullptr)) {
        return HBFSIM_UNSUPPORTED;
    }
    hipStream_t stream = static_cast<hipStream_t>(stream_ptr);
    e->last_passes = engine::Passes::none;
    if (hipSetDevice(e->device) != hipSuccess) {
        return HBFSIM_CUDA_ERROR;
    }
    if (e->ranges_dirty) {
        const int st = upload_ranges(e, stream);
        if (st != HBFSIM_OK) {
            return st;
        }
    }
    if (e->cfg.model == HBFSIM_AMD_MODEL_EMPIRICAL) {
        if (refresh_records) {
            return HBFSIM_UNSUPPORTED;
        }
        e->last_apply_waves = 0;  // (the empirical model's own kernels, no apply pass)
        return run_empirical(e, static_cast<const hbf_record32*>(d_rec), n, d_comp, d_status,
                             base_ps, stream, out, in_order);
    }
    KArgs a = e->args;
    a.disorder = in_order ? nullptr : e->d_disorder;
    a.tile = e->cfg.tile != 0 ? e->cfg.tile : auto_tile(n);
    if (ext_scratch != nullptr) {
        a.tile = fitting_tile(e, n, kNoAllocScratchBytes);
        if (a.tile == 0) {
            return HBFSIM_UNSUPPORTED;  // beyond the static scratch
        }
    }
    const std::size_t ntiles = (n + a.tile - 1) / a.tile;
    if (ntiles > 0x7fffffffull) {
        return HBFSIM_UNSUPPORTED;
    }
    RunScratch sc{};
    int st = HBFSIM_OK;
    if (ext_scratch != nullptr) {
        (void)carve_scratch(a, ntiles, (n + kWave - 1) / kWave, ext_scratch, &sc);
    } else {
        st = ensure_scratch(e, ntiles);
        if (st != HBFSIM_OK) {
            return st;
        }
        sc = RunScratch{e->d_psum, e->d_tmask, e->d_csum, e->d_pcarry, e->d_ccarry,
                        e->d_tcount, e->d_tseq, e->d_gpsum, e->d_gcsum, e->d_gpcarry,
                        e->d_gccarry, e->d_gcount, e->d_gseq, e->d_tile_rep, nullptr,
                        e->d_tsplit};
    }
    if (!refresh_records) {
        a.tile_split = sc.tsplit;  // the summary pass marks tiles with split steps
    }
    choose_match(a, e->ranges_pack);
    const std::size_t lds_a = lds_summary(a), lds_c = lds_apply(a);
    if (lds_a > kLdsPerBlockBytes || lds_c > kLdsPerBlockBytes) {
        return HBFSIM_UNSUPPORTED;
    }
    hipError_t err = hipSuccess;
    // warp grouping: mark the records that join their group's request
    // (refusing malformed groups before any state changes)
    std::uint8_t* d_lead = nullptr;
    std::uint32_t* d_gerr = nullptr;
    unsigned long long* d_frep = nullptr;
    auto free_group = [&]() {
        hfree(d_lead);
        hfree(d_gerr);
        hfree(d_frep);
    };
    if (grouping) {
        err = halloc(d_lead, n);
        if (err == hipSuccess) err = halloc(d_gerr, 1);
        if (err == hipSuccess) err = halloc(d_frep, 8);
        if (err == hipSuccess) err = hipMemsetAsync(d_gerr, 0, 4, stream);
        if (err == hipSuccess) err = hipMemsetAsync(d_frep, 0, 64, stream);
        if (err == hipSuccess) {
            const std::size_t nl = (n + kLeadSpan - 1) / kLeadSpan;
            KArgs la = a;
            la.r_lds = 0;  // k_lead looks ranges up through the fences
            hipLaunchKernelGGL(k_lead, dim3(static_cast<unsigned>(nl)), dim3(kWave),
                               static_cast<std::size_t>(a.r_nfence) * 8, stream, la,
                               static_cast<const hbf_record32*>(d_rec), n, d_lead, d_gerr);
            err = hipGetLastError();
        }
        std::uint32_t h_gerr = 0;
        if (err == hipSuccess)
            err = hipMemcpyAsync(&h_gerr, d_gerr, 4, hipMemcpyDeviceToHost, stream);
        if (err == hipSuccess) err = hipStreamSynchronize(stream);
        if (err != hipSuccess) {
            free_group();
            return HBFSIM_CUDA_ERROR;
        }
        if (h_gerr != 0) {
            free_group();
            return HBFSIM_INVALID_ARGUMENT;
        }
        a.lead = d_lead;
    }
    // two page registers: hits first, from their own scans
    const bool k2 = e->cfg.slots == 2;
    std::optional<ScratchLease> hit_lease;
    std::uint8_t* d_hits = nullptr;
    std::vector<std::uint64_t> k2_tags;
    if (k2) {
        hit_lease.emplace(n, stream);
        if (!hit_lease->ok()) {
            return HBFSIM_CUDA_ERROR;
        }
        d_hits = hit_lease->at<std::uint8_t>(0);
        st = k2_hits(e, a, static_cast<const hbf_record32*>(d_rec), n, base_ps, ntiles, stream,
                     d_hits, k2_tags);
        if (st != HBFSIM_OK) {
            return st;
        }
        a.ext_hits = 1;
    }
    // step descriptors, where the apply pass replays linear steps from them
    StepDesc* desc = nullptr;
    if (ext_scratch != nullptr) {
        desc = sc.desc;  // packed runs: one page register, no sampling; split
                         // steps go without descriptors (no side array)
    } else if ((k2 || a.slots == 1) && !grouping) {
        const std::size_t nsteps = (n + kWave - 1) / kWave;
        if (nsteps > e->desc_cap) {
            hfree(e->desc_block);
            e->desc_cap = 0;
            const std::size_t cap = nsteps + nsteps / 8;  // headroom, as for the tiles
            ScratchPlan plan;
            const std::size_t steps = plan.add<StepDesc>(cap);
            const std::size_t rids = plan.add<std::uint32_t>(cap);
            const std::size_t splits = plan.add<SplitDesc>(cap);
            if (halloc(e->desc_block, plan.bytes) != hipSuccess) {
                free_group();
                return HBFSIM_CUDA_ERROR;
            }
            place(e->d_desc, e->desc_block, steps);
            place(e->d_desc_rid, e->desc_block, rids);
            place(e->d_desc_split, e->desc_block, splits);
            e->desc_cap = cap;
        }
        desc = e->d_desc;
        a.desc_split = e->d_desc_split;
        if (a.hybrid != 0) {
            a.desc_rid = e->d_desc_rid;
        }
    }
    const dim3 grid(static_cast<unsigned>(ntiles));
    const std::uint8_t* hits = d_hits;
    // Scattered records: their own passes take the tiles that hold no runs of
    // lines.  An engine whose last run mostly hit its page registers (runs of
    // lines) does not look for them.
    const bool plain = !grouping && !k2 && !refresh_records && plain_run(a, e->ranges_pack);
    const bool plain_alone = plain && plain_takes_all(a, n);
    const bool plain_mixed = plain && !plain_alone &&
                             (e->last_modeled == 0 || e->last_hits * 8 < e->last_modeled);
    a.mixed = plain_mixed ? 1u : 0u;
    if (plain_alone || plain_mixed) {
        a.r_top = 1;
        while (a.r_top * 2 <= a.r_count) {
            a.r_top *= 2;
        }
        const auto summary = packed ? (plain_alone ? k_plain_summary<true, true>
                                                   : k_plain_summary<true, false>)
                                    : (plain_alone ? k_plain_summary<false, true>
                                                   : k_plain_summary<false, false>);
        hipLaunchKernelGGL(summary, grid, dim3(kWave), plain_summary_lds(a), stream, a, d_rec, n,
                           base_ps, sc.psum, sc.tmask, sc.csum, sc.tcount);
    }
    if (plain_alone) {
        // every tile is summarised
    } else if (k2) {
        (void)allow_lds(k_summary<false, true>, lds_a);
        hipLaunchKernelGGL((k_summary<false, true>), grid, dim3(kWave), lds_a, stream, a, d_rec,
                           n, base_ps, sc.psum, sc.tmask, sc.csum, sc.tcount,
                           hits, desc);
    } else if (refresh_records) {
        (void)allow_lds(k_summary<true, false>, lds_a);
        hipLaunchKernelGGL((k_summary<true, false>), grid, dim3(kWave), lds_a, stream, a, d_rec,
                           n, base_ps, sc.psum, sc.tmask, sc.csum, sc.tcount,
                           hits, desc);
    } else if (packed && kLdsPerCuBytes / lds_a <= 8) {  // LDS allows at most 8 waves per CU
        (void)allow_lds(k_summary<false, false, true, true>, lds_a);
        hipLaunchKernelGGL((k_summary<false, false, true, true>), grid, dim3(kWave), lds_a, stream,
                           a, d_rec, n, base_ps, sc.psum, sc.tmask, sc.csum, sc.tcount,
                           hits, desc);
    } else if (packed && ntiles <= kFewTiles) {
        (void)allow_lds(k_summary<false, false, true, false, true>, lds_a);
        hipLaunchKernelGGL((k_summary<false, false, true, false, true>), grid, dim3(kWave), lds_a,
                           stream, a, d_rec, n, base_ps, sc.psum, sc.tmask, sc.csum, sc.tcount,
                           hits, desc);
    } else if (packed) {
        (void)allow_lds(k_summary<false, false, true>, lds_a);
        hipLaunchKernelGGL((k_summary<false, false, true>), grid, dim3(kWave), lds_a, stream, a,
                           d_rec, n, base_ps, sc.psum, sc.tmask, sc.csum, sc.tcount,
                           hits, desc);
    } else {
        (void)allow_lds(k_summary<false, false>, lds_a);
        hipLaunchKernelGGL((k_summary<false, false>), grid, dim3(kWave), lds_a, stream, a, d_rec,
                           n, base_ps, sc.psum, sc.tmask, sc.csum, sc.tcount,
                           hits, desc);
    }
    {
        const std::size_t ngroups = (ntiles + kGroup - 1) / kGroup;
        const std::size_t rt = static_cast<std::size_t>(a.Rp) + a.Rc + 1;
        const unsigned wide = static_cast<unsigned>((ngroups * rt + 255) / 256);
        if (ntiles <= kOneCarryTiles) {
            const auto span = static_cast<std::uint32_t>((ntiles + kMidBlock - 1) / kMidBlock);
            hipLaunchKernelGGL(k_carry_one, dim3(static_cast<unsigned>(rt)), dim3(kMidBlock), 0,
                               stream, a, ntiles, span, sc.psum, sc.tmask, sc.csum,
                               sc.tcount, sc.pcarry, sc.ccarry, sc.tseq, e->d_pbusy, e->d_ptag,
                               e->d_cbusy, e->d_seq, e->d_ptot, e->d_ctot);
        } else {
            hipLaunchKernelGGL(k_carry_up, dim3(wide), dim3(256), 0, stream, a, ntiles, ngroups,
                               sc.psum, sc.tmask, sc.csum, sc.tcount, sc.gpsum,
                               sc.gcsum, sc.gcount);
            hipLaunchKernelGGL(k_carry_mid, dim3(a.Rp + a.Rc + 1), dim3(kMidBlock), 0, stream, a,
                               ngroups,
                               sc.gpsum, sc.gcsum, sc.gcount, sc.gpcarry, sc.gccarry,
                               sc.gseq, e->d_pbusy, e->d_ptag, e->d_cbusy, e->d_seq, e->d_ptot,
                               e->d_ctot);
            hipLaunchKernelGGL(k_carry_down, dim3(wide), dim3(256), 0, stream, a, ntiles, ngroups,
                               sc.psum, sc.tmask, sc.csum, sc.tcount, sc.gpcarry,
                               sc.gccarry, sc.gseq, sc.pcarry, sc.ccarry, sc.tseq);
        }
    }
    const bool staged = desc != nullptr && staged_steps(a) != 0;
    // the four-wave apply pass: a large stream whose last run on this engine
    // had few page-register hits (mostly general steps), where LDS leaves
    // room for four waves per SIMD
    const bool wide_apply = packed && n >= kWideApplyRecords &&
                            kLdsPerCuBytes / lds_c >= 4 * kSimdsPerCu && e->last_modeled != 0 &&
                            e->last_hits * 8 < e->last_modeled;
    // (k_plain_apply is built for four waves in either record form)
    e->last_apply_waves = plain_alone                             ? 4
                          : packed && !k2 && !refresh_records ? (wide_apply ? 4 : 3)
                                                              : 1;
    if (plain_alone || plain_mixed) {
        const auto apply = packed ? (plain_alone ? k_plain_apply<true, true>
                                                 : k_plain_apply<true, false>)
                                  : (plain_alone ? k_plain_apply<false, true>
                                                 : k_plain_apply<false, false>);
        hipLaunchKernelGGL(apply, grid, dim3(kWave), plain_apply_lds(a), stream, a, d_rec, n,
                           base_ps, sc.pcarry, sc.tmask, sc.ccarry, d_comp, d_status,
                           sc.tile_rep);
    }
    if (plain_alone) {
        // every tile is replayed
    } else if (k2) {
        (void)allow_lds(k_apply<false, true>, lds_c);
        hipLaunchKernelGGL((k_apply<false, true>), grid, dim3(kWave), lds_c, stream, a, d_rec, n,
                           base_ps, sc.pcarry, sc.tmask, sc.ccarry, sc.tseq, d_comp,
                           d_status, sc.tile_rep, hits, desc);
    } else if (refresh_records && staged) {
        (void)allow_lds(k_apply<true, false, true>, lds_c);
        hipLaunchKernelGGL((k_apply<true, false, true>), grid, dim3(kWave), lds_c, stream, a,
                           d_rec, n, base_ps, sc.pcarry, sc.tmask, sc.ccarry, sc.tseq,
                           d_comp, d_status, sc.tile_rep, hits, desc);
    } else if (refresh_records) {
        (void)allow_lds(k_apply<true, false>, lds_c);
        hipLaunchKernelGGL((k_apply<true, false>), grid, dim3(kWave), lds_c, stream, a, d_rec, n,
                           base_ps, sc.pcarry, sc.tmask, sc.ccarry, sc.tseq, d_comp,
                           d_status, sc.tile_rep, hits, desc);
    } else if (packed && staged && wide_apply) {
        (void)allow_lds(k_apply<false, false, true, true, true>, lds_c);
        hipLaunchKernelGGL((k_apply<false, false, true, true, true>), grid, dim3(kWave), lds_c,
                           stream, a, d_rec, n, base_ps, sc.pcarry, sc.tmask, sc.ccarry,
                           sc.tseq, d_comp, d_status, sc.tile_rep, hits, desc);
    } else if (packed && staged) {
        (void)allow_lds(k_apply<false, false, true, true>, lds_c);
        hipLaunchKernelGGL((k_apply<false, false, true, true>), grid, dim3(kWave), lds_c, stream,
                           a, d_rec, n, base_ps, sc.pcarry, sc.tmask, sc.ccarry,
                           sc.tseq, d_comp, d_status, sc.tile_rep, hits, desc);
    } else if (packed && wide_apply) {
        (void)allow_lds(k_apply<false, false, false, true, true>, lds_c);
        hipLaunchKernelGGL((k_apply<false, false, false, true, true>), grid, dim3(kWave), lds_c,
                           stream, a, d_rec, n, base_ps, sc.pcarry, sc.tmask, sc.ccarry,
                           sc.tseq, d_comp, d_status, sc.tile_rep, hits, desc);
    } else if (packed) {
        (void)allow_lds(k_apply<false, false, false, true>, lds_c);
        hipLaunchKernelGGL((k_apply<false, false, false, true>), grid, dim3(kWave), lds_c, stream,
                           a, d_rec, n, base_ps, sc.pcarry, sc.tmask, sc.ccarry,
                           sc.tseq, d_comp, d_status, sc.tile_rep, hits, desc);
    } else if (staged) {
        (void)allow_lds(k_apply<false, false, true>, lds_c);
        hipLaunchKernelGGL((k_apply<false, false, true>), grid, dim3(kWave), lds_c, stream, a,
                           d_rec, n, base_ps, sc.pcarry, sc.tmask, sc.ccarry, sc.tseq,
                           d_comp, d_status, sc.tile_rep, hits, desc);
    } else {
        (void)allow_lds(k_apply<false, false>, lds_c);
        hipLaunchKernelGGL((k_apply<false, false>), grid, dim3(kWave), lds_c, stream, a, d_rec, n,
                           base_ps, sc.pcarry, sc.tmask, sc.ccarry, sc.tseq, d_comp,
                           d_status, sc.tile_rep, hits, desc);
    }
    launch_report(stream, sc.tile_rep, ntiles, e->d_rep_parts, e->d_done, e->d_disorder,
                  e->d_stamp, e->h_out);
    unsigned long long h_frep[8] = {};
    if (grouping) {
        const std::size_t nb = (n + 255) / 256;
        hipLaunchKernelGGL(k_follow,
                           dim3(static_cast<unsigned>(nb < kFollowBlocks ? nb : kFollowBlocks)),
                           dim3(256), 0, stream, static_cast<const hbf_record32*>(d_rec), n,
                           base_ps, d_lead, d_comp, d_status, d_frep);
    }
    err = hipGetLastError();
    if (err == hipSuccess && grouping)
        err = hipMemcpyAsync(h_frep, d_frep, sizeof(h_frep), hipMemcpyDeviceToHost, stream);
    if (err == hipSuccess) err = hipStreamSynchronize(stream);
    const bool went_back = err == hipSuccess && e->h_out->back != 0;
    // two page registers: the tags the run leaves, unless it is timed again
    if (err == hipSuccess && k2 && !went_back) {
        err = hipMemcpyAsync(e->d_ptag, k2_tags.data(), k2_tags.size() * 8, hipMemcpyHostToDevice,
                             stream);
        if (err == hipSuccess) err = hipStreamSynchronize(stream);
    }
    if (err == hipSuccess && hit_lease) {
        hit_lease->synced(err);
    }
    hit_lease.reset();
    free_group();
    if (err != hipSuccess) {
        return HBFSIM_CUDA_ERROR;
    }
    if (went_back) {
        // Some record's issue time went back: the engine state is as the run
        // found it.  The stream is served in (issue time, position) order,
        // from a sorted copy, which the entry point without allocation
        // cannot make.
        if (ext_scratch != nullptr) {
            return HBFSIM_INVALID_ARGUMENT;
        }
        return run_in_issue_order(
            d_rec, packed, n, d_comp, d_status, stream_ptr,
            [&](const void* sorted, std::uint64_t* comp, std::uint8_t* status) {
                return engine_run_any(e, sorted, packed, n, comp, status, base_ps, stream_ptr,
                                      out, refresh_records, nullptr, true);
            });
    }
    e->last_modeled = e->h_out->rep.v[R_MODELED];
    e->last_hits = e->h_out->rep.v[R_HITS];
    if (ext_scratch == nullptr) {
        e->last_tiles = ntiles;
        e->last_passes = plain_alone   ? engine::Passes::scattered
                         : plain_mixed ? engine::Passes::both
                                       : engine::Passes::batched;
    }
    note_times(e);
    if (out != nullptr) {
        std::memcpy(out, &e->h_out->rep, sizeof(DevReport));
        if (grouping) {
            // the joined records: modeled, read or write, their latencies
            out->grouped = h_frep[0];
            out->modeled += h_frep[0];
            out->reads += h_frep[1];
            out->writes += h_frep[2];
            out->makespan_ps = std::max<std::uint64_t>(out->makespan_ps, h_frep[3]);
            const std::uint64_t lo = out->latency_sum_lo + h_frep[4];
            out->latency_sum_hi += h_frep[5] + (lo < out->latency_sum_lo ? 1u : 0u);
            out->latency_sum_lo = lo;
            out->latency_max_ps = std::max<std::uint64_t>(out->latency_max_ps, h_frep[6]);
        }
    }
    return HBFSIM_OK;
}

int engine_run_host(engine* e, const hbf_record32* records, std::size_t n,
                    std::uint64_t* completion, std::uint8_t* status, std::uint64_t base_ps,
                    hbfsim_amd_report* out)
{
    if (out != nullptr) {
        std::memset(out, 0, sizeof(*out));
    }
    if (n == 0) {
        return HBFSIM_OK;
    }
    if (records == nullptr || completion == nullptr) {
        return HBFSIM_INVALID_ARGUMENT;
    }
    if (hipSetDevice(e->device) != hipSuccess) {
        return HBFSIM_CUDA_ERROR;
    }
    hbf_record32* d_rec = nullptr;
    std::uint64_t* d_comp = nullptr;
    std::uint8_t* d_st = nullptr;
    hipError_t err = halloc(d_rec, n);
    if (err == hipSuccess) err = halloc(d_comp, n);
    if (err == hipSuccess && status != nullptr) err = halloc(d_st, n);
    if (err == hipSuccess)
        err = hipMemcpy(d_rec, records, n * sizeof(hbf_record32), hipMemcpyHostToDevice);
    int st = hip_status(err);
    if (st == HBFSIM_OK) {
        st = engine_run(e, d_rec, n, d_comp, d_st, base_ps, nullptr, out);
    }
    if (st == HBFSIM_OK) {
        err = hipMemcpy(completion, d_comp, n * 8, hipMemcpyDeviceToHost);
        if (err == hipSuccess && status != nullptr)
            err = hipMemcpy(status, d_st, n, hipMemcpyDeviceToHost);
        st = hip_status(err);
    }
    hfree(d_rec);
    hfree(d_comp);
    hfree(d_st);
    return st;
}

int engine_get_busy_totals(engine* e, std::uint64_t* plane_ps, std::size_t planes,
                           std::uint64_t* channel_ps, std::size_t channels)
{
    if (hipSetDevice(e->device) != hipSuccess) {
        return HBFSIM_CUDA_ERROR;
    }
    if (plane_ps != nullptr) {
        if (planes < e->args.Rp) return HBFSIM_INVALID_ARGUMENT;
        if (hipMemcpy(plane_ps, e->d_ptot, e->args.Rp * 8ull, hipMemcpyDeviceToHost) != hipSuccess)
            return HBFSIM_CUDA_ERROR;
    }
    if (channel_ps != nullptr) {
        if (channels < e->args.Rc) return HBFSIM_INVALID_ARGUMENT;
        if (hipMemcpy(channel_ps, e->d_ctot, e->args.Rc * 8ull, hipMemcpyDeviceToHost) !=
            hipSuccess)
            return HBFSIM_CUDA_ERROR;
    }
    return HBFSIM_OK;
}

int engine_get_state(engine* e, std::uint64_t* plane_busy, std::uint64_t* plane_tags,
                     std::uint64_t* channel_cursor, std::uint64_t* sequence, std::uint64_t* burst)
{
    if (hipSetDevice(e->device) != hipSuccess) {
        return HBFSIM_CUDA_ERROR;
    }
    const std::size_t rp = e->args.Rp, rc = e->args.Rc;
    hipError_t err = hipSuccess;
    if (plane_busy) err = hipMemcpy(plane_busy, e->d_pbusy, rp * 8, hipMemcpyDeviceToHost);
    if (err == hipSuccess && plane_tags)
        err = hipMemcpy(plane_tags, e->d_ptag, rp * 16, hipMemcpyDeviceToHost);
    if (err == hipSuccess && channel_cursor)
        err = hipMemcpy(channel_cursor, e->d_cbusy, rc * 8, hipMemcpyDeviceToHost);
    if (err == hipSuccess && sequence)
        err = hipMemcpy(sequence, e->d_seq, 8, hipMemcpyDeviceToHost);
    if (burst) *burst = e->burst;
    return hip_status(err);
}

int engine_set_state(engine* e, const std::uint64_t* plane_busy, const std::uint64_t* plane_tags,
                     const std::uint64_t* channel_cursor, std::uint64_t sequence,
                     std::uint64_t burst)
{
    if (hipSetDevice(e->device) != hipSuccess) {
        return HBFSIM_CUDA_ERROR;
    }
    const std::size_t rp = e->args.Rp, rc = e->args.Rc;
    hipError_t err = hipSuccess;
    if (plane_busy) err = hipMemcpy(e->d_pbusy, plane_busy, rp * 8, hipMemcpyHostToDevice);
    if (err == hipSuccess && plane_tags)
        err = hipMemcpy(e->d_ptag, plane_tags, rp * 16, hipMemcpyHostToDevice);
    if (err == hipSuccess && channel_cursor)
        err = hipMemcpy(e->d_cbusy, channel_cursor, rc * 8, hipMemcpyHostToDevice);
    if (err == hipSuccess) err = hipMemcpy(e->d_seq, &sequence, 8, hipMemcpyHostToDevice);
    e->burst = burst;
    return hip_status(err);
}

int engine_last_kernel_ms(const engine* e, float* ms, int max_kernels)
{
    const int k = std::min(3, max_kernels);
    for (int i = 0; i < k; ++i) {
        ms[i] = e->last_ms[i];
    }
    return k;
}

int engine_last_apply_waves(const engine* e)
{
    return e->last_apply_waves;
}

int engine_last_tiles(const engine* e, std::uint64_t* batched, std::uint64_t* scattered)
{
    *batched = e->last_passes == engine::Passes::batched ? e->last_tiles : 0;
    *scattered = e->last_passes == engine::Passes::scattered ? e->last_tiles : 0;
    if (e->last_passes != engine::Passes::both) {
        return HBFSIM_OK;
    }
    try {
        std::vector<std::uint8_t> kind(e->last_tiles);
        if (hipSetDevice(e->device) != hipSuccess ||
            hipMemcpy(kind.data(), e->d_tsplit, kind.size(), hipMemcpyDeviceToHost) !=
                hipSuccess) {
            return HBFSIM_CUDA_ERROR;
        }
        *scattered = static_cast<std::uint64_t>(std::count(kind.begin(), kind.end(), kTilePlain));
        *batched = kind.size() - *scattered;
    } catch (const std::bad_alloc&) {
        return HBFSIM_CUDA_ERROR;
    }
    return HBFSIM_OK;
}

int engine_window_counts(engine* e, const hbf_record32* d_rec, std::size_t n,
                         std::uint64_t window_ps, std::uint64_t windows, std::uint32_t* d_counts,
                         void* stream_ptr)
{
    if (n == 0) {
        return HBFSIM_OK;
    }
    if (d_rec == nullptr || d_counts == nullptr || window_ps == 0 ||
        (reinterpret_cast<std::uintptr_t>(d_rec) & 15u) != 0) {
        return HBFSIM_INVALID_ARGUMENT;
    }
    hipStream_t stream = static_cast<hipStream_t>(stream_ptr);
    if (hipSetDevice(e->device) != hipSuccess) {
        return HBFSIM_CUDA_ERROR;
    }
    if (e->ranges_dirty) {
        const int st = upload_ranges(e, stream);
        if (st != HBFSIM_OK) {
            return st;
        }
    }
    const KArgs& a = e->args;
    const std::uint32_t ndie = a.Rp / a.P;
    const std::size_t lds = 8ull * a.r_nfence + 4ull * kCountBins;
    const std::size_t blocks = (n + kCountChunk - 1) / kCountChunk;
    hipLaunchKernelGGL(k_window_counts, dim3(static_cast<unsigned>(blocks)), dim3(256), lds, stream,
                       a, d_rec, n, window_ps, windows, ndie, d_counts);
    return hip_status(hipGetLastError());
}

}  // namespace hbfamd
