// Device pieces of the halo-staged convs, shared by conv_halo.hip and
// conv_fold.hip: a tile's deduplication, its gather-plan record, and the LDS
// layout that the kernels stage rows in.
#pragma once

#include "conv_kernels.hpp"

#include <type_traits>

namespace s3dx {
namespace {

// s_waitcnt immediate waiting for vmcnt <= n (expcnt, lgkmcnt left at their maxima).
constexpr int vmcnt_imm(int n) { return (n & 15) | ((n >> 4) << 14) | 0x0F70; }

// f(integral_constant<int, I>) for I = B..E-1, unrolled at compile time.
template <int B, int E, class F>
__device__ __forceinline__ void static_for(F &&f) {
    if constexpr (B < E) {
        f(std::integral_constant<int, B>{});
        static_for<B + 1, E>(f);
    }
}

constexpr int kHChunk = 64;              // channels per halo chunk
constexpr int kHRowBytes = kHChunk * 2;  // 128 bytes per halo row

// 16-byte piece p of halo slot s sits at position p ^ halo_swizzle(s) of
// the slot's 128-byte row, so eight consecutive slots (the usual neighbours
// of consecutive output rows) read by one 16-byte LDS access spread over
// the eight positions.  ((s >> 1) & 7, which also separates 16 consecutive
// slots, halves the bank-conflict cycles but measured 1.5% slower.)
__device__ __forceinline__ int halo_swizzle(int s) { return s & 7; }
// Byte offset of slot s's row with its swizzle folded in: piece p of the
// slot sits at halo_offset(s) ^ (p << 4) (the row offset has bits 4-6 clear).
__device__ __forceinline__ uint32_t halo_offset(uint32_t s) {
    return s * kHRowBytes | static_cast<uint32_t>(halo_swizzle(static_cast<int>(s))) << 4;
}

template <int MB>
struct HaloSmem {
    static constexpr int ROWS = 32 * MB;
    static constexpr int RPH = MB == 4 ? 2 : 1;                  // row blocks reduced per phase
    static constexpr int CAP = MB == 4 ? 1088 : 511;             // halo rows (slot CAP is the zero row)
    static constexpr int BITWORDS = MB == 4 ? 1024 : 512;        // bitmap words (32 source rows each)
    static constexpr int ENTRIES = ROWS * kMaxKvol;
    static constexpr int STG_LD = 128 + 8;                       // padded FP32 output-tile row
    static constexpr int HALO_BYTES = (CAP + 1) * kHRowBytes;
    static constexpr int RED_BYTES = RPH * 4 * 4 * 4096;         // one reduction phase
    static constexpr int STG_BYTES = ROWS * STG_LD * 4 + 2 * ROWS * 16 * 4;
    static constexpr int R0A = HALO_BYTES > RED_BYTES ? HALO_BYTES : RED_BYTES;
    static constexpr int REGION0 = R0A > STG_BYTES ? R0A : STG_BYTES;
    static constexpr int TABLE_OFF = REGION0;
    static constexpr int BITMAP_OFF = TABLE_OFF + (ENTRIES * 2 + 15) / 16 * 16;
    static constexpr int PREFIX_OFF = BITMAP_OFF + BITWORDS * 4;
    static constexpr int ROWS_OFF = PREFIX_OFF + BITWORDS * 4;
    static constexpr int MISC_OFF = ROWS_OFF + (CAP * 4 + 15) / 16 * 16;
    static constexpr int TOTAL = MISC_OFF + 64;
    static_assert(TOTAL <= (MB == 4 ? 160 * 1024 : 80 * 1024), "LDS budget (two workgroups per CU for MB 2)");
    // The global-gather mode keeps 32-bit source rows (or -1) in region0,
    // which that mode does not use as a halo.
    static_assert(ENTRIES * 4 <= REGION0, "32-bit table fits region0");
};

// Wave-wide reductions through DPP (each 16-lane row by rotations, then the
// four rows by readlane); the result is wave-uniform.
__device__ __forceinline__ int dpp_ror(int x, int n) {
    switch (n) {
    case 8: return __builtin_amdgcn_update_dpp(0, x, 0x128, 0xf, 0xf, false);
    case 4: return __builtin_amdgcn_update_dpp(0, x, 0x124, 0xf, 0xf, false);
    case 2: return __builtin_amdgcn_update_dpp(0, x, 0x122, 0xf, 0xf, false);
    default: return __builtin_amdgcn_update_dpp(0, x, 0x121, 0xf, 0xf, false);
    }
}
template <class Op>
__device__ __forceinline__ int wave_reduce(int x, Op op) {
    x = op(x, dpp_ror(x, 8));
    x = op(x, dpp_ror(x, 4));
    x = op(x, dpp_ror(x, 2));
    x = op(x, dpp_ror(x, 1));
    return op(op(__builtin_amdgcn_readlane(x, 0), __builtin_amdgcn_readlane(x, 16)),
              op(__builtin_amdgcn_readlane(x, 32), __builtin_amdgcn_readlane(x, 48)));
}

// Exclusive prefix over the workgroup (256 threads) of one value each;
// returns the prefix, writes the total to *total.  Every thread must call it.
template <int WAVES = 4>
__device__ __forceinline__ uint32_t block_exclusive_scan(uint32_t v, uint32_t *wave_sums, uint32_t *total) {
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    uint32_t incl = v;
#pragma unroll
    for (int d = 1; d < 64; d <<= 1) {
        const uint32_t t = __shfl_up(incl, d, 64);
        if (lane >= d) incl += t;
    }
    if (lane == 63) wave_sums[wave] = incl;
    __syncthreads();
    uint32_t base = 0, all = 0;
#pragma unroll
    for (int w = 0; w < WAVES; ++w) {
        base += w < wave ? wave_sums[w] : 0u;
        all += wave_sums[w];
    }
    *total = all;
    return base + incl - v;
}

// Steps 1-4 of a tile's prologue: the tile's map slice deduplicated into LDS
// -- the [27][ROWS] slot table (or, when the slice cannot be staged, the
// 32-bit source-row table), the source row of every slot -- and the offset
// mask.  Every thread of the workgroup must call it; ends with a barrier.
struct TileDedupe {
    uint32_t mask, distinct;
    bool global_a;
};
// The tile's map slice read from memory: entries 4u..4u+3 of the tile
// (16-byte aligned, ROWS * 108 bytes per tile) by one unconditional 16-byte
// buffer load, whose resource ends at the map's last entry: a buffer load
// zero-fills each dword past the resource (checked on gfx950), and
// dedupe_tile marks entries past `count` invalid whatever they read.  (A
// load under a condition would compile to a branch, and the compiler waits
// for each such load at its join.)
struct SliceLoad {
    const int32_t *kmap;
    int32_t bytes;  // the map's size in bytes (rows * 108, under 2 GiB)
    __device__ __forceinline__ int4 operator()(int64_t m0, int u, int) const {
        const auto r = __builtin_amdgcn_make_buffer_rsrc(const_cast<int32_t *>(kmap), static_cast<short>(0), bytes,
                                                         0x00020000);
        const u32x4 v =
            __builtin_amdgcn_raw_buffer_load_b128(r, static_cast<int32_t>((m0 * kMaxKvol + 4 * u) * 4), 0, 0);
        return make_int4(static_cast<int32_t>(v.x), static_cast<int32_t>(v.y), static_cast<int32_t>(v.z),
                         static_cast<int32_t>(v.w));
    }
};

template <int MB, bool ENTRY_ORDER = false, int NTH = 256, class Fetch = SliceLoad>
__device__ __forceinline__ TileDedupe dedupe_tile(Fetch fetch, int64_t n_src, int32_t row_shift, int64_t m0,
                                                  int tile_rows, uint16_t *table, int32_t *table32,
                                                  uint32_t *bitmap, uint32_t *prefix, uint32_t *slot_row,
                                                  int32_t *misc) {
    using SM = HaloSmem<MB>;
    constexpr int ROWS = SM::ROWS, CAP = SM::CAP, ENTRIES = SM::ENTRIES;
    const int tid = threadIdx.x, lane = tid & 63;
    // ---- 1. this tile's map slice (ROWS * 27 entries) from `fetch`, as
    // source rows (-1: missing)
    constexpr int V4 = ENTRIES / 4;
    constexpr int Q = (V4 + NTH - 1) / NTH;
    const int count = tile_rows * kMaxKvol;
    int sj[Q][4];
    {
        // (slots past the slice fetch its last piece again and are marked
        // invalid below: a fetch under `u < V4` would be a branch, and the
        // compiler waits for each such load at its join)
#pragma unroll
        for (int q = 0; q < Q; ++q) {
            const int u = tid + q * NTH;
            const int4 v = fetch(m0, min(u, V4 - 1), count);
            const int jv[4] = {v.x, v.y, v.z, v.w};
#pragma unroll
            for (int k = 0; k < 4; ++k) {
                const bool valid = u < V4 && 4 * u + k < count && jv[k] >= 0 && jv[k] < n_src;
                sj[q][k] = valid ? (jv[k] >> row_shift) : -1;
            }
        }
    }
    // ---- 2. range of named source rows and the offset mask (the range,
    // mask and bitmap are reset while the slice's loads are in flight)
    if (tid == 0) {
        misc[0] = INT32_MAX;
        misc[1] = INT32_MIN;
        misc[2] = 0;
    }
    for (int w = tid; w < SM::BITWORDS; w += NTH) bitmap[w] = 0u;
    __syncthreads();
    {
        int lo = INT32_MAX, hi = INT32_MIN, m = 0;
#pragma unroll
        for (int q = 0; q < Q; ++q)
#pragma unroll
            for (int k = 0; k < 4; ++k)
                if (sj[q][k] >= 0) {
                    lo = min(lo, sj[q][k]);
                    hi = max(hi, sj[q][k]);
                    m |= 1 << ((4 * (tid + q * NTH) + k) % kMaxKvol);
                }
        lo = wave_reduce(lo, [](int x, int y) { return min(x, y); });
        hi = wave_reduce(hi, [](int x, int y) { return max(x, y); });
        m = wave_reduce(m, [](int x, int y) { return x | y; });
        if (lane == 0) {
            atomicMin(&misc[0], lo);
            atomicMax(&misc[1], hi);
            atomicOr(&misc[2], m);
        }
        __syncthreads();
    }
    const int rlo = misc[0], rhi = misc[1];
    const uint32_t mask = __builtin_amdgcn_readfirstlane(static_cast<uint32_t>(misc[2]));
    const int64_t span = rhi >= rlo ? static_cast<int64_t>(rhi) - rlo + 1 : 0;
    bool global_a = span > static_cast<int64_t>(SM::BITWORDS) * 32;
    uint32_t distinct = 0;
    if (!global_a && span > 0) {
        // ---- 3. bitmap of named rows -> slot = rank among them
        const int words = static_cast<int>((span + 31) / 32);
#pragma unroll
        for (int q = 0; q < Q; ++q)
#pragma unroll
            for (int k = 0; k < 4; ++k)
                if (sj[q][k] >= 0) {
                    const uint32_t r = static_cast<uint32_t>(sj[q][k] - rlo);
                    atomicOr(&bitmap[r >> 5], 1u << (r & 31));
                }
        __syncthreads();
        constexpr int WPT = SM::BITWORDS / NTH;  // words per thread
        uint32_t cnt[WPT], mine = 0;
#pragma unroll
        for (int k = 0; k < WPT; ++k) {
            const int w = tid * WPT + k;
            cnt[k] = w < words ? static_cast<uint32_t>(__popc(bitmap[w])) : 0u;
            mine += cnt[k];
        }
        uint32_t run = block_exclusive_scan<NTH / 64>(mine, reinterpret_cast<uint32_t *>(misc + 4), &distinct);
#pragma unroll
        for (int k = 0; k < WPT; ++k) {
            const int w = tid * WPT + k;
            if (w < words) prefix[w] = run;
            run += cnt[k];
        }
        global_a = distinct > static_cast<uint32_t>(CAP);
        __syncthreads();
    }
    // ---- 4. the slot (or, gathering from memory, the row) of every entry,
    // and the source row of every slot
#pragma unroll
    for (int q = 0; q < Q; ++q)
#pragma unroll
        for (int k = 0; k < 4; ++k) {
            const int e = 4 * (tid + q * NTH) + k;
            if (e >= ENTRIES) continue;
            const int r = e / kMaxKvol, o = e - r * kMaxKvol;
            const int ti = ENTRY_ORDER ? e : o * ROWS + r;
            if (global_a) {
                table32[ti] = sj[q][k];
            } else {
                uint32_t slot = CAP;
                if (sj[q][k] >= 0) {
                    const uint32_t d = static_cast<uint32_t>(sj[q][k] - rlo);
                    const uint32_t bits = bitmap[d >> 5];
                    slot = prefix[d >> 5] + static_cast<uint32_t>(__popc(bits & ((1u << (d & 31)) - 1u)));
                    slot_row[slot] = static_cast<uint32_t>(sj[q][k]);  // writers of one slot agree
                }
                table[ti] = static_cast<uint16_t>(slot);
            }
        }
    __syncthreads();
    return TileDedupe{mask, distinct, global_a};
}

// Gather plans: one record per 64-row tile of a kernel map, the result of
// dedupe_tile kept in memory so that every conv over the map skips it:
//   [0, 16)     mode (0: halo, 1: global gathers), distinct rows, offset mask, 0
//   [16, ...)   halo: the u16 slot table [27][64], then at kPlanSlots the
//               source row of each slot; global: the int32 row table [27][64]
constexpr int kPlanHeader = 16;
constexpr int kPlanSlots = kPlanHeader + 64 * kMaxKvol * 2;  // 3472
static_assert(kPlanSlots + HaloSmem<2>::CAP * 4 <= kGatherPlanRecord, "halo record fits");
static_assert(kPlanHeader + 64 * kMaxKvol * 4 <= kGatherPlanRecord, "global record fits");
static_assert(kGatherPlanRecord % 1024 == 0, "records copy as whole 1 KiB pieces");

// 128-row records (the 8-wave kernel): the same header; halo tiles hold the
// source row of each slot right after it, then at kPlan128Table the u32
// table [27][128] of halo byte offsets (halo_offset of each slot); global
// tiles the int32 row table [27][128] at kPlan128Table.  The header and the
// rows come first so that a kernel can start copying rows while the table
// is still on its way.
constexpr int kPlan128Slots = kPlanHeader;     // 16
constexpr int kPlan128Table = 4608;
constexpr int kPlan128HeadPieces = (kPlan128Slots + HaloSmem<4>::CAP * 4 + 1023) / 1024;  // 5 KiB
static_assert(kPlan128Slots + HaloSmem<4>::CAP * 4 <= kPlan128Table, "halo record fits");
static_assert(kPlan128Table + 128 * kMaxKvol * 4 <= kGatherPlanRecord128, "tables fit");
static_assert(kGatherPlanRecord128 % 1024 == 0, "records copy as whole 1 KiB pieces");
// Halo layout of the 8-wave kernel: two buffers of kH8BufRows rows (one per
// chunk, the next chunk's copied while the current one is in use) with the
// zero row at slot kH8Double, or, for tiles naming more distinct rows, one
// buffer with the zero row at kH8Single.
constexpr int kH8BufRows = 560;
constexpr int kH8Double = kH8BufRows - 1;        // 559
constexpr int kH8Single = HaloSmem<4>::CAP;      // 1088
constexpr int kH8HaloBytes = 2 * kH8BufRows * kHRowBytes;
// 1 KiB after the halo that nothing reads: the last chunk sends its unneeded
// copy pieces (zero fills, which read no memory) there.
constexpr int kH8Dump = kH8HaloBytes;
constexpr int kH8Bytes = 160 * 1024;  // the kernel's LDS: halo, dump, plan record, padding
static_assert(kH8Dump + 1024 + kGatherPlanRecord128 <= kH8Bytes, "halo, dump and record fit");
// The record header's last word, 0 as the plan builder writes it: in LDS,
// the 8-wave kernel's arrival counter for the four waves of column half 0.
constexpr int kHalfCounter = 12;
static_assert((kH8Single + 1) * kHRowBytes <= kH8HaloBytes, "single buffer fits");
static_assert(kH8BufRows % 8 == 0, "buffers keep the slot swizzle");

template <int MB, bool PLAN>
struct HaloLds {
    // Planned kernels keep region0 and the copied record; unplanned ones the
    // dedupe buffers of HaloSmem.
    static constexpr int TOTAL = PLAN ? HaloSmem<MB>::REGION0 + kGatherPlanRecord + 64 : HaloSmem<MB>::TOTAL;
    static_assert(!PLAN || MB == 2, "plans are for 64-row tiles");
    static_assert(TOTAL <= (MB == 4 ? 160 * 1024 : 80 * 1024), "LDS budget");
};

// Threads of a plan build's workgroup (one per tile): the dedupe's short
// dependent steps run on 16 (128-row) or 8 (64-row) waves, one bitmap word
// and about four map entries per thread.
constexpr int kPlanBuild128Threads = 1024;
constexpr int kPlanBuild64Threads = 512;

// One workgroup per tile (64 or 128 rows): dedupe_tile, then the record to
// memory.  128-row records hold halo byte offsets and name missing
// neighbours by the zero row of the kernel's halo layout: slot kH8Single when
// the tile's distinct rows need the single large buffer, else kH8Double (two
// buffers, one per chunk).
template <int MB, int NTH, class Fetch>
__device__ __forceinline__ TileDedupe plan_tile(Fetch fetch, int64_t n_out, int64_t n_src, int32_t row_shift, char *plan) {
    using SM = HaloSmem<MB>;
    constexpr int ROWS = SM::ROWS;
    constexpr int REC = MB == 2 ? kGatherPlanRecord : kGatherPlanRecord128;
    constexpr int SLOTS = MB == 2 ? kPlanSlots : kPlan128Slots;
    __shared__ __align__(16) int32_t table32[ROWS * kMaxKvol];
    __shared__ __align__(16) uint16_t table[ROWS * kMaxKvol];
    __shared__ __align__(16) uint32_t bitmap[SM::BITWORDS];
    __shared__ __align__(16) uint32_t prefix[SM::BITWORDS];
    __shared__ __align__(16) uint32_t slot_row[SM::CAP];
    __shared__ __align__(16) int32_t misc[4 + NTH / 64];
    const int tile = xcd_tile(blockIdx.x, gridDim.x), tid = threadIdx.x;
    const int64_t m0 = static_cast<int64_t>(tile) * ROWS;
    const int tile_rows = static_cast<int>(min(static_cast<int64_t>(ROWS), n_out - m0));
    // The tables come back in entry order (row-major, 27 per row: no LDS
    // bank conflicts on writing them); the record stores them offset-major.
    const TileDedupe dd = dedupe_tile<MB, true, NTH>(fetch, n_src, row_shift, m0, tile_rows, table, table32, bitmap,
                                                     prefix, slot_row, misc);
    char *rec = plan + static_cast<int64_t>(tile) * REC;
    if (tid == 0)
        *reinterpret_cast<uint4 *>(rec) = make_uint4(dd.global_a ? 1u : 0u, dd.distinct, dd.mask, 0u);
    auto entry = [](int i) { return (i % ROWS) * kMaxKvol + i / ROWS; };  // record index -> entry
    constexpr int TABLE = MB == 2 ? kPlanHeader : kPlan128Table;
    if (dd.global_a) {
        for (int i = tid; i < ROWS * kMaxKvol; i += NTH)
            reinterpret_cast<int32_t *>(rec + TABLE)[i] = table32[entry(i)];
    } else {
        if constexpr (MB == 4) {
            const uint32_t z = dd.distinct <= static_cast<uint32_t>(kH8Double) ? kH8Double : kH8Single;
            for (int i = tid; i < ROWS * kMaxKvol; i += NTH) {
                const uint32_t sl = table[entry(i)];
                reinterpret_cast<uint32_t *>(rec + TABLE)[i] = halo_offset(sl == static_cast<uint32_t>(SM::CAP) ? z : sl);
            }
        } else {
            for (int i = tid; i < ROWS * kMaxKvol / 2; i += NTH)  // two rows of one offset per word
                reinterpret_cast<uint32_t *>(rec + kPlanHeader)[i] =
                    static_cast<uint32_t>(table[entry(2 * i)]) | static_cast<uint32_t>(table[entry(2 * i + 1)]) << 16;
        }
        for (int i = tid; i < static_cast<int>(dd.distinct); i += NTH)
            reinterpret_cast<uint32_t *>(rec + SLOTS)[i] = slot_row[i];
    }
    return dd;
}

}  // namespace
}  // namespace s3dx
