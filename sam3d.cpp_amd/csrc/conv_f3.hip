// FP32 3x3x3 convs on the BF16 matrix units: every FP32 value is the sum of
// three BF16 terms (8 significant bits each; each remainder is exact in FP32),
// and a product x w is the six term products above 2^-27 of it,
//     x1 w1 + (x1 w2 + x2 w1) + (x1 w3 + x2 w2 + x3 w1),
// accumulated in FP32: x1 w1 in one set of accumulators, the five small ones
// in another, added once at the end.  Six BF16 products cost 6/16 of the FP32
// ones at the nominal rates, and the sums round less often (16 channels a
// matrix instruction against 2).
//
// One workgroup of 8 waves per 128-row x (32 * CG)-column tile of a 128-row
// gather plan (conv_halo.hip), no barrier inside a chunk: wave (row half,
// column block, k part) owns 64 rows x 32 columns; KS > 1 splits the chunk's
// (offset, k-step) tasks over KS waves, whose tiles are added at the end in a
// fixed order.  Per 32-channel chunk the tile's distinct rows are read as
// FP32 (into registers, while the chunk before is multiplied), split once and
// kept in LDS as three planes; the weights' terms, split once per layer, come
// straight from memory.
//
// What bounds it: the BF16 matrix rate (six products: 128 -> 128 on 28,265
// rows is 150 GFLOP in 124-135 us, 1.1-1.2 PFLOP/s; 1024 -> 1024 on 5,086 1.73 TFLOP
// in 1,473 us, 1.2; a large BF16 product reaches 1.26 here); the split of the
// rows, about 2.5K of 44K cycles a chunk, is what is left between.  The FP32
// kernels took 204-226 and 1,986-2,004 us.  64 rows x 32 columns a wave: each
// weight fragment feeds two row blocks and each row fragment six products, so
// that neither LDS (64 B a cycle) nor the weights (32) is the limit and no wave
// holds a partial sum of another's outputs (with KS 1).
//
// Tiles that name more rows than the planes hold (719; a union of sphere
// shells names about 470 in 128 rows, 534 at most, a solid bar of 24 x 24 x 60 up
// to 768) are multiplied in two parts.  Tiles without slots (rows in no order) stage
// five offsets' rows at a time, or, with fewer than 128 columns a workgroup, gather
// rows from memory and split them in registers.  Tiles whose rows hold a value with
// no finite first term (infinities, NaN), or whose sums overflow, are done again
// with FP32 matrix instructions, so that such values spread as in any FP32 sum.
#include "halo_tile.hpp"

namespace s3dx {
namespace {

constexpr int kF3Chunk = 32;                               // channels per chunk
constexpr int kF3MostRows = 719;                           // distinct rows that it stages at once
constexpr int kF3Part = 712;                               // of more, the first (whole swizzle periods, one row fewer)
constexpr int kF3Rows = kF3MostRows + 1;                   // rows a plane holds (the last is the zero row)
constexpr int kF3Sum = 8;                                  // chunks of a sum
constexpr int kF3Offsets = 5;                              // offsets of 128 rows that it stages at once
static_assert(kF3Part % 8 == 0 && kF3Part < kF3MostRows && kH8Single - kF3Part < kF3Part, "two parts");
static_assert(kF3Offsets * 128 <= kF3MostRows, "five offsets' rows");
constexpr int kF3Plane = kF3Rows * kF3Chunk * 2;           // bytes of one term's plane
constexpr int kF3Rec = 3 * kF3Plane;                       // the plan record, behind the planes
constexpr int kF3Flag = kF3Rec + kGatherPlanRecord128;     // a row held a value without terms
constexpr int kF3Lds = kF3Flag + 16;
static_assert(128 * 128 * 4 <= kF3Rec, "the output tile overlays the planes");
static_assert(kF3Lds <= 160 * 1024, "LDS");

// Rows and weights are split at 2^24 times their value and sums brought back: every
// FP32 value, subnormal ones too, then has three normal terms (unscaled, values
// below 2^-110 would lose low bits).  Values from 2^104 on, and sums from 2^80 on,
// overflow at that scale: their tiles are done again with FP32 matrix instructions.
constexpr float kF3Scale = 0x1p24f, kF3Unscale = 0x1p-48f;

// Three terms of two (scaled) floats, packed (first value in the low half).
__device__ __forceinline__ void split3(float a, float b, uint32_t (&t)[3]) {
    a *= kF3Scale;
    b *= kF3Scale;
#pragma unroll
    for (int i = 0; i < 3; ++i) {
        t[i] = pack_bf16x2(a, b);
        a -= __builtin_bit_cast(float, t[i] << 16);
        b -= __builtin_bit_cast(float, t[i] & 0xffff0000u);
    }
}

// The layer's FP32 fragments ([offset][k-step of 8][column block][lane][4])
// as three-term BF16 fragments ([offset][k-step of 16][column block][term][lane][8]).
// *bad: a weight without three finite terms.
__global__ void __launch_bounds__(256) f3_weights_kernel(const uint4 *w, uint4 *out, int64_t frags, int nbtot, uint32_t *bad) {
    for (int64_t i = blockIdx.x * 256ll + threadIdx.x; i < frags; i += gridDim.x * 256ll) {
        const int lane = static_cast<int>(i & 63);
        const int64_t r = i >> 6;  // (offset, k-step of 16) * nbtot + column block
        const int64_t ks = r / nbtot, cb = r - ks * nbtot;
        const int64_t src = ((2 * ks + (lane >> 5)) * nbtot + cb) * 64 + (lane & 31);
        const uint4 v[2] = {w[src], w[src + 32]};
        uint32_t t[4][3];
#pragma unroll
        for (int h = 0; h < 2; ++h) {
            split3(__builtin_bit_cast(float, v[h].x), __builtin_bit_cast(float, v[h].y), t[2 * h]);
            split3(__builtin_bit_cast(float, v[h].z), __builtin_bit_cast(float, v[h].w), t[2 * h + 1]);
        }
        bool none = false;
#pragma unroll
        for (int e = 0; e < 4; ++e)
            none = none || (t[e][0] & 0x7f80u) == 0x7f80u || (t[e][0] & 0x7f800000u) == 0x7f800000u;
        if (none) *bad = 1u;
#pragma unroll
        for (int k = 0; k < 3; ++k) out[(r * 3 + k) * 64 + lane] = make_uint4(t[0][k], t[1][k], t[2][k], t[3][k]);
    }
}

// FOLD: the folded conv over repeated parent rows (conv_fold.hip: 8 parents'
// summed weights in place of 27 children's).  Wave s owns slot s of 64 of the
// tile's 128 parents and 32 columns; its offsets are the slot's 8 of the parent
// map's 27.  Tiles that the fold plan marks are left to the FP32 kernel behind.
template <int CG, int KS, bool FOLD = false>
__global__ void __launch_bounds__(kHalo8Threads, 1) conv_f3_kernel(ConvArgs a) {
    static_assert(FOLD ? CG == 1 && KS == 1 : 2 * CG * KS == 8, "eight waves");
    constexpr int ROWS = 128, NTH = kHalo8Threads, LD = 32 * CG;
    __shared__ __align__(16) char smem[kF3Lds];
    char *planes = smem;
    char *rec = smem + kF3Rec;
    uint32_t *flag = reinterpret_cast<uint32_t *>(smem + kF3Flag);
    const uint32_t *table = reinterpret_cast<const uint32_t *>(rec + kPlan128Table);
    const uint32_t *slot_row = reinterpret_cast<const uint32_t *>(rec + kPlan128Slots);
    const int tid = threadIdx.x, lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int half = lane >> 5;
    const int unit = xcd_tile(blockIdx.x, gridDim.x);
    const int tile = FOLD ? unit >> 1 : unit;
    const int rg = FOLD ? unit & 1 : wave & 1, cb = FOLD ? 0 : (wave >> 1) % CG, kp = FOLD ? 0 : (wave >> 1) / CG;
    const int64_t n_rows = FOLD ? a.n_out / 8 : a.n_out;  // rows of the plan's map
    const int64_t m0 = static_cast<int64_t>(tile) * ROWS;
    const int tile_rows = static_cast<int>(min(static_cast<int64_t>(ROWS), n_rows - m0));
    const int nb0 = blockIdx.y * CG;
    const int nbtot = a.cout_pad / 32;

    // ---- the record into LDS
    {
        const int64_t plan_bytes = (n_rows + ROWS - 1) / ROWS * kGatherPlanRecord128;
        const auto p_rsrc = __builtin_amdgcn_make_buffer_rsrc(const_cast<void *>(a.plan), static_cast<short>(0),
                                                              static_cast<int32_t>(plan_bytes), 0x00020000);
        constexpr int PIECES = kGatherPlanRecord128 / 1024;
#pragma unroll
        for (int k = 0; k < (PIECES + 7) / 8; ++k) {
            const int i = wave + 8 * k;
            if (i < PIECES)
                __builtin_amdgcn_raw_ptr_buffer_load_lds(
                    p_rsrc, (__attribute__((address_space(3))) void *)(rec + i * 1024), 16, lane * 16,
                    tile * kGatherPlanRecord128 + i * 1024, 0, 0);
        }
        if (tid < 16) reinterpret_cast<uint32_t *>(planes + (kF3Rows - 1) * 64)[tid] = 0u;
        else if (tid < 32) reinterpret_cast<uint32_t *>(planes + kF3Plane + (kF3Rows - 1) * 64)[tid - 16] = 0u;
        else if (tid < 48) reinterpret_cast<uint32_t *>(planes + 2 * kF3Plane + (kF3Rows - 1) * 64)[tid - 32] = 0u;
        else if (tid == 48) *flag = 0u;
        __builtin_amdgcn_s_waitcnt(0x0F70);  // vmcnt(0)
        __syncthreads();
    }
    const uint32_t *hdr = reinterpret_cast<const uint32_t *>(rec);
    const uint32_t mode = __builtin_amdgcn_readfirstlane(hdr[0]);
    const int distinct = static_cast<int>(__builtin_amdgcn_readfirstlane(hdr[1]));
    const uint32_t mask = __builtin_amdgcn_readfirstlane(hdr[2]);
    if (FOLD && mode != 0u) return;  // left to the FP32 kernel behind
    // What the planes hold at a time (a pass over a chunk): the tile's distinct
    // rows; of more than they have room for, the first kF3Part, then the rest; in a
    // tile without slots (mode 1) the 128 rows that each of five offsets names.
    const bool slots = FOLD || mode == 0u;
    const int passes = slots ? (distinct > kF3MostRows ? 2 : 1) : (__popc(mask) + kF3Offsets - 1) / kF3Offsets;
    const int width = passes > 1 ? kF3Part : kF3MostRows;  // distinct rows a pass

    const auto x_rsrc = __builtin_amdgcn_make_buffer_rsrc(const_cast<void *>(a.x), static_cast<short>(0),
                                                          static_cast<int32_t>(a.x_bytes), 0x00020000);
    // (sums of kF3Sum chunks, which are then added to the total: 2048 channels
    // added one after another had 1.03 times the FP32 kernels' error)
    f32x16 hi[2], lo[2], total[2];
#pragma unroll
    for (int mb = 0; mb < 2; ++mb) hi[mb] = lo[mb] = total[mb] = f32x16{};

    bool none = false;  // a value without three finite terms was met
    if (mask != 0u) {
        const int chunks = a.cin / kF3Chunk;
        const int ksteps = a.cin / 16;
        const auto w_rsrc = __builtin_amdgcn_make_buffer_rsrc(
            const_cast<void *>(a.w3), static_cast<short>(0),
            static_cast<int32_t>(static_cast<int64_t>(FOLD ? 64 : kMaxKvol) * a.cin * a.cout_pad * 6), 0x00020000);
        // The wave's offsets: all present ones; KS 4: every other one.
        uint32_t mine = mask;
        if constexpr (FOLD) {
            // an axis' own parent, or the neighbour on the slot's side
            const uint32_t z = (wave & 1) ? 6u : 3u;
            const uint32_t y = (wave & 2) ? z << 3 | z << 6 : z | z << 3;
            mine &= (wave & 4) ? y << 9 | y << 18 : y | y << 9;
        }
        if constexpr (KS == 4) {
            mine = 0u;
            int k = 0;
            for (uint32_t r = mask; r != 0u; r &= r - 1u, ++k)
                if ((k & 1) == (kp >> 1)) mine |= r & (0u - r);
        }
        // The table entry of row block mb of this wave's rows at offset o.
        auto entry = [&](int o, int mb) __attribute__((always_inline)) {
            return table[o * ROWS + rg * 64 + mb * 32 + (lane & 31)];
        };
        // Mode 1: the offsets of pass q.
        auto group = [&](int q) __attribute__((always_inline)) {
            uint32_t rest = mask;
            for (int k = 0; k < q * kF3Offsets; ++k) rest &= rest - 1u;
            uint32_t after = rest;
            for (int k = 0; k < kF3Offsets; ++k) after &= after - 1u;
            return rest & ~after;
        };
        // The wave's offsets in the two passes over slots: those that name one of
        // the pass's rows (of the next plane of the set few offsets do, so that the
        // second pass is a short one).
        uint32_t part[2] = {mine, mine};
        if (slots && passes > 1) {
            part[0] = part[1] = 0u;
            for (uint32_t r = mine; r != 0u; r &= r - 1u) {
                const int o = __builtin_ctz(r);
                bool first = false, second = false;
#pragma unroll
                for (int mb = 0; mb < 2; ++mb) {
                    const int sl = static_cast<int>(entry(o, mb) >> 7);
                    first = first || sl < kF3Part;
                    second = second || (sl >= kF3Part && sl < distinct);
                }
                if (__builtin_amdgcn_ballot_w64(first)) part[0] |= r & (0u - r);
                if (__builtin_amdgcn_ballot_w64(second)) part[1] |= r & (0u - r);
            }
        }
        uint32_t cur = mine;  // the wave's offsets in this pass, and the last of them
        int olast = 0;
        auto advance = [&](uint32_t &rest) __attribute__((always_inline)) {
            const int o = __builtin_ctz(rest | 0x80000000u);
            rest &= rest - 1u;
            return o == 31 ? olast : o;
        };
        // A pass's rows: piece i of a thread is channels 4j .. 4j + 3 of place
        // 64 i + tid / 8, j = tid % 8 (eight lanes read a row's 128 bytes).
        constexpr int XP = (kF3Rows + 63) / 64;  // 12
        u32x4 xq[XP];
        auto load_x = [&](auto by_slot, int c, int q) __attribute__((always_inline)) {
            // (24-bit products: rows of at least 128 bytes, x below 2 GiB; the top
            // bit, set last: past the rows, zeros)
            const uint32_t p16 = (tid & 7) * 16u;
            uint32_t off[XP];
            if constexpr (by_slot.value) {
#pragma unroll
                for (int i = 0; i < XP; ++i) {
                    const int at = 64 * i + (tid >> 3), sl = at + q * kF3Part;
                    off[i] = (__umul24(slot_row[min(sl, kH8Single - 1)], 4u * static_cast<uint32_t>(a.cin)) + p16) |
                             (at < width && sl < distinct ? 0u : 0x80000000u);
                }
            } else {
                uint32_t rest = group(q);
#pragma unroll
                for (int i = 0; i < XP; ++i) {
                    const int o = __builtin_ctz(rest | 0x80000000u);
                    const uint32_t row = table[min(o, kMaxKvol - 1) * ROWS + 64 * (i & 1) + (tid >> 3)];
                    off[i] = (__umul24(row, 4u * static_cast<uint32_t>(a.cin)) + p16) |
                             (o < kMaxKvol && static_cast<int32_t>(row) >= 0 ? 0u : 0x80000000u);
                    if (i & 1) rest &= rest - 1u;
                }
            }
#pragma unroll
            for (int i = 0; i < XP; ++i)
                xq[i] = __builtin_amdgcn_raw_buffer_load_b128(x_rsrc, static_cast<int32_t>(off[i]), c * (kF3Chunk * 4), 0);
        };
        auto store_x = [&](char *p) __attribute__((always_inline)) {
#pragma unroll
            for (int i = 0; i < XP; ++i) {
                const int sl = 64 * i + (tid >> 3);
                uint32_t t0[3], t1[3];
                // (copied first: a bit cast of a vector's element takes element 0)
                const uint32_t v[4] = {xq[i].x, xq[i].y, xq[i].z, xq[i].w};
                split3(__builtin_bit_cast(float, v[0]), __builtin_bit_cast(float, v[1]), t0);
                split3(__builtin_bit_cast(float, v[2]), __builtin_bit_cast(float, v[3]), t1);
                none = none || (t0[0] & 0x7f80u) == 0x7f80u || (t0[0] & 0x7f800000u) == 0x7f800000u ||
                       (t1[0] & 0x7f80u) == 0x7f80u || (t1[0] & 0x7f800000u) == 0x7f800000u;
                // 16-byte piece q of slot s sits at q ^ ((s >> 1) & 3) of its 64 bytes
                char *dst = p + sl * 64 + ((((tid & 7) >> 1) ^ ((sl >> 1) & 3)) << 4) + (tid & 1) * 8;
                if (sl < kF3Rows - 1) {
#pragma unroll
                    for (int k = 0; k < 3; ++k) *reinterpret_cast<uint2 *>(dst + k * kF3Plane) = make_uint2(t0[k], t1[k]);
                }
            }
        };
        uint4 bq[2][3], aq[2][2][3];
        uint32_t ix[2];
        // (chunk c, offset o, k): this wave's three term fragments
        auto load_b = [&](int c, int o, int k, uint4 (&b)[3]) __attribute__((always_inline)) {
            // folded weights: [slot][group], the group's bits the axes on which
            // o is the own parent
            const int wo = FOLD ? wave * 8 + ((o / 9 == 1) << 2 | (o / 3 % 3 == 1) << 1 | int(o % 3 == 1)) : o;
            const int32_t sbase = ((wo * ksteps + c * 2 + k) * nbtot + nb0 + cb) * 3072;
#pragma unroll
            for (int t = 0; t < 3; ++t) {
                const u32x4 v = __builtin_amdgcn_raw_buffer_load_b128(w_rsrc, lane * 16, sbase + t * 1024, 0);
                b[t] = make_uint4(v.x, v.y, v.z, v.w);
            }
        };
        // The record's offsets are 128-byte ones (slot * 128 | swizzle): the
        // slot's 64 bytes and this kernel's swizzle from the same bits (kF3Part
        // slots keep the swizzle).  A missing neighbour is the record's zero slot,
        // 559 or 1088, past the rows of every tile that uses it: zeros; a slot of the
        // other pass is the place after this pass's, zeros too, as is the last row.
        uint32_t base = 0;   // bytes of the slots before this pass's
        uint32_t grp = 0;    // mode 1: the pass's offsets
        const uint32_t limit = static_cast<uint32_t>(passes > 1 ? kF3Part : kF3Rows - 1) * 64u;
        auto load_ix = [&](auto by_slot, int o) __attribute__((always_inline)) {
            if constexpr (by_slot.value) {
#pragma unroll
                for (int mb = 0; mb < 2; ++mb) {
                    const uint32_t v = entry(o, mb);
                    ix[mb] = min(((v >> 1) & ~63u) - base, limit) | (((v >> 4) & 0x30u) ^ (half << 4));
                }
            } else {
                const int j = __popc(grp & ((1u << o) - 1u));
#pragma unroll
                for (int mb = 0; mb < 2; ++mb) {
                    const int at = min(j, kF3Offsets - 1) * ROWS + rg * 64 + mb * 32 + (lane & 31);
                    ix[mb] = static_cast<uint32_t>(at * 64 + ((((at >> 1) & 3) ^ half) << 4));
                }
            }
        };
        auto load_a = [&](const char *p, int k, uint4 (&af)[2][3]) __attribute__((always_inline)) {
#pragma unroll
            for (int mb = 0; mb < 2; ++mb)
#pragma unroll
                for (int t = 0; t < 3; ++t)
                    af[mb][t] = *reinterpret_cast<const uint4 *>(p + t * kF3Plane + (ix[mb] ^ (k << 5)));
        };
        auto products = [&](const uint4 (&af)[2][3], const uint4 (&b)[3]) __attribute__((always_inline)) {
#pragma unroll
            for (int mb = 0; mb < 2; ++mb) lo[mb] = mfma_step<uint16_t>(af[mb][2], b[0], lo[mb]);
#pragma unroll
            for (int mb = 0; mb < 2; ++mb) lo[mb] = mfma_step<uint16_t>(af[mb][1], b[1], lo[mb]);
#pragma unroll
            for (int mb = 0; mb < 2; ++mb) lo[mb] = mfma_step<uint16_t>(af[mb][0], b[2], lo[mb]);
#pragma unroll
            for (int mb = 0; mb < 2; ++mb) lo[mb] = mfma_step<uint16_t>(af[mb][1], b[0], lo[mb]);
#pragma unroll
            for (int mb = 0; mb < 2; ++mb) lo[mb] = mfma_step<uint16_t>(af[mb][0], b[1], lo[mb]);
#pragma unroll
            for (int mb = 0; mb < 2; ++mb) hi[mb] = mfma_step<uint16_t>(af[mb][0], b[0], hi[mb]);
        };
        auto multiply = [&](auto by_slot) __attribute__((always_inline)) {
            load_x(by_slot, 0, 0);
            for (int c = 0, q = 0; c < chunks;) {
                if constexpr (!by_slot.value) grp = group(q);
                cur = by_slot.value ? part[q] : mine & grp;
                olast = cur != 0u ? 31 - __builtin_clz(cur) : 0;
                base = static_cast<uint32_t>(q) * (kF3Part * 64u);
                const int n = __popc(cur);
                const int qn = q + 1 < passes ? q + 1 : 0, cn = qn ? c : c + 1;
                // the pass's first weights, in flight while its rows are split
                uint32_t rest_b = cur, rest_i = cur;
                if constexpr (KS == 1) {
                    const int o = advance(rest_b);
                    load_b(c, o, 0, bq[0]);
                    load_b(c, o, 1, bq[1]);
                } else {
                    load_b(c, advance(rest_b), kp & 1, bq[0]);
                    load_b(c, advance(rest_b), kp & 1, bq[1]);
                }
                if (c + q > 0) __syncthreads();  // every wave is done with the planes
                store_x(planes);
                __syncthreads();
                if (cn < chunks) load_x(by_slot, cn, qn);
                sched_fence();
                load_ix(by_slot, advance(rest_i));
                if constexpr (KS == 1) {
                    load_a(planes, 0, aq[0]);
                    for (int i = 0; i < n; ++i) {
                        const int o = advance(rest_b);
                        load_a(planes, 1, aq[1]);
                        load_ix(by_slot, advance(rest_i));
                        products(aq[0], bq[0]);
                        sched_fence();
                        load_b(c, o, 0, bq[0]);
                        load_a(planes, 0, aq[0]);
                        products(aq[1], bq[1]);
                        sched_fence();
                        load_b(c, o, 1, bq[1]);
                    }
                } else {
                    const int k = kp & 1;
                    load_a(planes, k, aq[0]);
                    load_ix(by_slot, advance(rest_i));
                    int i = 0;
                    for (; i + 2 <= n; i += 2) {
                        load_a(planes, k, aq[1]);
                        load_ix(by_slot, advance(rest_i));
                        products(aq[0], bq[0]);
                        sched_fence();
                        load_b(c, advance(rest_b), k, bq[0]);
                        load_a(planes, k, aq[0]);
                        load_ix(by_slot, advance(rest_i));
                        products(aq[1], bq[1]);
                        sched_fence();
                        load_b(c, advance(rest_b), k, bq[1]);
                    }
                    if (i < n) products(aq[0], bq[0]);
                }
                if (cn != c && cn % kF3Sum == 0 && cn < chunks)
#pragma unroll
                    for (int mb = 0; mb < 2; ++mb) {
#pragma unroll
                        for (int r = 0; r < 16; ++r) total[mb][r] += hi[mb][r];
                        hi[mb] = f32x16{};
                    }
                c = cn;
                q = qn;
            }
        };
        if (slots) {
            multiply(std::true_type{});
        } else if constexpr (KS == 1 && !FOLD) {
            multiply(std::false_type{});
        } else if constexpr (KS > 1) {
            // (with fewer columns a workgroup, staging five offsets' rows takes longer
            // than their products: 192 -> 192 on 65,536 shuffled rows 1,181 us against
            // 943, 64 -> 64 on 28,265 80 against 66)
            // Rows from memory, split in registers: channels 16 k + 8 half .. + 7
            // of the lane's row for every (offset, k-step) of this wave.
            uint4 raw[2][2][2];  // [set][row block][16-byte half]
            auto load_raw = [&](const int32_t (&row)[2], int ks, uint4 (&q)[2][2]) __attribute__((always_inline)) {
#pragma unroll
                for (int mb = 0; mb < 2; ++mb)
#pragma unroll
                    for (int h = 0; h < 2; ++h)
                        q[mb][h] = gather_plain<float>(a.x, static_cast<int32_t>(a.x_bytes), row[mb], a.cin,
                                                       ks * 16 + half * 8 + h * 4);
            };
            auto split_raw = [&](const uint4 (&q)[2][2], uint4 (&af)[2][3]) __attribute__((always_inline)) {
#pragma unroll
                for (int mb = 0; mb < 2; ++mb) {
                    const uint32_t v[8] = {q[mb][0].x, q[mb][0].y, q[mb][0].z, q[mb][0].w,
                                           q[mb][1].x, q[mb][1].y, q[mb][1].z, q[mb][1].w};
                    uint32_t t[4][3];
#pragma unroll
                    for (int e = 0; e < 4; ++e) {
                        split3(__builtin_bit_cast(float, v[2 * e]), __builtin_bit_cast(float, v[2 * e + 1]), t[e]);
                        none = none || (t[e][0] & 0x7f80u) == 0x7f80u || (t[e][0] & 0x7f800000u) == 0x7f800000u;
                    }
#pragma unroll
                    for (int k = 0; k < 3; ++k) af[mb][k] = make_uint4(t[0][k], t[1][k], t[2][k], t[3][k]);
                }
            };
            // k-steps kp, kp + KS, ... of the layer's
            for (uint32_t rest = mask; rest != 0u; rest &= rest - 1u) {
                const int o = __builtin_ctz(rest);
                const int32_t row[2] = {static_cast<int32_t>(entry(o, 0)), static_cast<int32_t>(entry(o, 1))};
                if (kp < ksteps) {
                    load_raw(row, kp, raw[0]);
                    load_b(0, o, kp, bq[0]);
                }
                int ks = kp;
                for (; ks + KS < ksteps; ks += 2 * KS) {
                    load_raw(row, ks + KS, raw[1]);
                    load_b(0, o, ks + KS, bq[1]);
                    split_raw(raw[0], aq[0]);
                    products(aq[0], bq[0]);
                    if (ks + 2 * KS < ksteps) {
                        load_raw(row, ks + 2 * KS, raw[0]);
                        load_b(0, o, ks + 2 * KS, bq[0]);
                    }
                    split_raw(raw[1], aq[1]);
                    products(aq[1], bq[1]);
                }
                if (ks < ksteps) {
                    split_raw(raw[0], aq[0]);
                    products(aq[0], bq[0]);
                }
            }
        }
        if (chunks > kF3Sum)
#pragma unroll
            for (int mb = 0; mb < 2; ++mb)
#pragma unroll
                for (int r = 0; r < 16; ++r) hi[mb][r] += total[mb][r];
        float zero = 0.0f;  // (NaN once a sum is no finite number)
#pragma unroll
        for (int mb = 0; mb < 2; ++mb)
#pragma unroll
            for (int r = 0; r < 16; ++r) {
                const float v = hi[mb][r] + lo[mb][r];
                zero = __builtin_fmaf(v, 0.0f, zero);
                hi[mb][r] = v * kF3Unscale;
            }
        if (none || zero != 0.0f) *flag = 1u;
        __syncthreads();
    }
    if constexpr (FOLD) {
        // 32 columns of the slot's row of each parent, through this wave's 8 KiB
        // of LDS: 16-byte stores of 4 columns
        // (a sum that overflowed: the whole tile is left to the FP32 kernel behind)
        if (*flag != 0u && tid == 0)
            *const_cast<uint32_t *>(reinterpret_cast<const uint32_t *>(static_cast<const char *>(a.plan) +
                                                                       static_cast<int64_t>(tile) * kGatherPlanRecord128)) = kFoldGeneral;
        float *stg = reinterpret_cast<float *>(smem) + wave * 64 * 33;
#pragma unroll
        for (int mb = 0; mb < 2; ++mb)
#pragma unroll
            for (int r = 0; r < 16; ++r)
                stg[(mb * 32 + 4 * half + 8 * (r >> 2) + (r & 3)) * 33 + (lane & 31)] = hi[mb][r];
        const int c4 = (lane & 7) * 4, col = nb0 * 32 + c4;
        float bias[4] = {};
        if (a.bias)
#pragma unroll
            for (int k = 0; k < 4; ++k) bias[k] = a.bias[col + k];
#pragma unroll
        for (int i = 0; i < 8; ++i) {
            const int row = i * 8 + (lane >> 3);
            const int64_t p = m0 + rg * 64 + row;
            float v[4];
#pragma unroll
            for (int k = 0; k < 4; ++k) {
                v[k] = stg[row * 33 + c4 + k] + bias[k];
                if (a.silu) v[k] = silu(v[k]);
            }
            if (p < n_rows)
                *reinterpret_cast<float4 *>(static_cast<float *>(a.y) + (p * 8 + wave) * a.cout + col) =
                    make_float4(v[0], v[1], v[2], v[3]);
        }
        return;
    }
    if (__builtin_amdgcn_readfirstlane(*flag) != 0u) {
        // FP32 matrix instructions, rows from memory (k-steps of 8 channels,
        // every KS-th one this wave's); every fourth offset in a sum of its own, so
        // that the sums are no longer than the FP32 kernels'
        f32x16 sum[4][2];
#pragma unroll
        for (int j = 0; j < 4; ++j)
#pragma unroll
            for (int mb = 0; mb < 2; ++mb) sum[j][mb] = f32x16{};
        const uint4 *w = static_cast<const uint4 *>(a.w);
        for (uint32_t rest = mask; rest != 0u;)
            static_for<0, 4>([&](auto jc) __attribute__((always_inline)) {
                constexpr int j = decltype(jc)::value;
                if (rest == 0u) return;
                const int o = __builtin_ctz(rest);
                rest &= rest - 1u;
                int32_t row[2];
#pragma unroll
                for (int mb = 0; mb < 2; ++mb) {
                    const uint32_t v = table[o * ROWS + rg * 64 + mb * 32 + (lane & 31)];
                    const int sl = static_cast<int>(v >> 7);
                    row[mb] = mode != 0u ? static_cast<int32_t>(v)
                                         : sl < distinct ? static_cast<int32_t>(slot_row[min(sl, kH8Single - 1)]) : -1;
                }
                for (int s = kp; s < a.cin / 8; s += KS) {
                    const uint4 b = w[(static_cast<int64_t>(o * (a.cin / 8) + s) * nbtot + nb0 + cb) * 64 + lane];
#pragma unroll
                    for (int mb = 0; mb < 2; ++mb) {
                        const uint4 v = gather_plain<float>(a.x, static_cast<int32_t>(a.x_bytes), row[mb], a.cin, s * 8 + half * 4);
                        sum[j][mb] = mfma_step<float>(v, b, sum[j][mb]);
                    }
                }
            });
#pragma unroll
        for (int mb = 0; mb < 2; ++mb)
#pragma unroll
            for (int r = 0; r < 16; ++r) hi[mb][r] = (sum[0][mb][r] + sum[1][mb][r]) + (sum[2][mb][r] + sum[3][mb][r]);
    }
    __syncthreads();  // the planes become the output tile

    // ---- the tile in LDS (16-byte group q of row r at q ^ 8 when r & 4, for
    // 128 columns), the k parts added in order, then the row finish
    float *stg = reinterpret_cast<float *>(smem);
    constexpr bool SWZ = CG == 4;
    auto at = [&](int mb, int r) __attribute__((always_inline)) {
        const int row = rg * 64 + mb * 32 + 4 * half + 8 * (r >> 2) + (r & 3);
        const int col = cb * 32 + (lane & 31);
        return stg + row * LD + (SWZ ? col ^ (((row >> 2) & 1) << 5) : col);
    };
#pragma unroll
    for (int p = 0; p < KS; ++p) {
        if (p) __syncthreads();
        if (kp == p)
#pragma unroll
            for (int mb = 0; mb < 2; ++mb)
#pragma unroll
                for (int r = 0; r < 16; ++r) *at(mb, r) = p ? *at(mb, r) + hi[mb][r] : hi[mb][r];
    }
    constexpr int TPR = 4 * CG;
    RowParams params;
    load_row_params(a, nb0 * 32 + (tid % TPR) * 8, params);
    load_row_mod(a, nb0 * 32 + (tid % TPR) * 8, params);
    uint4 res[RowMap<TPR, ROWS, NTH>::PASSES][2];
    load_residual<TPR, ROWS, NTH>(a, m0, nb0, tile_rows, tid, res);
    __syncthreads();
    finish_rows<TPR, ROWS, LD, NTH, SWZ>(a, stg, stg, m0, nb0, tile_rows, tid, res, params);
}

// Folded FP32 weights: the sums of the offsets that reach one parent, formed in
// double precision, as three BF16 terms: [slot][group][k-step of 16][column
// block][term][lane][8], from the layer's packed FP32 ones.
__global__ void __launch_bounds__(256) f3_fold_weights_kernel(const float *w, uint4 *out, int ksteps, int nbtot, uint32_t *bad) {
    const int64_t total = static_cast<int64_t>(64) * ksteps * nbtot * 64;
    for (int64_t i = blockIdx.x * 256ll + threadIdx.x; i < total; i += gridDim.x * 256ll) {
        const int lane = static_cast<int>(i & 63);
        int64_t r = i >> 6;  // ((slot * 8 + group) * ksteps + k) * nbtot + column block
        const int64_t f = r;
        const int cb = static_cast<int>(r % nbtot);
        r /= nbtot;
        const int k = static_cast<int>(r % ksteps);
        const int sm = static_cast<int>(r / ksteps), s = sm >> 3, m = sm & 7;
        double sum[8] = {};
        for (int o = 0; o < kMaxKvol; ++o) {
            const int dx = o / 9 - 1, dy = o / 3 % 3 - 1, dz = o % 3 - 1;
            const int g = int((((s >> 2) & 1) + dx) >> 1 == 0) << 2 | int((((s >> 1) & 1) + dy) >> 1 == 0) << 1 |
                          int(((s & 1) + dz) >> 1 == 0);
            if (g != m) continue;
            // k-step 2k + lane / 32 of 8 channels, lanes l and l + 32 of the column
            const float *src = w + (((static_cast<int64_t>(o) * 2 * ksteps + 2 * k + (lane >> 5)) * nbtot + cb) * 64 + (lane & 31)) * 4;
#pragma unroll
            for (int e = 0; e < 4; ++e) {
                sum[e] += static_cast<double>(src[e]);
                sum[4 + e] += static_cast<double>(src[32 * 4 + e]);
            }
        }
        uint32_t t[4][3];
        bool none = false;
#pragma unroll
        for (int e = 0; e < 4; ++e) {
            double u = kF3Scale * sum[2 * e], v = kF3Scale * sum[2 * e + 1];
#pragma unroll
            for (int j = 0; j < 3; ++j) {
                t[e][j] = pack_bf16x2(static_cast<float>(u), static_cast<float>(v));
                u -= static_cast<double>(bf16_to_f32(static_cast<uint16_t>(t[e][j] & 0xffffu)));
                v -= static_cast<double>(bf16_to_f32(static_cast<uint16_t>(t[e][j] >> 16)));
            }
            none = none || (t[e][0] & 0x7f80u) == 0x7f80u || (t[e][0] & 0x7f800000u) == 0x7f800000u;
        }
        if (none) *bad = 1u;
#pragma unroll
        for (int j = 0; j < 3; ++j) out[(f * 3 + j) * 64 + lane] = make_uint4(t[0][j], t[1][j], t[2][j], t[3][j]);
    }
}

}  // namespace

int64_t f3_weight_bytes(int cin, int cout_pad) { return static_cast<int64_t>(kMaxKvol) * cin * cout_pad * 6; }

void launch_f3_weights(const void *w, void *out, int cin, int cout_pad, uint32_t *bad, hipStream_t stream) {
    const int64_t frags = static_cast<int64_t>(kMaxKvol) * (cin / 16) * (cout_pad / 32) * 64;
    hipLaunchKernelGGL(f3_weights_kernel, dim3(static_cast<unsigned>(std::min<int64_t>((frags + 255) / 256, 8192))),
                       dim3(256), 0, stream, static_cast<const uint4 *>(w), static_cast<uint4 *>(out), frags,
                       cout_pad / 32, bad);
}

int64_t f3_fold_weight_bytes(int cin, int cout_pad) { return static_cast<int64_t>(64) * cin * cout_pad * 6; }

void launch_f3_fold_weights(const void *w, void *out, int cin, int cout_pad, uint32_t *bad, hipStream_t stream) {
    const int64_t frags = static_cast<int64_t>(64) * (cin / 16) * (cout_pad / 32) * 64;
    hipLaunchKernelGGL(f3_fold_weights_kernel, dim3(static_cast<unsigned>(std::min<int64_t>((frags + 255) / 256, 8192))),
                       dim3(256), 0, stream, static_cast<const float *>(w), static_cast<uint4 *>(out), cin / 16,
                       cout_pad / 32, bad);
}

void launch_conv_f3_fold(const ConvArgs &a, hipStream_t stream) {
    const unsigned tiles = static_cast<unsigned>((a.n_out / 8 + 127) / 128);
    const KernelFn fn = conv_f3_kernel<1, 1, true>;
    hipLaunchKernelGGL(fn, dim3(2 * tiles, static_cast<unsigned>(a.cout_pad / 32)), dim3(kHalo8Threads), 0, stream, a);
}

KernelFn pick_f3(int cg) {
    return cg == 4 ? conv_f3_kernel<4, 1> : cg == 2 ? conv_f3_kernel<2, 2> : cg == 1 ? conv_f3_kernel<1, 4> : nullptr;
}

}  // namespace s3dx
