// Folded 3x3x3 convs over repeated parent rows (the mesh decoder's first conv
// of an upsample block: repeat_children, then the 27-offset convolution,
// mesh_decoder_graph.cpp:32-38, 81-103).
//
// A child's 27 neighbours lie in only eight parents: along an axis, the child
// at bit b reads offset -1, 0, +1 from the parent at floor((b + offset) / 2),
// so two of the three offsets read the same parent row.  All children of a
// parent hold the same feature row, so
//     sum over 27 offsets of W_o x[parent(child + o)]
//   = sum over 8 parents of (sum of the W_o that reach it) x[parent],
// with one set of eight folded matrices per child slot.  A matrix that one
// offset alone reaches is that offset's; where two reach it both are
// multiplied as they are (two products either way); sums of four and eight are
// held as three BF16 terms, 2^-27 of the sum, below the rounding of the FP32
// accumulation that every kernel here has: 19 matrix products per child in
// place of 27.  (Two terms, and 15 products, would lose what lies 2^-18 below
// a sum.)
//
// Output rows 8p .. 8p + 7 of one parent are one row of 8 * cout columns, so
// the product is a conv over the PARENTS' map whose column groups (one per
// slot) each read 8 of the 27 parent offsets: a parent tile is staged once for
// all eight slots' 64 * 27 child entries.
//
// Three steps, all of each run (nothing is kept by the map's address):
//   fold_plan_kernel   per 128 parents: the parent map read out of the child
//                      map, its gather-plan record, and a check that every
//                      one of the 8 * 27 child entries reaches the parent that
//                      the folding assumes.  Tiles that fail it (a map that no
//                      subdivide made), that name more rows than the halo
//                      holds (1,088), or any when a row holds an infinity or
//                      NaN, are marked for the general kernel.
//   conv_fold_kernel   the tiles that pass.
//   the general halo kernel, over the marked tiles (conv_halo.hip).
#include "halo_tile.hpp"

namespace s3dx {
namespace {

// Parent offset group m (3 bits, x y z) of a child at slot s (3 bits): an axis
// bit of m set: the child's own parent (two offsets), clear: the neighbour
// on the child's side (one offset).
constexpr int kFoldSlots = 8;
constexpr int kFoldGroups = 8;
// Weight products of a group, per k-step: 1, 2, 3 or 3 for 1, 2, 4 or 8 offsets.
__host__ __device__ constexpr int fold_terms(int m) {
    const int axes = (m & 1) + ((m >> 1) & 1) + (m >> 2);
    return axes < 3 ? axes + 1 : 3;
}
// Weight steps of one (slot, 64-channel chunk): by group, k-step (four), term.
__host__ __device__ constexpr int fold_step(int m, int k, int term) {
    int at = 0;
    for (int g = 0; g < m; ++g) at += 4 * fold_terms(g);
    return at + k * fold_terms(m) + term;
}
constexpr int kFoldSteps = fold_step(kFoldGroups - 1, 3, 2) + 1;  // 76
static_assert(kFoldSteps == 76, "1 + 3 * 2 + 4 * 3 products a k-step");
// The group that step t belongs to.
constexpr int fold_group(int t) {
    int m = 0;
    while (t >= fold_step(m + 1, 0, 0)) ++m;
    return m;
}

// ---------------------------------------------------------------------------
// Folded weights from the layer's packed ones ([offset][k-step][column
// block][lane][8]): [chunk][slot][step][column block][lane][8], the order
// conv_fold_kernel reads them in.  One thread per (slot, group, k-step, block,
// lane); a weight or sum that is no finite number raises *bad.
// ---------------------------------------------------------------------------
__global__ void __launch_bounds__(256) fold_weights_kernel(const uint4 *w, uint4 *out, int ksteps, int nbtot,
                                                           uint32_t *bad_out) {
    // thread: (chunk, slot, group m, k, block, lane)
    const int64_t total = static_cast<int64_t>(nbtot) * ksteps * kFoldSlots * kFoldGroups * 64;
    for (int64_t i = blockIdx.x * 256ll + threadIdx.x; i < total; i += gridDim.x * 256ll) {
        const int lane = static_cast<int>(i & 63);
        int64_t r = i >> 6;
        const int nb = static_cast<int>(r % nbtot);
        r /= nbtot;
        const int k = static_cast<int>(r & 3), m = static_cast<int>((r >> 2) & 7), s = static_cast<int>((r >> 5) & 7);
        const int c = static_cast<int>(r >> 8);
        const int terms = fold_terms(m);
        uint4 *dst = out + (static_cast<int64_t>(c) * kFoldSlots + s) * kFoldSteps * nbtot * 64;
        double sum[8] = {};  // (exact: eight values of eight bits, unless 42 binary places apart)
        bool bad = false;
        int seen = 0;
        for (int dx = -1; dx <= 1; ++dx)
            for (int dy = -1; dy <= 1; ++dy)
                for (int dz = -1; dz <= 1; ++dz) {
                    // the offset reaches group m: its own-parent axes are m's
                    const bool ox = (((s >> 2) & 1) + dx) >> 1 == 0, oy = (((s >> 1) & 1) + dy) >> 1 == 0,
                               oz = ((s & 1) + dz) >> 1 == 0;
                    if ((ox << 2 | oy << 1 | int(oz)) != m) continue;
                    const int o = (dx + 1) * 9 + (dy + 1) * 3 + dz + 1;
                    const uint4 v = w[((static_cast<int64_t>(o) * ksteps + c * 4 + k) * nbtot + nb) * 64 + lane];
                    const uint32_t q[4] = {v.x, v.y, v.z, v.w};
#pragma unroll
                    for (int e = 0; e < 4; ++e) {
                        bad = bad || (q[e] & 0x7f80u) == 0x7f80u || (q[e] & 0x7f800000u) == 0x7f800000u;
                        sum[2 * e] += static_cast<double>(bf16_to_f32(static_cast<uint16_t>(q[e] & 0xffffu)));
                        sum[2 * e + 1] += static_cast<double>(bf16_to_f32(static_cast<uint16_t>(q[e] >> 16)));
                    }
                    if (terms < 3) dst[(fold_step(m, k, seen++) * nbtot + nb) * 64 + lane] = v;
                }
        if (terms == 3) {
            uint32_t t[4][3];
#pragma unroll
            for (int e = 0; e < 4; ++e) {
                double u = sum[2 * e], v = sum[2 * e + 1];
#pragma unroll
                for (int j = 0; j < 3; ++j) {
                    t[e][j] = pack_bf16x2(static_cast<float>(u), static_cast<float>(v));
                    u -= static_cast<double>(bf16_to_f32(static_cast<uint16_t>(t[e][j] & 0xffffu)));
                    v -= static_cast<double>(bf16_to_f32(static_cast<uint16_t>(t[e][j] >> 16)));
                }
                bad = bad || (t[e][0] & 0x7f80u) == 0x7f80u || (t[e][0] & 0x7f800000u) == 0x7f800000u;
            }
#pragma unroll
            for (int j = 0; j < 3; ++j)  // the smallest first
                dst[(fold_step(m, k, 2 - j) * nbtot + nb) * 64 + lane] = make_uint4(t[0][j], t[1][j], t[2][j], t[3][j]);
        }
        if (bad) *bad_out = 1u;
    }
}

// ---------------------------------------------------------------------------
// fold_plan_kernel: one workgroup per 128 parents (1,024 children).
// ---------------------------------------------------------------------------
// The tile's parent entries, collected in LDS by the kernel below.
struct FoldSlice {
    const int32_t *parents;
    __device__ __forceinline__ int4 operator()(int64_t, int u, int) const {
        return *reinterpret_cast<const int4 *>(parents + 4 * u);
    }
};

__global__ void __launch_bounds__(kPlanBuild128Threads) fold_plan_kernel(const int32_t *kmap, int64_t n_parents,
                                                                         char *plan, const uint32_t *state) {
    // A parent's 8 * 27 child entries are 54 16-byte pieces; 864 of the threads
    // take the pieces of 16 parents a pass, each thread the same piece of
    // every parent, so that what its four entries are (the parent offset they
    // reach, whether they are the ones kept) is worked out once.  (Worked
    // out per entry, the pass over 195 MB of map took 127 us.)
    constexpr int ROWS = 128, NTH = kPlanBuild128Threads;
    constexpr int PIECES = kFoldSlots * kMaxKvol / 4;  // 54
    constexpr int PASS = 16, Q = ROWS / PASS;          // parents a pass, passes
    static_assert(PASS * PIECES <= NTH, "one piece a thread");
    __shared__ __align__(16) int32_t parents[ROWS * kMaxKvol];
    __shared__ uint32_t wrong;
    const int tid = threadIdx.x;
    const int tile = xcd_tile(blockIdx.x, gridDim.x);
    const int64_t m0 = static_cast<int64_t>(tile) * ROWS;
    const int64_t n_children = 8 * n_parents;
    const int sub = tid / PIECES, pc = tid - sub * PIECES;
    const bool active = sub < PASS;
    // 16-byte buffer loads that end at the map's last entry (zeros past it,
    // marked missing below); the map is under 2 GiB
    const auto rsrc = __builtin_amdgcn_make_buffer_rsrc(const_cast<int32_t *>(kmap), static_cast<short>(0),
                                                        static_cast<int32_t>(n_children * kMaxKvol * 4), 0x00020000);
    u32x4 v[Q];
#pragma unroll
    for (int q = 0; q < Q; ++q)
        v[q] = __builtin_amdgcn_raw_buffer_load_b128(
            rsrc, static_cast<int32_t>(((m0 + q * PASS + min(sub, PASS - 1)) * PIECES + pc) * 16), 0, 0);
    // entry k of the piece: slot s, offset o; it reaches parent offset d[k];
    // kept is the entry of the child on d's side (bit 1 for +1, else 0) at
    // the same child offset
    int d[4];
    bool kept[4];
#pragma unroll
    for (int k = 0; k < 4; ++k) {
        const int so = 4 * pc + k, s = so / kMaxKvol, o = so - s * kMaxKvol;
        const int px = (((s >> 2) & 1) + o / 9 - 1) >> 1, py = (((s >> 1) & 1) + o / 3 % 3 - 1) >> 1,
                  pz = ((s & 1) + o % 3 - 1) >> 1;
        d[k] = (px + 1) * 9 + (py + 1) * 3 + pz + 1;
        kept[k] = o == d[k] && s == ((px == 1) << 2 | (py == 1) << 1 | int(pz == 1));
    }
    if (tid == 0) wrong = state[kFoldBadRows];
    int32_t pj[Q][4];
#pragma unroll
    for (int q = 0; q < Q; ++q) {
        const bool in = m0 + q * PASS + sub < n_parents;
        const int32_t jv[4] = {static_cast<int32_t>(v[q].x), static_cast<int32_t>(v[q].y),
                               static_cast<int32_t>(v[q].z), static_cast<int32_t>(v[q].w)};
#pragma unroll
        for (int k = 0; k < 4; ++k) {
            pj[q][k] = in && jv[k] >= 0 && jv[k] < n_children ? jv[k] >> 3 : -1;
            if (active && kept[k]) parents[(q * PASS + sub) * kMaxKvol + d[k]] = pj[q][k];
        }
    }
    __syncthreads();
    bool ok = true;
#pragma unroll
    for (int q = 0; q < Q; ++q)
#pragma unroll
        for (int k = 0; k < 4; ++k)
            ok = ok && (!active || parents[(q * PASS + sub) * kMaxKvol + d[k]] == pj[q][k]);
    if (!ok) wrong = 1u;
    const TileDedupe dd = plan_tile<4, NTH>(FoldSlice{parents}, n_parents, n_parents, 0, plan);
    // (plan_tile's barriers order the writes of `wrong` before this read, and
    // thread 0 wrote the record's header)
    if (tid == 0 && (wrong != 0u || dd.global_a))
        *reinterpret_cast<uint32_t *>(plan + static_cast<int64_t>(tile) * kGatherPlanRecord128) = kFoldGeneral;
}

// ---------------------------------------------------------------------------
// conv_fold_kernel: 128 parents x 8 slots x (32 * NBW) columns per workgroup
// of 8 waves; wave s owns slot s (4 x NBW accumulator blocks, the whole sum:
// nothing to reduce between waves).
//
// The weights are the matrix instruction's first operand, so a lane holds
// one parent's row and its registers run over output channels: rows leave
// with 16-byte stores straight from the accumulators.
//
// LDS holds the parent record and two 64-channel chunks of the tile's
// distinct rows (the next chunk's copy is spread over the current one's
// steps).  Per (group, k-step) the four A fragments are read once for all its
// weight products; weight fragments come straight from memory, RB steps ahead.
//
// What bounds it: the matrix units' sustained rate.  768 -> 192 on 28,265
// parents is 1.27 TFLOP of products in 876-929 us with the row pass and the
// plan (1.4 PFLOP/s; a large BF16 matrix product reaches 1.26 on this card), 192
// -> 96 on 226,120 parents the same in 1,005, and moving the copies, the order
// of the products or the waves' priorities changes neither.  The 27-offset
// kernel takes 1,499-1,538 and 1,718 us.
// ---------------------------------------------------------------------------
template <int NBW>
__global__ void __launch_bounds__(kHalo8Threads, 1) conv_fold_kernel(ConvArgs a) {
    constexpr int ROWS = 128;
    constexpr int RB = NBW == 3 ? 2 : 4;  // weight sets in flight
    __shared__ __align__(16) char smem[kH8Bytes];
    char *halo = smem;
    char *rec = smem + kH8Dump + 1024;
    const uint32_t *table = reinterpret_cast<const uint32_t *>(rec + kPlan128Table);
    const uint32_t *slot_row = reinterpret_cast<const uint32_t *>(rec + kPlan128Slots);
    const int tid = threadIdx.x;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    // 16 * lane, from which every lane-dependent address is formed where it
    // is used: beside 192 accumulators there is no register to hold them in
    const int l16 = (tid & 63) * 16;
    const int tile = xcd_tile(blockIdx.x, gridDim.x);
    const int64_t p0 = static_cast<int64_t>(tile) * ROWS;
    const int64_t parents = a.n_out / kFoldSlots;
    const int chunks = a.cin / kHChunk;

    // ---- the record into LDS
    {
        const int64_t plan_bytes = (parents + ROWS - 1) / ROWS * kGatherPlanRecord128;
        const auto p_rsrc = __builtin_amdgcn_make_buffer_rsrc(const_cast<void *>(a.plan), static_cast<short>(0),
                                                              static_cast<int32_t>(plan_bytes), 0x00020000);
        constexpr int PIECES = kGatherPlanRecord128 / 1024;
#pragma unroll
        for (int k = 0; k < (PIECES + 7) / 8; ++k) {
            const int i = wave + 8 * k;
            if (i < PIECES)
                __builtin_amdgcn_raw_ptr_buffer_load_lds(
                    p_rsrc, (__attribute__((address_space(3))) void *)(rec + i * 1024), 16, l16,
                    tile * kGatherPlanRecord128 + i * 1024, 0, 0);
        }
        __builtin_amdgcn_s_waitcnt(0x0F70);  // vmcnt(0)
        __syncthreads();
    }
    const uint32_t *hdr = reinterpret_cast<const uint32_t *>(rec);
    if (__builtin_amdgcn_readfirstlane(hdr[0]) != 0u) return;  // the general kernel's
    const int distinct = static_cast<int>(__builtin_amdgcn_readfirstlane(hdr[1]));
    // Tiles of more rows than two buffers hold (no thin shell's: of a solid bar of
    // 24 x 24 x 60 most) take one, whose copy nothing hides: about 5% of a chunk.
    const bool single = distinct > kH8Double;
    if (tid < 2 * (kHRowBytes / 16)) {  // each buffer's zero row, or the one's
        const int zero = single ? kH8Single : (tid / (kHRowBytes / 16)) * kH8BufRows + kH8Double;
        reinterpret_cast<uint4 *>(halo + zero * kHRowBytes)[tid % (kHRowBytes / 16)] = make_uint4(0, 0, 0, 0);
    }

    const auto x_rsrc = __builtin_amdgcn_make_buffer_rsrc(const_cast<void *>(a.x), static_cast<short>(0),
                                                          static_cast<int32_t>(a.x_bytes), 0x00020000);
    const int groups = max((distinct + 7) >> 3, 1);
    constexpr int kPieces = (kH8Double + 1 + 63) / 64;  // 9 pieces of 8 rows a wave
    // piece j of chunk c into buffer dst: row group min(wave + 8j, last) (a
    // clamped piece copies its group again: the same bytes to the same place)
    auto piece = [&](int j, int c, char *dst, const uint32_t *rows) __attribute__((always_inline)) {
        // (opaque: none of the nine pieces' addresses is held across chunks)
        const int g = min(opaque_scalar<true>(wave) + 8 * j, opaque_scalar<true>(groups) - 1);
        int ln = l16;
        asm volatile("" : "+v"(ln));
        ln >>= 4;
        const int sl = g * 8 + (ln >> 3);
        const int p = (ln & 7) ^ halo_swizzle(sl);
        // (24 bits: rows * 128 bytes at least are below 2 GiB; the top bit
        // puts a slot past the last row out of range: zeros)
        const uint32_t off = (__umul24(rows[min(sl, kH8Single - 1)], 2u * static_cast<uint32_t>(a.cin)) + p * 16u) |
                             (sl < distinct ? 0u : 0x80000000u);
        __builtin_amdgcn_raw_ptr_buffer_load_lds(x_rsrc, (__attribute__((address_space(3))) void *)(dst + g * 1024), 16,
                                                 static_cast<int32_t>(off), c * kHRowBytes, 0, 0);
    };

    f32x16 acc[4][NBW];
#pragma unroll
    for (int mb = 0; mb < 4; ++mb)
#pragma unroll
        for (int nb = 0; nb < NBW; ++nb) acc[mb][nb] = f32x16{};

    // this wave's weights: one run of steps per chunk
    const int32_t step_bytes = a.cout_pad * 32;  // cout_pad / 32 blocks of 1 KiB
    const int32_t slot_bytes = kFoldSteps * step_bytes;
    const int32_t w_first = wave * slot_bytes + static_cast<int32_t>(blockIdx.y) * NBW * 1024;
    const auto w_rsrc = __builtin_amdgcn_make_buffer_rsrc(const_cast<void *>(a.w), static_cast<short>(0),
                                                          chunks * kFoldSlots * slot_bytes, 0x00020000);
    uint4 bf[RB][NBW];
    auto load_b = [&](int32_t sbase, int nb, uint4 (&b)[NBW]) __attribute__((always_inline)) {
        const u32x4 v = __builtin_amdgcn_raw_buffer_load_b128(w_rsrc, l16, sbase + nb * 1024, 0);
        b[nb] = make_uint4(v.x, v.y, v.z, v.w);
    };
    // parent offsets of the wave's groups, as table rows
    const int bx = (wave >> 2) & 1, by = (wave >> 1) & 1, bz = wave & 1;
    const int ox = bx ? 18 : 0, oy = by ? 6 : 0, oz = bz ? 2 : 0;

    constexpr int kPiecesSingle = (kH8Single + 63) / 64;
    if (single) {
#pragma nounroll
        for (int j = 0; j < kPiecesSingle; ++j) piece(j, 0, halo, slot_row);
    } else {
#pragma unroll
        for (int j = 0; j < kPieces; ++j) piece(j, 0, halo, slot_row);
    }
#pragma unroll
    for (int k = 0; k < RB; ++k) {
#pragma unroll
        for (int nb = 0; nb < NBW; ++nb) load_b(w_first + k * step_bytes, nb, bf[k]);
        sched_fence();
    }
    // Chunk c from `buf`, the next one's rows copied into `nxt` and its first
    // weights requested over the last steps.
    auto chunk = [&](int c, const char *__restrict__ buf, char *__restrict__ nxt, const uint32_t *__restrict__ tbl,
                     const uint32_t *__restrict__ rows) __attribute__((always_inline)) {
        const bool last = c + 1 == chunks, copy = !last && !single;
        int32_t wb = w_first + c * kFoldSlots * slot_bytes + RB * step_bytes;  // the next step to request
        // the steps past this chunk's are the next chunk's first (the last
        // chunk reads its own first ones again: unused)
        const int32_t wn = w_first + (last ? c : c + 1) * kFoldSlots * slot_bytes;
        uint32_t ix[4];
        uint4 af[4];
        auto load_ix = [&](auto mc) __attribute__((always_inline)) {
            constexpr int m = decltype(mc)::value;
            const int o = opaque_scalar<true>(((m & 4) ? 9 : ox) + ((m & 2) ? 3 : oy) + ((m & 1) ? 1 : oz));
            int l = l16;
            asm volatile("" : "+v"(l));
            const uint32_t *row = reinterpret_cast<const uint32_t *>(reinterpret_cast<const char *>(tbl) + ((l & 0x1f0) >> 2));
#pragma unroll
            for (int mb = 0; mb < 4; ++mb) ix[mb] = row[o * ROWS + mb * 32] ^ ((l >> 5) & 16);
        };
        auto load_a = [&](int mb, int k) __attribute__((always_inline)) {
            af[mb] = *reinterpret_cast<const uint4 *>(buf + (ix[mb] ^ (k << 5)));
        };
        load_ix(std::integral_constant<int, 0>{});
#pragma unroll
        for (int mb = 0; mb < 4; ++mb) load_a(mb, 0);
        sched_fence();
        static_for<0, kFoldSteps>([&](auto tc) __attribute__((always_inline)) {
            constexpr int t = decltype(tc)::value;
            // step t: group m, k-step k, weight term
            constexpr int m = fold_group(t), terms = fold_terms(m);
            constexpr int k = (t - fold_step(m, 0, 0)) / terms;
            constexpr bool last_term = t == fold_step(m, k, terms - 1);
            constexpr bool more = t + 1 < kFoldSteps;
            // the next group's rows, once this group's last fragments are read
            if constexpr (last_term && k == 3 && more) load_ix(std::integral_constant<int, m + 1 < 8 ? m + 1 : 0>{});
            if constexpr (t % 2 == 0 && t / 2 < kPieces)
                if (copy) piece(t / 2, c + 1, nxt, rows);
            // Row blocks 0 and 1 over all column blocks, then 2 and 3: an A
            // fragment is refilled half a step before its next use, a weight
            // fragment a step and a third (fenced: each takes the registers
            // just read).
            if constexpr (t + RB == kFoldSteps) wb = wn;
            static_for<0, 2 * NBW>([&](auto ic) __attribute__((always_inline)) {
                constexpr int i = decltype(ic)::value, h = 2 * (i / NBW), nb = i % NBW;
                acc[h][nb] = mfma_step<uint16_t>(bf[t % RB][nb], af[h], acc[h][nb]);
                sched_fence();
                if constexpr (nb == NBW - 1 && last_term && more) load_a(h, k == 3 ? 0 : k + 1);
                acc[h + 1][nb] = mfma_step<uint16_t>(bf[t % RB][nb], af[h + 1], acc[h + 1][nb]);
                sched_fence();
                if constexpr (h == 2) load_b(wb, nb, bf[t % RB]);
                sched_fence();
                if constexpr (nb == NBW - 1 && last_term && more) load_a(h + 1, k == 3 ? 0 : k + 1);
                sched_fence();
            });
            wb = opaque_scalar<true>(wb + step_bytes);  // (a running sum: no table of 76 steps)
        });
    };
    static_assert(kFoldSteps % RB == 0, "a chunk leaves every weight set at its place");
    static_assert(2 * kPieces < kFoldSteps - RB, "the pieces go out before the chunk's last weight loads");
    for (int c = 0; c < chunks; ++c) {
        // chunk c's pieces precede the RB weight sets in flight; after the
        // barrier no wave reads the buffer of chunk c - 1
        if (single && c > 0) {
            __syncthreads();
#pragma nounroll
            for (int j = 0; j < kPiecesSingle; ++j) piece(j, c, halo, slot_row);
            __builtin_amdgcn_s_waitcnt(vmcnt_imm(0));
        } else {
            __builtin_amdgcn_s_waitcnt(vmcnt_imm(RB * NBW));
        }
        __syncthreads();
        char *cur = single ? halo : halo + (c & 1) * (kH8BufRows * kHRowBytes);
        char *nxt = halo + ((c + 1) & 1) * (kH8BufRows * kHRowBytes);
        chunk(c, cur, nxt, table, slot_row);
    }

    // ---- rows out: lane l holds parent mb * 32 + l % 32; register 4q + i of a
    // block is channel 8q + 4 * (l / 32) + i.  Two quads swapped between the
    // lane halves give each lane eight channels: 8 * (2h + half) .. + 7.
    const int col0 = blockIdx.y * NBW * 32;
    const int lane = l16 >> 4, half = lane >> 5;
#pragma unroll
    for (int nb = 0; nb < NBW; ++nb) {
        float4 bias[4];
#pragma unroll
        for (int q = 0; q < 4; ++q)
            bias[q] = a.bias ? *reinterpret_cast<const float4 *>(a.bias + col0 + nb * 32 + 8 * q + 4 * half)
                             : make_float4(0, 0, 0, 0);
#pragma unroll
        for (int mb = 0; mb < 4; ++mb) {
            const int64_t p = p0 + mb * 32 + (lane & 31);
            uint16_t *row = static_cast<uint16_t *>(a.y) + (p * kFoldSlots + wave) * a.cout + col0 + nb * 32;
            uint32_t lo[4], hi[4];
#pragma unroll
            for (int q = 0; q < 4; ++q) {
                float v[4] = {acc[mb][nb][4 * q] + bias[q].x, acc[mb][nb][4 * q + 1] + bias[q].y,
                              acc[mb][nb][4 * q + 2] + bias[q].z, acc[mb][nb][4 * q + 3] + bias[q].w};
                if (a.silu)
#pragma unroll
                    for (int i = 0; i < 4; ++i) v[i] = silu(v[i]);
                lo[q] = pack_bf16x2(v[0], v[1]);
                hi[q] = pack_bf16x2(v[2], v[3]);
            }
#pragma unroll
            for (int h = 0; h < 2; ++h) {
                const auto s0 = __builtin_amdgcn_permlane32_swap(lo[2 * h], lo[2 * h + 1], false, false);
                const auto s1 = __builtin_amdgcn_permlane32_swap(hi[2 * h], hi[2 * h + 1], false, false);
                if (p < parents)
                    *reinterpret_cast<uint4 *>(row + 8 * (2 * h + half)) = make_uint4(s0[0], s1[0], s0[1], s1[1]);
            }
        }
    }
}

}  // namespace

int64_t fold_weight_bytes(int cin, int blocks) {
    return static_cast<int64_t>(cin / kHChunk) * blocks * kFoldSlots * kFoldSteps * 1024;
}

// Column blocks per workgroup of the folded conv, or 0 where the general
// kernel suits the size.  Both sides by what they take per 64-channel chunk, in
// microseconds: a pass of folded workgroups (one per CU) 11.4 per column block
// and 18 for the plan and a tile's ends; the general kernel's 64-row tiles
// 5.2 (96 columns) with one per CU, 9.8 with two, and 11.  Measured, folded against
// general: 768 -> 192 on 2,000 parents 157 / 126 us, 3,000 152-168 / 176-187,
// 28,265 876-929 / 1,499-1,538; 192 -> 96 on 4,800 parents 56 / 55, 6,000 58 /
// 60, 7,200 60 / 71, 226,120 1,005 / 1,718.  Column blocks: fewer per workgroup where that
// fills the CUs; a pass costs about the same per block (768 -> 192 on 16,000
// parents: three blocks, one pass, 496; two blocks, two passes, 558; one
// block, three passes, 526.  On 20,000: 813, 625 and 669).
int fold_blocks(int cin, int blocks, int general_nb, int64_t n_parents, int64_t cus) {
    const int chunks = cin / kHChunk;
    const int64_t wgs = (n_parents + 7) / 8 * (blocks / general_nb);
    double least = chunks * general_nb / 3.0 *
                       (wgs <= cus ? 5.2 : 9.8 * static_cast<double>(wgs) / (2.0 * static_cast<double>(cus))) + 11.0;
    int best = 0;
    const int64_t tiles = (n_parents + 127) / 128;
    for (int nbw : {3, 2, 1}) {
        if (blocks % nbw != 0) continue;
        const int64_t passes = (tiles * (blocks / nbw) + cus - 1) / cus;
        const double t = 18.0 + 11.4 * static_cast<double>(passes * nbw * chunks);
        if (t < least) {
            best = nbw;
            least = t;
        }
    }
    return best;
}

void launch_fold_weights(const void *w, void *out, int cin, int blocks, uint32_t *bad, hipStream_t stream) {
    const int64_t total = static_cast<int64_t>(blocks) * (cin / 16) * kFoldSlots * kFoldGroups * 64;
    hipLaunchKernelGGL(fold_weights_kernel, dim3(static_cast<unsigned>(std::min<int64_t>((total + 255) / 256, 4096))),
                       dim3(256), 0, stream, static_cast<const uint4 *>(w), static_cast<uint4 *>(out), cin / 16, blocks,
                       bad);
}

void launch_fold_plan(const int32_t *kmap, int64_t n_parents, void *plan, const uint32_t *state, hipStream_t stream) {
    hipLaunchKernelGGL(fold_plan_kernel, dim3(static_cast<unsigned>((n_parents + 127) / 128)),
                       dim3(kPlanBuild128Threads), 0, stream, kmap, n_parents, static_cast<char *>(plan), state);
}

void launch_conv_fold(const ConvArgs &a, int nbw, hipStream_t stream) {
    const dim3 grid(static_cast<unsigned>((a.n_out / kFoldSlots + 127) / 128),
                    static_cast<unsigned>(a.cout_pad / 32 / nbw));
    if (nbw == 3) hipLaunchKernelGGL(conv_fold_kernel<3>, grid, dim3(kHalo8Threads), 0, stream, a);
    else if (nbw == 2) hipLaunchKernelGGL(conv_fold_kernel<2>, grid, dim3(kHalo8Threads), 0, stream, a);
    else hipLaunchKernelGGL(conv_fold_kernel<1>, grid, dim3(kHalo8Threads), 0, stream, a);
}

}  // namespace s3dx
