// BF16 3x3x3 convs over many rows with few channels (the mesh decoder's last
// conv, 96 -> 96 on up to 1.8M children): 512 rows x 96 columns per workgroup,
// each wave 128 rows x 96 columns with the whole sum.
//
// Why: with 64- or 128-row tiles, the k-steps go to different waves, whose
// partial tiles cost LDS traffic and time per tile that a layer of Cin 96 does
// not repay, and every weight fragment feeds two row blocks.  Here
// nothing is reduced between waves, a weight fragment feeds four row blocks
// (32 B a cycle for a CU at the full matrix rate) and an A fragment three column
// blocks (43 B a cycle of LDS).
//
// One wave per SIMD (192 accumulators of 512 registers): the rows of the next
// 32-channel chunk are read into registers while the current one is
// multiplied, the weights six steps ahead, the A fragments one.
//
// What bounds it: one wave per SIMD hides nothing between a chunk's ends and a
// tile's, so the matrix units are busy 53% of the time.  96 -> 96 on 1.81M rows:
// 845-950 us and the plan 100, against 1,372-1,434 for 64-row split-K tiles.
// (Persistent workgroups that read the next tile's record and rows ahead took
// 825-912; more weights in flight and other orders of the row reads, the same.
// 192 -> 192 on 226,120 rows: 488 with the plan against 497 for the 64-row halo
// kernel, and 220 against 170 on 72,000, so layers with a halo kernel keep it.)
//
//   rows_plan_kernel   per 512 rows: the distinct source rows of the tile's
//                      27 * 512 map entries and each entry's slot among them
//   conv_rows_kernel   the tiles with all 27 offsets (any 2x2x2 block of
//                      children has them) and at most 1,535 distinct rows
//   the 64-row split-K kernel, over the other tiles (conv_kernels.hpp)
#include "halo_tile.hpp"

namespace s3dx {
namespace {

constexpr int kRowsTile = 512;
constexpr int kRowsCap = 1536;                     // slots; the last is the zero row
constexpr int kRowsSlots = 16;                     // record: header, the slots' source rows,
constexpr int kRowsTable = 16 + kRowsCap * 4;      // 6,160: then the u16 table [27][wave][lane % 32][row block]
constexpr int kRowsTableBytes = kMaxKvol * kRowsTile * 2;  // 27,648
static_assert(kRowsTable % 16 == 0 && kRowsTable + kRowsTableBytes <= kRowsRecord, "the record fits");
static_assert(kRowsRecord % 1024 == 0, "whole KiB");

// Slot s's 64 bytes of a chunk; 16-byte piece p of it at p ^ ((s >> 1) & 3), so
// that the same piece of eight consecutive slots lies in eight bank groups.
// Table entries: the offset of piece 0 in 16-byte units.
__device__ __forceinline__ uint32_t rows_entry(uint32_t s) { return s * 4 + ((s >> 1) & 3); }

// One workgroup per tile; tiles from `most` on are left to the general kernel.
__global__ void __launch_bounds__(1024) rows_plan_kernel(const int32_t *kmap, int64_t n_out, int64_t n_src, int most, char *plan) {
    constexpr int NTH = 1024, WORDS = 4096;  // a bitmap over 131,072 rows
    constexpr int V4 = kRowsTile * kMaxKvol / 4, Q = (V4 + NTH - 1) / NTH;
    __shared__ __align__(16) uint16_t table[kRowsTile * kMaxKvol];
    __shared__ uint32_t bitmap[WORDS], prefix[WORDS];
    __shared__ uint32_t slot_row[kRowsCap];
    __shared__ int32_t misc[4];
    __shared__ uint32_t sums[NTH / 64];
    const int tid = threadIdx.x, lane = tid & 63;
    const int tile = xcd_tile(blockIdx.x, gridDim.x);
    if (tile >= most) {
        if (tid == 0) *reinterpret_cast<uint4 *>(plan + static_cast<int64_t>(tile) * kRowsRecord) = make_uint4(kFoldGeneral, 0u, 0u, 0u);
        return;
    }
    const int64_t m0 = static_cast<int64_t>(tile) * kRowsTile;
    const int count = static_cast<int>(min(static_cast<int64_t>(kRowsTile), n_out - m0)) * kMaxKvol;
    // 16-byte buffer loads that end at the map's last entry (zeros past it)
    const auto rsrc = __builtin_amdgcn_make_buffer_rsrc(const_cast<int32_t *>(kmap), static_cast<short>(0),
                                                        static_cast<int32_t>(n_out * kMaxKvol * 4), 0x00020000);
    int32_t sj[Q][4];
#pragma unroll
    for (int q = 0; q < Q; ++q) {
        const int u = tid + q * NTH;
        const u32x4 v = __builtin_amdgcn_raw_buffer_load_b128(
            rsrc, static_cast<int32_t>((m0 * kMaxKvol + 4 * min(u, V4 - 1)) * 4), 0, 0);
        const int32_t jv[4] = {static_cast<int32_t>(v.x), static_cast<int32_t>(v.y), static_cast<int32_t>(v.z),
                               static_cast<int32_t>(v.w)};
#pragma unroll
        for (int k = 0; k < 4; ++k)
            sj[q][k] = u < V4 && 4 * u + k < count && jv[k] >= 0 && jv[k] < n_src ? jv[k] : -1;
    }
    if (tid == 0) {
        misc[0] = INT32_MAX;
        misc[1] = INT32_MIN;
        misc[2] = 0;
    }
    for (int w = tid; w < WORDS; w += NTH) bitmap[w] = 0u;
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
    const int64_t span = rhi >= rlo ? static_cast<int64_t>(rhi) - rlo + 1 : 0;
    bool left = misc[2] != (1 << kMaxKvol) - 1 || span > static_cast<int64_t>(WORDS) * 32;
    uint32_t distinct = 0;
    if (!left) {
#pragma unroll
        for (int q = 0; q < Q; ++q)
#pragma unroll
            for (int k = 0; k < 4; ++k)
                if (sj[q][k] >= 0) {
                    // (a row is named about eleven times: most bits are found
                    // set, and a plain read of a word that a wave shares costs
                    // one access where its atomics would take turns: 162 -> 110
                    // us on 1.81M rows)
                    const uint32_t r = static_cast<uint32_t>(sj[q][k] - rlo), bit = 1u << (r & 31);
                    if ((__hip_atomic_load(&bitmap[r >> 5], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP) & bit) == 0u)
                        atomicOr(&bitmap[r >> 5], bit);
                }
        __syncthreads();
        constexpr int WPT = WORDS / NTH;
        uint32_t cnt[WPT], own = 0;
#pragma unroll
        for (int k = 0; k < WPT; ++k) {
            cnt[k] = static_cast<uint32_t>(__popc(bitmap[tid * WPT + k]));
            own += cnt[k];
        }
        uint32_t run = block_exclusive_scan<NTH / 64>(own, sums, &distinct);
#pragma unroll
        for (int k = 0; k < WPT; ++k) {
            prefix[tid * WPT + k] = run;
            run += cnt[k];
        }
        left = distinct >= static_cast<uint32_t>(kRowsCap);
        __syncthreads();
    }
    char *rec = plan + static_cast<int64_t>(tile) * kRowsRecord;
    if (left) {
        if (tid == 0) *reinterpret_cast<uint4 *>(rec) = make_uint4(kFoldGeneral, 0u, 0u, 0u);
        return;
    }
#pragma unroll
    for (int q = 0; q < Q; ++q)
#pragma unroll
        for (int k = 0; k < 4; ++k) {
            const int e = 4 * (tid + q * NTH) + k;
            if (e >= kRowsTile * kMaxKvol) continue;
            const int r = e / kMaxKvol, o = e - r * kMaxKvol;
            uint32_t slot = kRowsCap - 1;
            if (sj[q][k] >= 0) {
                const uint32_t d = static_cast<uint32_t>(sj[q][k] - rlo);
                slot = prefix[d >> 5] + static_cast<uint32_t>(__popc(bitmap[d >> 5] & ((1u << (d & 31)) - 1u)));
                slot_row[slot] = static_cast<uint32_t>(sj[q][k]);  // writers of one slot agree
            }
            table[((o * 4 + (r >> 7)) * 32 + (r & 31)) * 4 + ((r >> 5) & 3)] = static_cast<uint16_t>(rows_entry(slot));
        }
    __syncthreads();
    if (tid == 0) *reinterpret_cast<uint4 *>(rec) = make_uint4(0u, distinct, 0u, 0u);
    for (int i = tid; i < kRowsTableBytes / 16; i += NTH)
        reinterpret_cast<uint4 *>(rec + kRowsTable)[i] = reinterpret_cast<const uint4 *>(table)[i];
    for (int i = tid; i < static_cast<int>(distinct); i += NTH)
        reinterpret_cast<uint32_t *>(rec + kRowsSlots)[i] = slot_row[i];
}

__global__ void __launch_bounds__(256, 1) conv_rows_kernel(ConvArgs a) {
    constexpr int NB = 3, RB = 6;
    constexpr int kChunk = 32, kSteps = kMaxKvol * 2;  // (offset, k-step) of a chunk
    static_assert(kSteps % RB == 0, "a chunk leaves every weight set at its place");
    __shared__ __align__(16) char smem[kRowsCap * 64 + kRowsTableBytes];
    char *rows = smem;
    const char *table = smem + kRowsCap * 64;
    const int tid = threadIdx.x, lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int half = lane >> 5;
    const int tile = xcd_tile(blockIdx.x, gridDim.x);
    const int64_t m0 = static_cast<int64_t>(tile) * kRowsTile;
    const int nb0 = blockIdx.y * NB;
    const int nbtot = a.cout_pad / 32;
    const int chunks = a.cin / kChunk, ksteps = a.cin / 16;
    const char *rec = static_cast<const char *>(a.plan) + static_cast<int64_t>(tile) * kRowsRecord;
    const uint4 hdr = *reinterpret_cast<const uint4 *>(rec);
    if (__builtin_amdgcn_readfirstlane(hdr.x) != 0u) return;  // left to the general kernel
    const int distinct = static_cast<int>(__builtin_amdgcn_readfirstlane(hdr.y));

    const auto x_rsrc = __builtin_amdgcn_make_buffer_rsrc(const_cast<void *>(a.x), static_cast<short>(0),
                                                          static_cast<int32_t>(a.x_bytes), 0x00020000);
    const auto w_rsrc = __builtin_amdgcn_make_buffer_rsrc(
        const_cast<void *>(a.w), static_cast<short>(0),
        static_cast<int32_t>(static_cast<int64_t>(kMaxKvol) * a.cin * a.cout_pad * 2), 0x00020000);
    const auto r_rsrc = __builtin_amdgcn_make_buffer_rsrc(const_cast<char *>(rec), static_cast<short>(0), kRowsRecord,
                                                          0x00020000);
    // Piece i of a thread: 16-byte piece tid % 4 of slot 64 i + tid / 4 (four
    // lanes read a row's 64 bytes); past the tile's rows: zeros.
    constexpr int XP = kRowsCap / 64;  // 24
    uint32_t xoff[XP];
#pragma unroll
    for (int i = 0; i < XP; ++i)
        xoff[i] = __builtin_amdgcn_raw_buffer_load_b32(r_rsrc, kRowsSlots + (64 * i + (tid >> 2)) * 4, 0, 0);
    // the table, straight into LDS
#pragma unroll
    for (int k = 0; k < (kRowsTableBytes / 1024 + 3) / 4; ++k) {
        const int i = wave + 4 * k;
        if (i < kRowsTableBytes / 1024)
            __builtin_amdgcn_raw_ptr_buffer_load_lds(
                r_rsrc, (__attribute__((address_space(3))) void *)(smem + kRowsCap * 64 + i * 1024), 16, lane * 16,
                kRowsTable + i * 1024, 0, 0);
    }
    // (a full 32-bit product: at Cin 32, 64 bytes a row, x below 2 GiB holds
    // rows above 2^24)
#pragma unroll
    for (int i = 0; i < XP; ++i)
        xoff[i] = (xoff[i] * (2u * static_cast<uint32_t>(a.cin)) + (tid & 3) * 16u) |
                  (64 * i + (tid >> 2) < distinct ? 0u : 0x80000000u);
    u32x4 xq[XP];
    auto load_x = [&](int i, int c) __attribute__((always_inline)) {
        xq[i] = __builtin_amdgcn_raw_buffer_load_b128(x_rsrc, static_cast<int32_t>(xoff[i]), c * (kChunk * 2), 0);
    };
    uint4 bf[RB][NB];
    auto load_b = [&](int32_t sbase, int nb, uint4 (&b)[NB]) __attribute__((always_inline)) {
        const u32x4 v = __builtin_amdgcn_raw_buffer_load_b128(w_rsrc, lane * 16, sbase + nb * 1024, 0);
        b[nb] = make_uint4(v.x, v.y, v.z, v.w);
    };
    const int32_t w_step = nbtot * 1024, w_offset = ksteps * w_step;
#pragma unroll
    for (int i = 0; i < XP; ++i) load_x(i, 0);
    sched_fence();
#pragma unroll
    for (int t = 0; t < RB; ++t) {
#pragma unroll
        for (int nb = 0; nb < NB; ++nb) load_b(nb0 * 1024 + (t / 2) * w_offset + (t & 1) * w_step, nb, bf[t]);
        sched_fence();
    }
    f32x16 acc[4][NB];
#pragma unroll
    for (int mb = 0; mb < 4; ++mb)
#pragma unroll
        for (int nb = 0; nb < NB; ++nb) acc[mb][nb] = f32x16{};

    for (int c = 0; c < chunks; ++c) {
        if (c > 0) __syncthreads();  // every wave is done with the rows
#pragma unroll
        for (int i = 0; i < XP; ++i) {
            const int s = 64 * i + (tid >> 2);
            *reinterpret_cast<u32x4 *>(rows + s * 64 + (((tid & 3) ^ ((s >> 1) & 3)) << 4)) = xq[i];
        }
        __builtin_amdgcn_s_waitcnt(vmcnt_imm(RB * NB));  // chunk 0: the table (before the weights in flight)
        __syncthreads();
        const bool last = c + 1 == chunks;
        const int32_t wc = nb0 * 1024 + 2 * c * w_step;
        const int32_t wn = nb0 * 1024 + 2 * (last ? c : c + 1) * w_step;
        uint2 ix[2];
        uint4 af[2][4];
        // the four row blocks' entries at offset o: one 8-byte read (decoded
        // where they are used, a step on)
        auto load_ix = [&](int o, uint2 &x) __attribute__((always_inline)) {
            x = *reinterpret_cast<const uint2 *>(table + ((o * 4 + wave) * 32 + (lane & 31)) * 8);
        };
        auto load_a = [&](int mb, int k, const uint2 &x, uint4 (&f)[4]) __attribute__((always_inline)) {
            const uint32_t v = mb < 2 ? x.x : x.y;
            const uint32_t at = (((mb & 1) ? v >> 16 : v & 0xffffu) << 4) ^ static_cast<uint32_t>(half << 4 ^ k << 5);
            f[mb] = *reinterpret_cast<const uint4 *>(rows + at);
        };
        load_ix(0, ix[0]);
#pragma unroll
        for (int mb = 0; mb < 4; ++mb) load_a(mb, 0, ix[0], af[0]);
        load_ix(1, ix[1]);
        sched_fence();
        static_for<0, kSteps>([&](auto tc) __attribute__((always_inline)) {
            constexpr int t = decltype(tc)::value, o = t / 2, k = t % 2, S = t % RB;
            // (the row pieces of the next chunk, one a step)
            if constexpr (t < XP)
                if (!last) load_x(t, c + 1);
            static_for<0, 4 * NB>([&](auto ic) __attribute__((always_inline)) {
                constexpr int i = decltype(ic)::value, nb = i / 4, mb = i % 4;
                acc[mb][nb] = mfma_step<uint16_t>(bf[S][nb], af[k][mb], acc[mb][nb]);
                // the next step's fragments between the first products, the
                // weights RB steps on once a column block's are used
                if constexpr (i < 4 && t + 1 < kSteps) load_a(i, 1 - k, ix[(o + k) & 1], af[1 - k]);
                if constexpr (i == 6 && k == 1 && o + 2 < kMaxKvol) load_ix(o + 2, ix[o & 1]);
                if constexpr (mb == 3) {
                    sched_fence();
                    constexpr int u = t + RB;
                    load_b((u < kSteps ? wc + (u / 2) * w_offset : wn + (u - kSteps) / 2 * w_offset) + (u & 1) * w_step,
                           nb, bf[S]);
                    sched_fence();
                }
            });
        });
    }

    // ---- rows out: lane l holds row mb * 32 + l % 32 of the wave's 128, its
    // registers channels 8q + 4 * (l / 32) + i; two quads swapped between the
    // lane halves give each lane eight channels
    const int col0 = nb0 * 32;
    const int64_t res_rows = (a.n_out + (int64_t(1) << a.residual_shift) - 1) >> a.residual_shift;
#pragma unroll
    for (int nb = 0; nb < NB; ++nb) {
        float4 bias[4];
#pragma unroll
        for (int q = 0; q < 4; ++q)
            bias[q] = a.bias ? *reinterpret_cast<const float4 *>(a.bias + col0 + nb * 32 + 8 * q + 4 * half)
                             : make_float4(0, 0, 0, 0);
#pragma unroll
        for (int mb = 0; mb < 4; ++mb) {
            const int64_t row = m0 + wave * 128 + mb * 32 + (lane & 31);
            // residual: channels 8q + 4 half .. + 3 of the row
            uint2 res[4];
            if (a.residual) {
                const uint16_t *rp = static_cast<const uint16_t *>(a.residual) +
                                     min(row >> a.residual_shift, res_rows - 1) * a.cout + col0 + nb * 32 + 4 * half;
#pragma unroll
                for (int q = 0; q < 4; ++q) res[q] = *reinterpret_cast<const uint2 *>(rp + 8 * q);
            }
            uint32_t lo[4], hi[4];
#pragma unroll
            for (int q = 0; q < 4; ++q) {
                float v[4] = {acc[mb][nb][4 * q] + bias[q].x, acc[mb][nb][4 * q + 1] + bias[q].y,
                              acc[mb][nb][4 * q + 2] + bias[q].z, acc[mb][nb][4 * q + 3] + bias[q].w};
                if (a.silu)
#pragma unroll
                    for (int i = 0; i < 4; ++i) v[i] = silu(v[i]);
                if (a.residual) {
                    v[0] += bf16_to_f32(static_cast<uint16_t>(res[q].x & 0xffffu));
                    v[1] += bf16_to_f32(static_cast<uint16_t>(res[q].x >> 16));
                    v[2] += bf16_to_f32(static_cast<uint16_t>(res[q].y & 0xffffu));
                    v[3] += bf16_to_f32(static_cast<uint16_t>(res[q].y >> 16));
                }
                lo[q] = pack_bf16x2(v[0], v[1]);
                hi[q] = pack_bf16x2(v[2], v[3]);
            }
            uint16_t *yp = static_cast<uint16_t *>(a.y) + row * a.cout + col0 + nb * 32;
#pragma unroll
            for (int h = 0; h < 2; ++h) {
                const auto s0 = __builtin_amdgcn_permlane32_swap(lo[2 * h], lo[2 * h + 1], false, false);
                const auto s1 = __builtin_amdgcn_permlane32_swap(hi[2 * h], hi[2 * h + 1], false, false);
                if (row < a.n_out)
                    *reinterpret_cast<uint4 *>(yp + 8 * (2 * h + half)) = make_uint4(s0[0], s1[0], s0[1], s1[1]);
            }
        }
    }
}

}  // namespace

void launch_rows_plan(const int32_t *kmap, int64_t n_out, int64_t n_src, int64_t tiles, void *plan, hipStream_t stream) {
    hipLaunchKernelGGL(rows_plan_kernel, dim3(static_cast<unsigned>((n_out + kRowsTile - 1) / kRowsTile)), dim3(1024), 0,
                       stream, kmap, n_out, n_src, static_cast<int>(tiles), static_cast<char *>(plan));
}

void launch_conv_rows(const ConvArgs &a, int64_t tiles, hipStream_t stream) {
    hipLaunchKernelGGL(conv_rows_kernel, dim3(static_cast<unsigned>(tiles), static_cast<unsigned>(a.cout_pad / 96)), dim3(256), 0,
                       stream, a);
}

}  // namespace s3dx
