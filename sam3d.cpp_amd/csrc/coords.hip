// Occupancy -> sparse coordinates on the GPU: the steps between the sparse
// structure decoder's occupancy grid and the SLat stage's coordinate table.
//
// Reference (host C++, src/objects_runtime/session.cpp):
//   threshold occ > 0 in x-major order, batch 0        :1437-1441
//   prune_surface_coords (max_neighbor_axes_dist = 1)   :133-163
//   downsample_coords (max 42000, factor 2, seed 42)    :168-233
//
// Each is an ordered stream compaction, so outputs keep the reference's input
// order: two launches, one counting the flagged items of each of at most 1,024
// runs, one that adds the counts before its run and writes the rows out.  The
// steps are bound by their launches and their one synchronization each: a flag
// pass, a scan of five launches and a scatter each, with the tables' clears
// apart, were 32 launches and 242 us for the three steps on a 64^3 grid; these
// are 13 and 136 us.  The
// reference identifies cells by coordinate_key (:122-127: b<<48 | x<<32 |
// y<<16 | z&0xffff, each field zero-extended, so the fields overlap); the
// hash here is keyed by that same 64-bit value, so cells that alias in the
// reference (negative or wide coordinates) alias here too.
#include "coord_hash.hpp"

#include <algorithm>
#include <cmath>
#include <numeric>
#include <random>
#include <vector>

namespace s3dx {
namespace {

// coordinate_key (session.cpp:122-127) as the hash's int4 key: its low and
// high 32-bit words.
__device__ __forceinline__ int4 cell_key(int32_t b, int32_t x, int32_t y, int32_t z) {
    const uint64_t k = (static_cast<uint64_t>(static_cast<uint32_t>(b)) << 48) |
                       (static_cast<uint64_t>(static_cast<uint32_t>(x)) << 32) |
                       (static_cast<uint64_t>(static_cast<uint32_t>(y)) << 16) |
                       static_cast<uint64_t>(static_cast<uint32_t>(z) & 0xffffu);
    return make_int4(static_cast<int32_t>(static_cast<uint32_t>(k)),
                     static_cast<int32_t>(static_cast<uint32_t>(k >> 32)), 0, 0);
}

// ---- ordered compaction -----------------------------------------------------
// Items per run of the two passes, and the runs: whole multiples of 1,024
// items, at most 1,024 runs, so that a block adds up the counts before its own
// with a few loads a thread.
constexpr int64_t kRunItems = 1024;
constexpr int64_t kMaxRuns = 1024;
inline int64_t run_span(int64_t n) {
    const int64_t runs = std::min<int64_t>((n + kRunItems - 1) / kRunItems, kMaxRuns);
    return ((n + runs - 1) / runs + kRunItems - 1) / kRunItems * kRunItems;
}
inline unsigned run_count(int64_t n) { return static_cast<unsigned>((n + run_span(n) - 1) / run_span(n)); }

// counts[run] = the run's items i with flag(i).
template <class Flag>
__global__ void __launch_bounds__(kThreads) count_kernel(Flag flag, int64_t n, int64_t span, int32_t *counts) {
    __shared__ int32_t sums[kThreads / 64];
    const int64_t b = blockIdx.x * span, e = min(n, b + span);
    int32_t c = 0;
    for (int64_t i = b + threadIdx.x; i < e; i += kThreads) c += flag(i) ? 1 : 0;
#pragma unroll
    for (int d = 32; d >= 1; d >>= 1) c += __shfl_xor(c, d, 64);
    if ((threadIdx.x & 63) == 0) sums[threadIdx.x >> 6] = c;
    __syncthreads();
    if (threadIdx.x == 0) {
        for (int w = 1; w < kThreads / 64; ++w) c += sums[w];
        counts[blockIdx.x] = c;
    }
}

// emit(i, position) for every flagged item, positions in item order; *total:
// their count.
template <class Flag, class Emit>
__global__ void __launch_bounds__(kThreads) emit_kernel(Flag flag, Emit emit, int64_t n, int64_t span, const int32_t *counts,
                                                        int32_t *total) {
    constexpr int WAVES = kThreads / 64;
    __shared__ int32_t sums[WAVES];
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    int32_t at = 0;
    for (unsigned r = threadIdx.x; r < blockIdx.x; r += kThreads) at += counts[r];
#pragma unroll
    for (int d = 32; d >= 1; d >>= 1) at += __shfl_xor(at, d, 64);
    if (lane == 0) sums[wave] = at;
    __syncthreads();
    at = 0;
    for (int w = 0; w < WAVES; ++w) at += sums[w];
    const int64_t b = blockIdx.x * span, e = min(n, b + span);
    for (int64_t base = b; base < e; base += kThreads) {
        const int64_t i = base + threadIdx.x;
        const bool f = i < e && flag(i);
        const uint64_t m = __builtin_amdgcn_ballot_w64(f);
        __syncthreads();  // the sums of the pass before are read
        if (lane == 0) sums[wave] = __popcll(m);
        __syncthreads();
        int32_t before = 0, all = 0;
        for (int w = 0; w < WAVES; ++w) {
            before += w < wave ? sums[w] : 0;
            all += sums[w];
        }
        if (f) emit(i, at + before + __popcll(m & ((uint64_t(1) << lane) - 1)));
        at += all;
    }
    if (blockIdx.x == gridDim.x - 1 && threadIdx.x == 0) *total = at;
}

struct OccFlag {
    const float *occ;
    __device__ bool operator()(int64_t i) const { return occ[i] > 0.0f; }
};
// Cell i = (x*ny + y)*nz + z becomes the row (0, x, y, z).
struct OccEmit {
    int32_t ny, nz;
    int4 *out;
    __device__ void operator()(int64_t i, int32_t pos) const {
        const int64_t yz = static_cast<int64_t>(ny) * nz;
        const int64_t x = i / yz;
        const int64_t r = i - x * yz;
        out[pos] = make_int4(0, static_cast<int32_t>(x), static_cast<int32_t>(r / nz), static_cast<int32_t>(r % nz));
    }
};
struct RowFlag {
    const int32_t *flag;
    __device__ bool operator()(int64_t i) const { return flag[i] != 0; }
};
struct RowEmit {
    const int4 *in;
    int4 *out;
    __device__ void operator()(int64_t i, int32_t pos) const { out[pos] = in[i]; }
};
// Rows into `all`, the first `most` of them into `out` as well.
struct TwoRowEmit {
    const int4 *in;
    int4 *all, *out;
    int64_t most;
    __device__ void operator()(int64_t i, int32_t pos) const {
        const int4 c = in[i];
        all[pos] = c;
        if (pos < most) out[pos] = c;
    }
};
// The first row of each key (h built on them), kept for the second pass.
struct FirstFlag {
    Hash h;
    int32_t *flag;
    __device__ bool operator()(int64_t i) const {
        const bool f = hash_find(h, h.keys[i]) == static_cast<int32_t>(i);
        flag[i] = f ? 1 : 0;
        return f;
    }
};

// The prune's cell keys and zeroed flags, and the emptied table, in one grid
// over the table.
__global__ void __launch_bounds__(kThreads)
prune_prepare_kernel(const int4 *__restrict__ coords, int32_t n, Hash h, int4 *__restrict__ keys, int32_t *__restrict__ flag) {
    const uint32_t i = blockIdx.x * kThreads + threadIdx.x;
    hash_clear(h, i);
    if (i >= static_cast<uint32_t>(n)) return;
    const int4 c = coords[i];
    keys[i] = cell_key(c.x, c.y, c.z, c.w);
    flag[i] = 0;
}

// One thread per (voxel, offset): flag[i] = 1 when the cell key of
// coords[i] + d(o) (same b; int32 arithmetic wrapping as on the host) is
// not among the voxels' keys (h built on them).  flag starts at zero; every
// writer writes 1.
__global__ void __launch_bounds__(kThreads)
surface_flag_kernel(const int4 *__restrict__ coords, int32_t n, Hash h, int32_t *__restrict__ flag) {
    const int32_t g = blockIdx.x * kThreads + threadIdx.x;
    if (g >= n * 27) return;
    const int32_t i = g / 27;
    const int32_t o = g - i * 27;
    const int4 c = coords[i];
    auto step = [](int32_t v, int d) {
        return static_cast<int32_t>(static_cast<uint32_t>(v) + static_cast<uint32_t>(d));
    };
    const int4 q = cell_key(c.x, step(c.y, o / 9 - 1), step(c.z, (o / 3) % 3 - 1), step(c.w, o % 3 - 1));
    if (hash_find(h, q) < 0) flag[i] = 1;
}

// Bounding boxes of (x, y, z), one per block: [0..2] min, [3..5] max.
__global__ void __launch_bounds__(kThreads)
xyz_bounds_kernel(const int4 *__restrict__ coords, int32_t n, int32_t *boxes) {
    int v[6] = {INT32_MAX, INT32_MAX, INT32_MAX, INT32_MIN, INT32_MIN, INT32_MIN};
    for (int32_t i = blockIdx.x * kThreads + threadIdx.x; i < n; i += gridDim.x * kThreads) {
        const int4 c = coords[i];
        v[0] = min(v[0], c.y); v[1] = min(v[1], c.z); v[2] = min(v[2], c.w);
        v[3] = max(v[3], c.y); v[4] = max(v[4], c.z); v[5] = max(v[5], c.w);
    }
    block_bounds<3>(v, boxes + blockIdx.x * 6);
}

// One axis of downsample_coords (session.cpp:180-211): the coordinate's
// position in [lo, hi] mapped onto the centred target range of
// (hi - lo + 1) / factor cells, rounded half up, clamped to the range's
// truncated ends.  Double precision, every operation rounded on its own (no
// fused multiply-add), so the results are the host's bit for bit.
__device__ __forceinline__ int32_t downsample_axis(int32_t v, int32_t lo, int32_t hi, int32_t factor) {
#pragma clang fp contract(off)
    const double original = static_cast<double>(hi - lo + 1);
    const double target = original / static_cast<double>(factor);
    const double offset = (original - target) * 0.5;
    const double target_min = static_cast<double>(lo) + offset;
    const double target_max = target_min + target - 1.0;
    const int32_t tmin = static_cast<int32_t>(target_min);  // truncation toward zero
    const int32_t tmax = static_cast<int32_t>(target_max);
    const double denom = static_cast<double>(hi - lo);
    const double normalized = denom > 0.0 ? (static_cast<double>(v) - lo) / denom : 0.0;
    const double value = normalized * (target - 1.0) + target_min;
    int64_t r = static_cast<int64_t>(floor(value + 0.5));
    r = r < tmin ? tmin : r;
    r = r > tmax ? tmax : r;
    return static_cast<int32_t>(r);
}

// The mapped rows, their cell keys and the emptied table, in one grid over the
// table; blocks that map rows first join the `nboxes` (at most 128) boxes.
__global__ void __launch_bounds__(kThreads)
downsample_prepare_kernel(const int4 *__restrict__ coords, int32_t n, const int32_t *__restrict__ boxes, int nboxes,
                          int32_t factor, Hash h, int4 *__restrict__ mapped, int4 *__restrict__ keys) {
    __shared__ int32_t bbox[6];
    const uint32_t i = blockIdx.x * kThreads + threadIdx.x;
    hash_clear(h, i);
    if (blockIdx.x * static_cast<uint32_t>(kThreads) >= static_cast<uint32_t>(n)) return;
    int v[6] = {INT32_MAX, INT32_MAX, INT32_MAX, INT32_MIN, INT32_MIN, INT32_MIN};
    if (static_cast<int>(threadIdx.x) < nboxes)
#pragma unroll
        for (int k = 0; k < 6; ++k) v[k] = boxes[threadIdx.x * 6 + k];
    block_bounds<3>(v, bbox);
    __syncthreads();
    if (i >= static_cast<uint32_t>(n)) return;
    const int4 c = coords[i];
    const int4 m = make_int4(c.x, downsample_axis(c.y, bbox[0], bbox[3], factor),
                             downsample_axis(c.z, bbox[1], bbox[4], factor),
                             downsample_axis(c.w, bbox[2], bbox[5], factor));
    mapped[i] = m;
    keys[i] = cell_key(m.x, m.y, m.z, m.w);
}

__global__ void __launch_bounds__(kThreads)
gather_rows_kernel(const int4 *__restrict__ in, const int32_t *__restrict__ idx, int32_t m,
                   int4 *__restrict__ out) {
    const int32_t j = blockIdx.x * kThreads + threadIdx.x;
    if (j < m) out[j] = in[idx[j]];
}

void check_coord_rows(const int32_t *coords, int64_t n, int64_t max_n) {
    require(coords != nullptr, "coords is NULL");
    require(aligned(coords, 16), "coords must be 16-byte aligned");
    require(n > 0, "voxel count must be positive");
    require(n <= max_n, "voxel count out of range");
}

int64_t read_count(const int32_t *total, hipStream_t s) {
    int32_t v = 0;
    hip_check(hipMemcpyAsync(&v, total, sizeof(v), hipMemcpyDeviceToHost, s), "hipMemcpyAsync count");
    hip_check(hipStreamSynchronize(s), "hipStreamSynchronize");
    return v;
}

// ---- workspace layouts (runs: the run counts, or at most 128 boxes) ----------
struct OccLayout {
    int32_t *runs, *totals;
};
template <class W>
void occ_layout(W &w, OccLayout *l) {
    if constexpr (std::is_same_v<W, Carver>) {
        l->runs = w.template take<int32_t>(kMaxRuns);
        l->totals = w.template take<int32_t>(8);
    } else {
        w.template take<int32_t>(kMaxRuns);
        w.template take<int32_t>(8);
    }
}

struct PruneLayout {
    Hash hash;
    int4 *keys;
    int32_t *flag, *runs, *totals;
};
template <class W>
void prune_layout(W &w, int64_t n, PruneLayout *l) {
    const uint64_t u = static_cast<uint64_t>(n);
    if constexpr (std::is_same_v<W, Carver>) {
        hash_layout(w, n, &l->hash);
        l->keys = w.template take<int4>(u);
        l->flag = w.template take<int32_t>(u);
        l->runs = w.template take<int32_t>(kMaxRuns);
        l->totals = w.template take<int32_t>(8);
    } else {
        hash_layout(w, n, static_cast<Hash *>(nullptr));
        w.template take<int4>(u);
        w.template take<int32_t>(u);
        w.template take<int32_t>(kMaxRuns);
        w.template take<int32_t>(8);
    }
}

struct DownsampleLayout {
    Hash hash;
    int32_t *flag, *idx, *runs, *totals;
    int4 *mapped, *keys, *unique;
};
template <class W>
void downsample_layout(W &w, int64_t n, DownsampleLayout *l) {
    const uint64_t u = static_cast<uint64_t>(n);
    if constexpr (std::is_same_v<W, Carver>) {
        hash_layout(w, n, &l->hash);
        l->flag = w.template take<int32_t>(u);
        l->idx = w.template take<int32_t>(u);
        l->runs = w.template take<int32_t>(kMaxRuns);
        l->totals = w.template take<int32_t>(8);
        l->mapped = w.template take<int4>(u);
        l->keys = w.template take<int4>(u);
        l->unique = w.template take<int4>(u);
    } else {
        hash_layout(w, n, static_cast<Hash *>(nullptr));
        for (int k = 0; k < 2; ++k) w.template take<int32_t>(u);
        w.template take<int32_t>(kMaxRuns);
        w.template take<int32_t>(8);
        for (int k = 0; k < 3; ++k) w.template take<int4>(u);
    }
}

}  // namespace
}  // namespace s3dx

using namespace s3dx;

extern "C" {

S3DX_API s3dx_status s3dx_occupancy_workspace_size(int32_t nx, int32_t ny, int32_t nz, uint64_t *bytes,
                                                   char *error, uint64_t error_capacity) {
    return boundary(error, error_capacity, [&] {
        require(bytes != nullptr, "bytes is NULL");
        require(nx > 0 && ny > 0 && nz > 0, "grid extents must be positive");
        const int64_t cells = static_cast<int64_t>(nx) * ny * nz;
        require(cells <= INT32_MAX, "grid has more than INT32_MAX cells");
        Sizer s;
        occ_layout(s, nullptr);
        *bytes = s.used;
    });
}

S3DX_API s3dx_status s3dx_occupancy_coords(const float *occupancy, int32_t nx, int32_t ny, int32_t nz,
                                           int32_t *coords, int64_t *count, void *workspace,
                                           uint64_t workspace_bytes, s3dx_stream stream, char *error,
                                           uint64_t error_capacity) {
    return boundary(error, error_capacity, [&] {
        require(occupancy && coords && count && workspace, "NULL argument");
        require(aligned(coords, 16), "coords must be 16-byte aligned");
        require(nx > 0 && ny > 0 && nz > 0, "grid extents must be positive");
        const int64_t cells = static_cast<int64_t>(nx) * ny * nz;
        require(cells <= INT32_MAX, "grid has more than INT32_MAX cells");
        const hipStream_t s = as_stream(stream);
        Carver w(workspace, workspace_bytes);
        OccLayout l;
        occ_layout(w, &l);
        const OccFlag flag{occupancy};
        count_kernel<<<run_count(cells), kThreads, 0, s>>>(flag, cells, run_span(cells), l.runs);
        launch_check("occ_count");
        emit_kernel<<<run_count(cells), kThreads, 0, s>>>(flag, OccEmit{ny, nz, reinterpret_cast<int4 *>(coords)}, cells,
                                                          run_span(cells), l.runs, l.totals);
        launch_check("occ_emit");
        *count = read_count(l.totals, s);
    });
}

S3DX_API s3dx_status s3dx_prune_surface_workspace_size(int64_t n, uint64_t *bytes, char *error,
                                                       uint64_t error_capacity) {
    return boundary(error, error_capacity, [&] {
        require(bytes != nullptr, "bytes is NULL");
        require(n > 0 && n <= INT32_MAX / 27, "voxel count out of range");
        Sizer s;
        prune_layout(s, n, nullptr);
        *bytes = s.used;
    });
}

S3DX_API s3dx_status s3dx_prune_surface(const int32_t *coords, int64_t n, int32_t *surface,
                                        int64_t *count, void *workspace, uint64_t workspace_bytes,
                                        s3dx_stream stream, char *error, uint64_t error_capacity) {
    return boundary(error, error_capacity, [&] {
        check_coord_rows(coords, n, INT32_MAX / 27);
        require(surface && count && workspace, "NULL argument");
        require(aligned(surface, 16), "surface must be 16-byte aligned");
        const hipStream_t s = as_stream(stream);
        const int32_t ni = static_cast<int32_t>(n);
        Carver w(workspace, workspace_bytes);
        PruneLayout l;
        prune_layout(w, n, &l);
        const int4 *c4 = reinterpret_cast<const int4 *>(coords);
        l.hash.keys = l.keys;
        prune_prepare_kernel<<<blocks_for(static_cast<int64_t>(l.hash.mask) + 1), kThreads, 0, s>>>(c4, ni, l.hash, l.keys,
                                                                                                   l.flag);
        launch_check("prune_prepare");
        hash_insert(l.hash, ni, s);
        surface_flag_kernel<<<blocks_for(n * 27), kThreads, 0, s>>>(c4, ni, l.hash, l.flag);
        launch_check("surface_flag");
        const RowFlag flag{l.flag};
        count_kernel<<<run_count(n), kThreads, 0, s>>>(flag, n, run_span(n), l.runs);
        launch_check("surface_count");
        emit_kernel<<<run_count(n), kThreads, 0, s>>>(flag, RowEmit{c4, reinterpret_cast<int4 *>(surface)}, n, run_span(n),
                                                      l.runs, l.totals);
        launch_check("surface_emit");
        *count = read_count(l.totals, s);
    });
}

S3DX_API s3dx_status s3dx_downsample_coords_workspace_size(int64_t n, uint64_t *bytes, char *error,
                                                           uint64_t error_capacity) {
    return boundary(error, error_capacity, [&] {
        require(bytes != nullptr, "bytes is NULL");
        require(n > 0 && n <= INT32_MAX, "voxel count out of range");
        Sizer s;
        downsample_layout(s, n, nullptr);
        *bytes = s.used;
    });
}

S3DX_API s3dx_status s3dx_downsample_coords(const int32_t *coords, int64_t n, int64_t max_coords,
                                            int32_t factor, uint32_t seed, int32_t *out, int64_t *count,
                                            void *workspace, uint64_t workspace_bytes, s3dx_stream stream,
                                            char *error, uint64_t error_capacity) {
    return boundary(error, error_capacity, [&] {
        check_coord_rows(coords, n, INT32_MAX);
        require(out && count && workspace, "NULL argument");
        require(aligned(out, 16), "out must be 16-byte aligned");
        require(max_coords >= 0, "max_coords must be non-negative");
        require(factor > 0, "downsample factor must be positive");
        const hipStream_t s = as_stream(stream);
        // At most max_coords rows: the set is returned as it is
        // (session.cpp:174), duplicates included.
        if (n <= max_coords) {
            hip_check(hipMemcpyAsync(out, coords, static_cast<size_t>(n) * 16, hipMemcpyDeviceToDevice, s),
                      "hipMemcpyAsync");
            *count = n;
            return;
        }
        const int32_t ni = static_cast<int32_t>(n);
        Carver w(workspace, workspace_bytes);
        DownsampleLayout l;
        downsample_layout(w, n, &l);
        const int4 *c4 = reinterpret_cast<const int4 *>(coords);
        const unsigned boxes = bounds_blocks(n);
        xyz_bounds_kernel<<<boxes, kThreads, 0, s>>>(c4, ni, l.runs);
        launch_check("xyz_bounds");
        l.hash.keys = l.keys;
        downsample_prepare_kernel<<<blocks_for(static_cast<int64_t>(l.hash.mask) + 1), kThreads, 0, s>>>(
            c4, ni, l.runs, static_cast<int>(boxes), factor, l.hash, l.mapped, l.keys);
        launch_check("downsample_prepare");
        // First occurrence of each mapped cell key, in input order (:213-215).
        hash_insert(l.hash, ni, s);
        count_kernel<<<run_count(n), kThreads, 0, s>>>(FirstFlag{l.hash, l.flag}, n, run_span(n), l.runs);
        launch_check("first_count");
        emit_kernel<<<run_count(n), kThreads, 0, s>>>(
            RowFlag{l.flag}, TwoRowEmit{l.mapped, l.unique, reinterpret_cast<int4 *>(out), max_coords}, n, run_span(n),
            l.runs, l.totals);
        launch_check("first_emit");
        const int64_t unique_n = read_count(l.totals, s);
        if (unique_n <= max_coords) {
            *count = unique_n;
            return;
        }
        // More than max_coords cells: the reference's sample, the first
        // max_coords entries of a std::shuffle of 0..unique_n-1 under
        // std::mt19937(seed) (:217-229).  The permutation depends only on
        // unique_n and the seed, so the host draws it with the same standard
        // library and the GPU gathers the rows.
        std::mt19937 rng(seed);
        std::vector<size_t> order(static_cast<size_t>(unique_n));
        std::iota(order.begin(), order.end(), size_t(0));
        std::shuffle(order.begin(), order.end(), rng);
        std::vector<int32_t> pick(static_cast<size_t>(max_coords));
        for (size_t j = 0; j < pick.size(); ++j) pick[j] = static_cast<int32_t>(order[j]);
        if (!pick.empty()) {
            hip_check(hipMemcpyAsync(l.idx, pick.data(), pick.size() * sizeof(int32_t), hipMemcpyHostToDevice, s),
                      "hipMemcpyAsync");
            gather_rows_kernel<<<blocks_for(max_coords), kThreads, 0, s>>>(
                l.unique, l.idx, static_cast<int32_t>(max_coords), reinterpret_cast<int4 *>(out));
            launch_check("gather_rows");
            hip_check(hipStreamSynchronize(s), "hipStreamSynchronize");  // pick stays alive until the copy ends
        }
        *count = max_coords;
    });
}

}  // extern "C"
