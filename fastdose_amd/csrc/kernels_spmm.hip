// kernels_spmm.hip -- 16-bit packing of the dose-loading matrix and D^T X products (gfx950).
//
// The optimiser of the reference multiplies the dose-loading matrix by fluence vectors
// (dose = D^T x, IMRTOpt/src/IMRTOptimize.cu:604-625 through cuSPARSE; IMRTDebug.cu:211-315).
// Here the ensemble of per-beam CSR matrices (rows = beamlets, columns = voxels) is:
//   - packed: per row a FP32 scale (the row maximum) and values q = v / scale rounded to
//     BF16 or FP16 (round to nearest even);
//   - transposed to a voxel-major copy (CSC): a column's entries sorted by row, so every product
//     sums in a fixed order and is bitwise reproducible;
//   - multiplied with FP32 accumulation, the lanes of a wavefront spread over right-hand sides,
//     entries and columns according to k and the columns' lengths.
#include <hip/hip_runtime.h>

#include <cfloat>
#include <type_traits>

#include "kernels.h"

namespace fdi {
namespace {

__device__ __forceinline__ uint16_t f32_to_bf16_rne(float f) {
    const uint32_t u = __float_as_uint(f);
    return (uint16_t)((u + 0x7FFFu + ((u >> 16) & 1u)) >> 16);  // finite inputs only
}
__device__ __forceinline__ float bf16_to_f32(uint16_t h) { return __uint_as_float((uint32_t)h << 16); }
__device__ __forceinline__ uint16_t f32_to_fp16_rne(float f) {
    const _Float16 h = (_Float16)f;
    return __builtin_bit_cast(uint16_t, h);
}
__device__ __forceinline__ float fp16_to_f32(uint16_t h) { return (float)__builtin_bit_cast(_Float16, h); }

// rowptr[r] (global, r in [0, R]) from the ensemble's per-matrix local offsets.
__global__ void global_rows_kernel(int n_mat, const uint64_t* __restrict__ row_first,
                                   const uint64_t* __restrict__ off_off, const uint64_t* __restrict__ nnz_off,
                                   const uint64_t* __restrict__ offsets, uint64_t R, uint64_t total_nnz,
                                   uint64_t* __restrict__ rowptr) {
    const uint64_t r = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (r > R) return;
    if (r == R) {
        rowptr[R] = total_nnz;
        return;
    }
    int lo = 0, hi = n_mat - 1;  // matrix k with row_first[k] <= r < row_first[k + 1]
    while (lo < hi) {
        const int mid = (lo + hi + 1) >> 1;
        if (row_first[mid] <= r) lo = mid; else hi = mid - 1;
    }
    rowptr[r] = nnz_off[lo] + offsets[off_off[lo] + (r - row_first[lo])];
}

// ---- Voxel-major copy of rows with ascending columns.
//
// The columns are cut into tiles of kTileCols or kNarrowTile.  A row's entries of one tile are contiguous, so one
// pass over the rows (row_tiles_kernel, HBM-bound on the 8-byte columns) writes where every tile
// starts in every row, and one workgroup per tile then places the tile's entries: it lists the rows
// that reach the tile (list_rows), counts the entries per column in LDS, scans the counts into the
// column pointers, and takes the listed rows in order, up to 64 rows and 64 units of 64 entries at a
// time (row_group).  Within such a group each entry sets the bit of its row in its column's 64-bit LDS
// mask; after a barrier the entry's place is its column's running offset plus the mask's bits below
// its row.  Every column comes out sorted by row without a sort, and without global atomics.  Before,
// an atomic scatter and one insertion sort per column took 16.9 ms for 52 M entries (20 beams, 2 726
// rows, 200 x 200 x 160 voxels; 14.2 of them the sort: the voxels of the target hold hundreds of
// entries each).  Placing takes 1.06 ms of the 1.3 now; it took 1.55 with groups of 64 consecutive rows
// of the matrix, of which about 15 reach a tile (few loads in flight per barrier), 1.22 with the tiles in
// volume order.  What is left waits for scattered loads and stores (1.4 GB of HBM traffic, 1.3 TB/s).
// kTileCols: a beamlet's footprint is about ten voxels wide, so 2048 columns (ten x-rows of a
// 200-voxel plane) hold about one wavefront of a row's entries, and the tile's LDS (39.5 KiB) lets
// four workgroups of eight wavefronts share a CU.
// kNarrowTile: in small volumes, where the tiles are fewer than the CUs, and with enough rows for a tile's
// serial part (the rounds over its rows) to weigh more than a tile table of four times the size: an
// operator of 60 pencil rows on 61 x 63 x 65 voxels is built in 95 us instead of 111, of 400 rows in 222
// instead of 267; 7 rows would take 82 instead of 77.  The general path still is up to 15 % faster for
// rows of a few entries scattered over a small volume, but its sort of one crowded column can take seconds.
constexpr int kTileCols = 2048, kNarrowTile = 512;
constexpr uint64_t kNarrowBelow = 192 * (uint64_t)kTileCols, kNarrowRow = 8192;
constexpr int kPlaceThreads = 512;

// tiles[r * (n_tiles + 1) + t] = entries of row r before tile t (t = n_tiles: all of them), and for
// 16-bit values scale[r] = the row maximum.  Sets *unsorted when a row's columns do not ascend
// strictly or reach beyond C (the caller then takes the general path).
__global__ __launch_bounds__(256) void row_tiles_kernel(const uint64_t* __restrict__ rowptr,
                                                        const uint64_t* __restrict__ columns,
                                                        const float* __restrict__ values, uint64_t C,
                                                        uint32_t shift, uint32_t n_tiles,
                                                        uint32_t* __restrict__ tiles, float* __restrict__ scale,
                                                        uint32_t* __restrict__ unsorted) {
    __shared__ float s_max[4];
    const uint64_t r = blockIdx.x;
    const uint64_t a = rowptr[r], n = rowptr[r + 1] - a;
    uint32_t* row = tiles + r * (uint64_t)(n_tiles + 1);
    float m = 0.0f;
    bool bad = false;
    for (uint64_t i = threadIdx.x; i <= n; i += blockDim.x) {
        const uint64_t c = i < n ? columns[a + i] : C;
        const uint64_t p = i > 0 ? columns[a + i - 1] : 0;
        bad |= (i > 0 && p >= c) || (i < n && c >= C);
        // tiles after the previous entry's, up to this one's, start here
        uint64_t t = i > 0 ? (p >> shift) + 1 : 0;
        uint64_t t1 = i < n ? c >> shift : n_tiles;
        t1 = t1 < n_tiles ? t1 : n_tiles;
        for (; t <= t1; t++) row[t] = (uint32_t)i;
        if (scale && i < n) m = fmaxf(m, values[a + i]);
    }
    if (__any(bad) && (threadIdx.x & 63) == 0) atomicOr(unsorted, 1u);
    if (!scale) return;
#pragma unroll
    for (int o = 32; o > 0; o >>= 1) m = fmaxf(m, __shfl_xor(m, o, 64));
    if ((threadIdx.x & 63) == 0) s_max[threadIdx.x >> 6] = m;
    __syncthreads();
    if (threadIdx.x == 0) scale[r] = fmaxf(fmaxf(s_max[0], s_max[1]), fmaxf(s_max[2], s_max[3]));
}

// total[t] (zeroed by the caller) += entries of tile t in this workgroup's kTotalRows rows, all in flight
// (64 rows one after the other: 19 us against 8 for 3000 rows of 98 tiles)
constexpr uint32_t kTotalRows = 16;
__global__ __launch_bounds__(256) void tile_totals_kernel(uint64_t R, uint32_t n_tiles,
                                                          const uint32_t* __restrict__ tiles,
                                                          uint32_t* __restrict__ total) {
    const uint32_t t = blockIdx.x * blockDim.x + threadIdx.x;
    if (t >= n_tiles) return;
    uint32_t lo[kTotalRows], hi[kTotalRows], sum = 0;
#pragma unroll
    for (uint32_t i = 0; i < kTotalRows; i++) {
        const uint64_t r = (uint64_t)blockIdx.y * kTotalRows + i;
        const uint32_t* row = tiles + (r < R ? r : R - 1) * (uint64_t)(n_tiles + 1) + t;
        lo[i] = row[0];
        hi[i] = r < R ? row[1] : lo[i];
    }
#pragma unroll
    for (uint32_t i = 0; i < kTotalRows; i++) sum += hi[i] - lo[i];
    if (sum) atomicAdd(&total[t], sum);
}

template <int VT>
struct StoredValue {
    typedef uint16_t type;
};
template <>
struct StoredValue<FD_VAL_F32> {
    typedef float type;
};
template <int VT>
__device__ __forceinline__ typename StoredValue<VT>::type stored(float v, const float* __restrict__ scale, uint64_t r) {
    if constexpr (VT == FD_VAL_F32)
        return v;
    else if constexpr (VT == FD_VAL_BF16)
        return f32_to_bf16_rne(v / scale[r]);
    else
        return f32_to_fp16_rne(v / scale[r]);
}

// lane `src` of a value (src wave-uniform)
__device__ __forceinline__ uint32_t lane_u32(uint32_t v, int src) {
    return (uint32_t)__builtin_amdgcn_readlane((int)v, src);
}
__device__ __forceinline__ uint64_t lane_u64(uint64_t v, int src) {
    return ((uint64_t)lane_u32((uint32_t)(v >> 32), src) << 32) | lane_u32((uint32_t)v, src);
}

// The rows that reach a tile, in order: appended to a list in LDS, kPlaceThreads rows of the matrix at
// a time, until it could overflow or the rows end.  Called by the whole workgroup.
constexpr int kListRows = 1984;  // four workgroups to a CU with the masks and offsets
constexpr int kRowBits = 20;  // of a list word; the entries of a row in a tile (kTileCols at most) above
static_assert(kTileCols < (1 << (32 - kRowBits)), "a list word holds a row's entry count");
struct TileRows {
    uint32_t* before;  // [kListRows] entries of the row before the tile
    uint32_t* word;    // [kListRows] row | entries << kRowBits
    uint32_t* wave;    // [kPlaceThreads / 64 + 1]
};
__device__ __forceinline__ uint32_t list_rows(const TileRows& T, uint64_t& r0, uint64_t R, uint32_t n_tiles,
                                              uint32_t tile, const uint32_t* __restrict__ tiles) {
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    uint32_t n = 0;
    while (r0 < R && n + kPlaceThreads <= kListRows) {
        const uint64_t r = r0 + threadIdx.x;
        uint32_t lo = 0, len = 0;
        if (r < R) {
            const uint32_t* row = tiles + r * (uint64_t)(n_tiles + 1) + tile;
            lo = row[0];
            len = row[1] - lo;
        }
        const uint64_t some = __ballot(len != 0);
        if (lane == 0) T.wave[wave] = (uint32_t)__popcll(some);
        __syncthreads();
        uint32_t at = n + (uint32_t)__popcll(some & ((1ull << lane) - 1ull));
        for (int w = 0; w < kPlaceThreads / 64; w++) {
            const uint32_t c = T.wave[w];
            at += w < wave ? c : 0u;
            n += c;
        }
        if (len != 0) {
            T.before[at] = lo;
            T.word[at] = (uint32_t)r | (len << kRowBits);
        }
        r0 += kPlaceThreads;
        __syncthreads();
    }
    return n;
}

// Rows g .. g + taken - 1 of the list, cut into units of up to 64 entries: lane l holds row g + l's first
// entry, list word and the number of units before it.
struct RowGroup {
    uint64_t start;
    uint32_t word, first;
    int taken;       // rows
    uint32_t units;
    // unit u's row (its place in the group), first entry and number of entries, all wavefront-uniform
    __device__ __forceinline__ int unit(uint32_t u, uint64_t& e0, uint32_t& n) const {
        const int l = __popcll(__ballot((int)(threadIdx.x & 63) < taken && first <= u)) - 1;
        const uint32_t skip = 64u * (u - lane_u32(first, l));
        e0 = lane_u64(start, l) + skip;
        n = min((lane_u32(word, l) >> kRowBits) - skip, 64u);
        return l;
    }
};
// most: units the group may have (a single row has at most kTileCols / 64); at most 64 rows
__device__ __forceinline__ RowGroup row_group(const TileRows& T, const uint64_t* __restrict__ rowptr, uint32_t g,
                                              uint32_t n_list, uint32_t most) {
    const int lane = threadIdx.x & 63;
    const uint32_t i = g + lane;
    RowGroup G;
    G.word = i < n_list ? T.word[i] : 0u;
    G.start = i < n_list ? rowptr[G.word & ((1u << kRowBits) - 1u)] + T.before[i] : 0u;
    const uint32_t nu = ((G.word >> kRowBits) + 63) >> 6;
    uint32_t x = nu;
#pragma unroll
    for (int o = 1; o < 64; o <<= 1) {
        const uint32_t y = __shfl_up(x, o, 64);
        if (lane >= o) x += y;
    }
    G.first = x - nu;
    G.taken = __popcll(__ballot(nu != 0 && x <= most));
    G.units = lane_u32(x, G.taken - 1);
    return G;
}

// Order in which the tiles are placed.  Neighbouring tiles share lines of the tile table, so groups of
// kTileGroup of them go to one XCD (the dispatcher deals workgroups to the 8 XCDs round-robin); the
// fullest groups first, since the tiles of the target, in the middle of the volume, hold many times
// the entries of the others and would finish last (CUs busy for 60 % of the kernel in volume order).
// order[i] = the i-th group, by falling totals in classes of a quarter octave; one workgroup.
constexpr uint32_t kXcd = 8, kTileGroup = 16;
__device__ __forceinline__ uint32_t size_class(uint64_t n) {  // 0: fullest
    if (n < 4) return 255u - (uint32_t)n;
    const uint32_t e = 63u - (uint32_t)__builtin_clzll(n);
    return 255u - (4u * (e - 1u) + (uint32_t)((n >> (e - 2)) & 3u));
}
__global__ __launch_bounds__(1024) void tile_order_kernel(uint32_t n_tiles, const uint64_t* __restrict__ tile_base,
                                                          uint32_t* __restrict__ order) {
    __shared__ uint32_t s_at[256];
    const uint32_t n_groups = (n_tiles + kTileGroup - 1) / kTileGroup;
    auto cls = [&](uint32_t g) {
        return size_class(tile_base[min((g + 1) * kTileGroup, n_tiles)] - tile_base[g * kTileGroup]);
    };
    if (threadIdx.x < 256) s_at[threadIdx.x] = 0;
    __syncthreads();
    for (uint32_t g = threadIdx.x; g < n_groups; g += blockDim.x) atomicAdd(&s_at[cls(g)], 1u);
    __syncthreads();
    if (threadIdx.x < 64) {  // exclusive scan, four classes per lane
        uint32_t c[4], sum = 0;
        for (int i = 0; i < 4; i++) {
            c[i] = s_at[4 * threadIdx.x + i];
            sum += c[i];
        }
        uint32_t x = sum;
        for (int o = 1; o < 64; o <<= 1) {
            const uint32_t y = __shfl_up(x, o, 64);
            if ((int)threadIdx.x >= o) x += y;
        }
        uint32_t run = x - sum;
        for (int i = 0; i < 4; i++) {
            s_at[4 * threadIdx.x + i] = run;
            run += c[i];
        }
    }
    __syncthreads();
    for (uint32_t g = threadIdx.x; g < n_groups; g += blockDim.x) order[atomicAdd(&s_at[cls(g)], 1u)] = g;
}

template <int VT, int COLS>
__global__ __launch_bounds__(kPlaceThreads) void place_tile_kernel(
    uint64_t R, uint64_t C, uint32_t n_tiles, const uint32_t* __restrict__ tiles, const uint64_t* __restrict__ rowptr,
    const uint64_t* __restrict__ columns, const float* __restrict__ values, const float* __restrict__ scale,
    const uint64_t* __restrict__ tile_base, const uint32_t* __restrict__ order, uint64_t* __restrict__ colptr,
    uint32_t* __restrict__ crow, void* __restrict__ cval_out) {
    typedef typename StoredValue<VT>::type V;
    __shared__ uint32_t s_next[COLS];     // counts, then where each column's next entry goes
    __shared__ uint32_t s_mask[2][COLS];  // rows of the block that hold the column (low, high half)
    __shared__ uint32_t s_wave[kPlaceThreads / 64 + 1];
    __shared__ uint32_t s_before[kListRows];
    __shared__ uint32_t s_word[kListRows];
    constexpr int kWaves = kPlaceThreads / 64, kCols = COLS / kPlaceThreads;
    constexpr uint32_t kUnits = 64;  // a group's units: eight to a wavefront, all in flight
    static_assert(kUnits >= kTileCols / 64 && kUnits == 8 * kWaves, "any row fits a group");
    const uint32_t turn = blockIdx.x / kXcd;  // workgroup blockIdx.x runs on XCD blockIdx.x % kXcd
    const uint32_t slot = turn / kTileGroup * kXcd + blockIdx.x % kXcd;
    if (slot >= (n_tiles + kTileGroup - 1) / kTileGroup) return;
    const uint32_t tile = order[slot] * kTileGroup + turn % kTileGroup;
    if (tile >= n_tiles) return;
    const uint64_t c0 = (uint64_t)tile * COLS;
    const uint64_t base = tile_base[tile];
    const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const TileRows T{s_before, s_word, s_wave};
    V* __restrict__ cval = (V*)cval_out;
    for (int i = tid; i < COLS; i += kPlaceThreads) {
        s_next[i] = 0u;
        s_mask[0][i] = 0u;
        s_mask[1][i] = 0u;
    }
    // entries per column
    uint64_t r_next = 0;
    uint32_t n_list = 0;
    bool whole = true;  // the list holds every row that reaches the tile
    do {
        n_list = list_rows(T, r_next, R, n_tiles, tile, tiles);
        whole = whole && r_next >= R;
        for (uint32_t g = 0; g < n_list;) {
            const RowGroup G = row_group(T, rowptr, g, n_list, ~0u);
            for (uint32_t u0 = wave; u0 < G.units; u0 += kUnits) {
                uint32_t col[8];
#pragma unroll
                for (int q = 0; q < 8; q++) {
                    const uint32_t u = u0 + kWaves * q;
                    uint64_t e0 = 0;
                    uint32_t n = 0;
                    if (u < G.units) G.unit(u, e0, n);
                    col[q] = (uint32_t)lane < n ? (uint32_t)(columns[e0 + lane] - c0) : ~0u;
                }
#pragma unroll
                for (int q = 0; q < 8; q++)
                    if (col[q] != ~0u) atomicAdd(&s_next[col[q]], 1u);
            }
            g += (uint32_t)G.taken;
        }
        __syncthreads();
    } while (r_next < R);
    // column pointers, and offsets within the tile: thread tid owns columns kCols tid ...
    {
        uint32_t n[kCols], sum = 0;
#pragma unroll
        for (int i = 0; i < kCols; i++) {
            n[i] = s_next[kCols * tid + i];
            sum += n[i];
        }
        uint32_t x = sum;
#pragma unroll
        for (int o = 1; o < 64; o <<= 1) {
            const uint32_t y = __shfl_up(x, o, 64);
            if (lane >= o) x += y;
        }
        if (lane == 63) s_wave[wave] = x;
        __syncthreads();
        uint32_t run = x - sum;
        for (int w = 0; w < wave; w++) run += s_wave[w];
#pragma unroll
        for (int i = 0; i < kCols; i++) {
            const uint64_t c = c0 + (uint64_t)(kCols * tid + i);
            if (c < C) colptr[c] = base + run;
            s_next[kCols * tid + i] = run;
            run += n[i];
        }
        if (tid == kPlaceThreads - 1 && tile == n_tiles - 1) colptr[C] = base + run;
    }
    __syncthreads();
    if (!whole) r_next = 0;
    do {
        if (!whole) n_list = list_rows(T, r_next, R, n_tiles, tile, tiles);
        for (uint32_t g = 0; g < n_list;) {
            const RowGroup G = row_group(T, rowptr, g, n_list, kUnits);
            auto group = [&](auto slots) {
                constexpr int Q = decltype(slots)::value;
                uint32_t col[Q], r[Q];
                float val[Q];
                int at[Q];  // the row's place in the group: its bit in the masks
#pragma unroll
                for (int q = 0; q < Q; q++) {
                    const uint32_t u = wave + kWaves * q;
                    uint64_t e0 = 0;
                    uint32_t n = 0;
                    at[q] = u < G.units ? G.unit(u, e0, n) : 0;
                    r[q] = lane_u32(G.word, at[q]) & ((1u << kRowBits) - 1u);
                    const bool on = (uint32_t)lane < n;
                    col[q] = on ? (uint32_t)(columns[e0 + lane] - c0) : ~0u;
                    val[q] = on ? values[e0 + lane] : 0.0f;
                }
#pragma unroll
                for (int q = 0; q < Q; q++)
                    if (col[q] != ~0u) atomicOr(&s_mask[at[q] >> 5][col[q]], 1u << (at[q] & 31));
                __syncthreads();
#pragma unroll
                for (int q = 0; q < Q; q++) {
                    if (col[q] == ~0u) continue;
                    const uint32_t below = (1u << (at[q] & 31)) - 1u;
                    const uint32_t lo = s_mask[0][col[q]];
                    const uint32_t before =
                        at[q] < 32 ? __popc(lo & below) : __popc(lo) + __popc(s_mask[1][col[q]] & below);
                    const uint64_t pos = base + s_next[col[q]] + before;
                    crow[pos] = r[q];
                    cval[pos] = stored<VT>(val[q], scale, r[q]);
                }
            };
            if (G.units > 2 * kWaves)
                group(std::integral_constant<int, 8>{});
            else
                group(std::integral_constant<int, 2>{});
            __syncthreads();
#pragma unroll
            for (int i = 0; i < kCols; i++) {
                const int c = tid + kPlaceThreads * i;
                s_next[c] += __popc(s_mask[0][c]) + __popc(s_mask[1][c]);
                s_mask[0][c] = 0u;
                s_mask[1][c] = 0u;
            }
            __syncthreads();
            g += (uint32_t)G.taken;
        }
    } while (!whole && r_next < R);
}

// ---- The general path (columns in any order, or rows too short for the tile table).

// one wavefront per row: scale = row maximum; q = v / scale in 16 bits (scale 0 for an empty row)
__global__ __launch_bounds__(256) void pack_rows_kernel(uint64_t R, const uint64_t* __restrict__ rowptr,
                                                        const float* __restrict__ values, int vtype,
                                                        float* __restrict__ scale, uint16_t* __restrict__ q) {
    const uint64_t r = ((uint64_t)blockIdx.x * blockDim.x + threadIdx.x) >> 6;
    const int lane = threadIdx.x & 63;
    if (r >= R) return;
    const uint64_t a = rowptr[r], b = rowptr[r + 1];
    float m = 0.0f;
    for (uint64_t e = a + lane; e < b; e += 64) m = fmaxf(m, values[e]);
#pragma unroll
    for (int o = 32; o > 0; o >>= 1) m = fmaxf(m, __shfl_xor(m, o, 64));
    if (lane == 0) scale[r] = m;
    for (uint64_t e = a + lane; e < b; e += 64) {
        const float t = values[e] / m;
        q[e] = vtype == FD_VAL_BF16 ? f32_to_bf16_rne(t) : f32_to_fp16_rne(t);
    }
}

__global__ void col_count_kernel(uint64_t nnz, const uint64_t* __restrict__ columns, uint32_t* __restrict__ count) {
    for (uint64_t e = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x; e < nnz; e += (uint64_t)gridDim.x * blockDim.x)
        atomicAdd(&count[columns[e]], 1u);
}

// one wavefront per row: entries to their column segment (order inside a column fixed later)
template <typename V>
__global__ __launch_bounds__(256) void col_scatter_kernel(uint64_t R, const uint64_t* __restrict__ rowptr,
                                                          const uint64_t* __restrict__ columns,
                                                          const V* __restrict__ vals,
                                                          const uint64_t* __restrict__ colptr,
                                                          uint32_t* __restrict__ cursor, uint32_t* __restrict__ crow,
                                                          V* __restrict__ cval) {
    const uint64_t r = ((uint64_t)blockIdx.x * blockDim.x + threadIdx.x) >> 6;
    const int lane = threadIdx.x & 63;
    if (r >= R) return;
    for (uint64_t e = rowptr[r] + lane; e < rowptr[r + 1]; e += 64) {
        const uint64_t c = columns[e];
        const uint64_t pos = colptr[c] + atomicAdd(&cursor[c], 1u);
        crow[pos] = (uint32_t)r;
        cval[pos] = vals[e];
    }
}

// one thread per column: insertion sort of its (row, value) entries by row
template <typename V>
__global__ void col_sort_kernel(uint64_t C, const uint64_t* __restrict__ colptr, uint32_t* __restrict__ crow,
                                V* __restrict__ cval) {
    const uint64_t c = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (c >= C) return;
    const uint64_t a = colptr[c], b = colptr[c + 1];
    for (uint64_t i = a + 1; i < b; i++) {
        const uint32_t kr = crow[i];
        const V kv = cval[i];
        uint64_t j = i;
        while (j > a && crow[j - 1] > kr) {
            crow[j] = crow[j - 1];
            cval[j] = cval[j - 1];
            j--;
        }
        crow[j] = kr;
        cval[j] = kv;
    }
}

// An entry's stored number, and its value (16-bit numbers are fractions of the row maximum)
template <int VT>
__device__ __forceinline__ float stored_number(const void* cval, uint64_t e) {
    if (VT == FD_VAL_F32) return ((const float*)cval)[e];
    const uint16_t h = ((const uint16_t*)cval)[e];
    return VT == FD_VAL_BF16 ? bf16_to_f32(h) : fp16_to_f32(h);
}
template <int VT>
__device__ __forceinline__ float entry_value(const void* cval, uint64_t e, const float* scale, uint32_t r) {
    const float q = stored_number<VT>(cval, e);
    return VT == FD_VAL_F32 ? q : q * scale[r];
}

typedef float v4f __attribute__((ext_vector_type(4)));

// Y[c][j] = sum over column c's entries (r, v) of v * X[r][j], for 128 < k a multiple of four: a
// wavefront takes tiles of 64 consecutive columns: one coalesced load brings the tile's column
// pointers into lanes, then the wavefront walks the columns (pointers read across lanes), lanes along
// j (4 per lane, 16-byte X loads), and streams each Y row out with one 16-byte store per lane (empty
// columns store zeros).  Bound by writing Y: 2 097 152 voxels x 256 vectors (2.15 GB) take 0.52 ms,
// 4.1 TB/s.
template <int VT>
__global__ __launch_bounds__(256) void spmm_wide_kernel(uint64_t C, const uint64_t* __restrict__ colptr,
                                                        const uint32_t* __restrict__ crow,
                                                        const void* __restrict__ cval,
                                                        const float* __restrict__ scale, const float* __restrict__ X,
                                                        int k, float* __restrict__ Y) {
    const int lane = threadIdx.x & 63;
    const uint64_t waves = ((uint64_t)gridDim.x * blockDim.x) >> 6;
    const uint64_t tiles = (C + 63) / 64;
    for (uint64_t tile = ((uint64_t)blockIdx.x * blockDim.x + threadIdx.x) >> 6; tile < tiles; tile += waves) {
        const uint64_t c0 = tile * 64;
        const uint64_t cl = c0 + lane < C ? c0 + lane : C;
        const uint64_t lo = colptr[cl];
        const uint64_t hi = colptr[cl + 1 <= C ? cl + 1 : C];
        const int ncol = (int)(C - c0 < 64 ? C - c0 : 64);
        for (int jc = 0; jc < ncol; jc++) {
            const uint64_t c = c0 + jc;
            const uint64_t a = lane_u64(lo, jc), e_end = lane_u64(hi, jc);
            for (int j0 = 0; j0 < k; j0 += 256) {
                const int j = j0 + 4 * lane;
                if (j >= k) continue;
                float4 acc = make_float4(0.0f, 0.0f, 0.0f, 0.0f);
                for (uint64_t e = a; e < e_end; e++) {
                    const uint32_t r = crow[e];
                    const float v = entry_value<VT>(cval, e, scale, r);
                    const float4 x = *(const float4*)(X + (uint64_t)r * k + j);
                    acc.x = fmaf(v, x.x, acc.x);
                    acc.y = fmaf(v, x.y, acc.y);
                    acc.z = fmaf(v, x.z, acc.z);
                    acc.w = fmaf(v, x.w, acc.w);
                }
                const v4f o = {acc.x, acc.y, acc.z, acc.w};
                __builtin_nontemporal_store(o, (v4f*)(Y + c * (uint64_t)k + j));
            }
        }
    }
}

// The same for fewer vectors, and for k not a multiple of four: a wavefront's 64 lanes are S columns
// x E entries x G groups of V consecutive vectors (V = 4 where k is a multiple of four, else 1; G the
// power of two that covers k / V, 64 at most), so a few vectors do not leave the other lanes idle.  E
// follows the tile's mean column length: one lane per entry stream in sparse parts of the volume
// (neighbouring columns are neighbouring lanes), all lanes on one column inside the target.  Each
// lane sums every E-th entry in order and the E partial sums meet in a fixed tree, so results are
// bitwise reproducible.  A workgroup takes 256 columns, one tile of 64 per wavefront; a tile with many
// entries is split over the four wavefronts (the longest tile would otherwise outlast the rest).
// One BF16 vector product over 49 M entries (6.4 M voxels, 2 660 rows) takes 0.17 ms where one column
// per wavefront with lanes along k took 5.4 ms; reading the entries and column pointers (350 MB) is
// 0.07 ms of it, the rest the data path of vector memory (79 % busy with SCALED, 92 % with FP32 values, 55 and
// 85 M L1 accesses: short runs of entries, and the gathers of scales and x).  Limits of E
// and kSplitEntries: a factor of two either way costs 5-10 %.
// SCALED (16-bit values, one vector): the workgroup holds scale times x of all rows in LDS, one gather
// instead of two, and takes kScaledGroups times 256 columns to be worth it (which is not so everywhere,
// worth_scaling): 0.17 -> 0.15 ms (512 columns the same, 2048 0.17).  With FP32 values, which have no scale, x in LDS takes 10 % longer, and with
// four vectors the table's size costs what it saves.  Its length: 16 KiB leave eight workgroups to a CU.
// Where scale times x is not finite (the row's other entries times x may be), the product is taken entry by
// entry as without the table.
// M (k above 64, no multiple of four): a lane takes M vectors 64 apart, so a column's entries are read once
// for 128 or 256 vectors.  Such rows of Y are no whole lines, and streamed out in parts they cost more than
// the entries where columns are short: tiles without entries are written as one run of zeros, tiles with
// few entries through L2, which merges the lines' parts; the others are streamed (through L2 they take 5-10 %
// longer, the entries and X no longer stay there).  129 vectors, FP32: 262 144 columns with 32 000 entries
// 79 us with four words per lane and a column per wavefront, 96 with a pass per 64 vectors, 59 so;
// 2 097 152 columns with 65 000 entries 434, 543, 218; 128^3 voxels with 256 pencil rows 1087, 741, 384.
constexpr uint32_t kSplitEntries = 1024;  // entries of a 64-column tile that is worth splitting
constexpr uint64_t kScaledRows = 4096, kScaledGroups = 4;
constexpr uint32_t kMergeEntries = 128;  // of a 64-column tile: below, its rows go through L2 (M > 1)

template <int VT, int V, int G, bool SCALED = false, int M = 1>
__global__ __launch_bounds__(256) void spmm_narrow_kernel(uint64_t C, const uint64_t* __restrict__ colptr,
                                                          const uint32_t* __restrict__ crow,
                                                          const void* __restrict__ cval,
                                                          const float* __restrict__ scale,
                                                          const float* __restrict__ X, int k, uint64_t R,
                                                          float* __restrict__ Y) {
    typedef float vec __attribute__((ext_vector_type(V)));
    static_assert(!SCALED || (V == 1 && G == 1 && VT != FD_VAL_F32), "one vector, 16-bit values");
    static_assert(M == 1 || (V == 1 && G == 64), "several parts of a row");
    extern __shared__ float s_scaled[];  // SCALED: scale[r] X[r]
    constexpr int N = 64 / G;  // entry lanes of a wavefront
    constexpr int kUnroll = 4;
    __shared__ uint64_t s_ptr[257];
    const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int j = lane % G, slot = lane / G;
    const uint64_t groups = (C + 255) / 256;
    auto product = [&](auto scaled) {
        constexpr bool kScaled = decltype(scaled)::value;
        for (uint64_t grp = blockIdx.x; grp < groups; grp += gridDim.x) {
            const uint64_t c0 = grp * 256;
            const int ncol = (int)(C - c0 < 256 ? C - c0 : 256);
            __syncthreads();
            s_ptr[tid] = colptr[tid < ncol ? c0 + tid : C];
            if (tid == 0) s_ptr[256] = colptr[ncol == 256 ? c0 + 256 : C];
            __syncthreads();
            for (int t = 0; t < 4; t++) {
                const uint64_t n64 = s_ptr[64 * t + 64] - s_ptr[64 * t];
                const uint32_t n = __builtin_amdgcn_readfirstlane((uint32_t)(n64 < 0xFFFFFFFFull ? n64 : 0xFFFFFFFFull));
                const bool split = n > kSplitEntries;
                if (!split && t != wave) continue;
                if (M > 1 && n == 0 && 64 * t + 64 <= ncol && (reinterpret_cast<uintptr_t>(Y) & 15) == 0) {
                    v4f* out = (v4f*)(Y + (c0 + 64 * (uint64_t)t) * (uint64_t)k);  // 64 rows of zeros, whole lines
                    for (int i = lane; i < 16 * k; i += 64) __builtin_nontemporal_store(v4f{}, out + i);
                    continue;
                }
                const bool merge = M > 1 && n < kMergeEntries;
                const int first = 64 * t + (split ? 16 * wave : 0);
                const int last = min(first + (split ? 16 : 64), ncol);
                const uint32_t mean = n / 64;
                const int want = mean < 12 ? 1 : (mean < 48 ? 4 : (mean < 192 ? 16 : 64));
                const int E = min(want, N), S = N / E;
                const int e0 = slot % E, s = slot / E;
                for (int cb = first; cb < last; cb += S) {
                    const bool on = cb + s < last;
                    const int cc = on ? cb + s : cb;
                    const uint64_t a = s_ptr[cc], b = on ? s_ptr[cc + 1] : a;
                    for (int j0 = 0; j0 < k; j0 += V * G * M) {
                        const int jj = j0 + V * j;
                        vec acc[M] = {};
                        if (jj < k) {
                            // kUnroll entries in flight; those past the column's end read its last entry
                            // and count as 0 x 0
                            for (uint64_t e = a + e0; e < b; e += (uint64_t)kUnroll * E) {
                                uint32_t r[kUnroll];
                                float v[kUnroll];
                                vec x[kUnroll][M];
#pragma unroll
                                for (int u = 0; u < kUnroll; u++) {
                                    const uint64_t eu = e + (uint64_t)u * E;
                                    r[u] = crow[eu < b ? eu : b - 1];
                                }
#pragma unroll
                                for (int u = 0; u < kUnroll; u++) {
                                    const uint64_t eu = e + (uint64_t)u * E;
                                    const uint64_t at = eu < b ? eu : b - 1;
                                    v[u] = kScaled ? stored_number<VT>(cval, at) : entry_value<VT>(cval, at, scale, r[u]);
#pragma unroll
                                    for (int m = 0; m < M; m++) {
                                        x[u][m] = vec{};
                                        if (m == 0 || jj + m * V * G < k)
                                            x[u][m] = kScaled ? *(const vec*)(s_scaled + r[u])
                                                              : *(const vec*)(X + (uint64_t)r[u] * k + jj + m * V * G);
                                    }
                                }
#pragma unroll
                                for (int u = 0; u < kUnroll; u++) {
                                    const bool in = e + (uint64_t)u * E < b;
#pragma unroll
                                    for (int m = 0; m < M; m++)
#pragma unroll
                                        for (int i = 0; i < V; i++)
                                            acc[m][i] = fmaf(in ? v[u] : 0.0f, in ? x[u][m][i] : 0.0f, acc[m][i]);
                                }
                            }
                        }
                        for (int o = E / 2; o > 0; o >>= 1)  // (one entry lane where M > 1)
#pragma unroll
                            for (int i = 0; i < V; i++) acc[0][i] += __shfl_xor(acc[0][i], o * G, 64);
#pragma unroll
                        for (int m = 0; m < M; m++) {
                            if (!(on && e0 == 0 && jj + m * V * G < k)) continue;
                            vec* out = (vec*)(Y + (c0 + (uint64_t)(cb + s)) * (uint64_t)k + jj + m * V * G);
                            if (merge)
                                *out = acc[m];
                            else
                                __builtin_nontemporal_store(acc[m], out);
                        }
                    }
                }
            }
        }
    };
    if constexpr (SCALED) {
        bool over = false;
        for (uint64_t r = threadIdx.x; r < R; r += blockDim.x) {
            const float sx = scale[r] * X[r];
            over |= !(fabsf(sx) <= FLT_MAX);
            s_scaled[r] = sx;
        }
        if (__syncthreads_or(over))
            product(std::false_type{});
        else
            product(std::true_type{});
    } else {
        product(std::false_type{});
    }
}

unsigned blocks_for(uint64_t threads, unsigned cap = 1u << 20) {
    const uint64_t b = (threads + 255) / 256;
    return (unsigned)(b < cap ? (b ? b : 1) : cap);
}

}  // namespace

hipError_t launch_global_rows(int n_mat, const uint64_t* row_first, const uint64_t* off_off, const uint64_t* nnz_off,
                              const uint64_t* offsets, uint64_t R, uint64_t total_nnz, uint64_t* rowptr,
                              hipStream_t stream) {
    hipLaunchKernelGGL(global_rows_kernel, dim3(blocks_for(R + 1, 0xFFFFFFFFu)), dim3(256), 0, stream, n_mat,
                       row_first, off_off, nnz_off, offsets, R, total_nnz, rowptr);
    return hipGetLastError();
}

hipError_t launch_pack_rows(uint64_t R, const uint64_t* rowptr, const float* values, int vtype, float* scale,
                            uint16_t* q, hipStream_t stream) {
    if (R == 0) return hipSuccess;
    hipLaunchKernelGGL(pack_rows_kernel, dim3(blocks_for(R * 64, 0xFFFFFFFFu)), dim3(256), 0, stream, R, rowptr,
                       values, vtype, scale, q);
    return hipGetLastError();
}

uint32_t csc_tile_cols(uint64_t R, uint64_t C, bool narrow) {
    return narrow && C < kNarrowBelow && C <= kNarrowRow * R ? kNarrowTile : kTileCols;
}
uint64_t csc_tiles(uint64_t C, uint32_t tile_cols) { return (C + tile_cols - 1) / tile_cols; }
uint64_t csc_tile_groups(uint64_t C, uint32_t tile_cols) {
    return (csc_tiles(C, tile_cols) + kTileGroup - 1) / kTileGroup;
}

hipError_t launch_row_tiles(uint64_t R, const uint64_t* rowptr, const uint64_t* columns, const float* values,
                            uint64_t C, uint32_t tile_cols, uint32_t* tiles, float* scale, uint32_t* unsorted,
                            hipStream_t stream) {
    if (R == 0) return hipSuccess;
    hipLaunchKernelGGL(row_tiles_kernel, dim3((unsigned)R), dim3(256), 0, stream, rowptr, columns, values, C,
                       (uint32_t)__builtin_ctz(tile_cols), (uint32_t)csc_tiles(C, tile_cols), tiles, scale, unsorted);
    return hipGetLastError();
}

hipError_t launch_tile_totals(uint64_t R, uint64_t C, uint32_t tile_cols, const uint32_t* tiles, uint32_t* total, hipStream_t stream) {
    if (R == 0 || C == 0) return hipSuccess;
    const uint32_t n_tiles = (uint32_t)csc_tiles(C, tile_cols);
    hipLaunchKernelGGL(tile_totals_kernel, dim3((n_tiles + 255) / 256, (unsigned)((R + kTotalRows - 1) / kTotalRows)),
                       dim3(256), 0, stream, R, n_tiles, tiles, total);
    return hipGetLastError();
}

hipError_t launch_place_tiles(int vtype, uint64_t R, uint64_t C, uint32_t tile_cols, const uint32_t* tiles, const uint64_t* rowptr,
                              const uint64_t* columns, const float* values, const float* scale,
                              const uint64_t* tile_base, uint32_t* order, uint64_t* colptr, uint32_t* crow,
                              void* cval, hipStream_t stream) {
    if (C == 0) return hipSuccess;
    const uint32_t n_tiles = (uint32_t)csc_tiles(C, tile_cols);
    const uint32_t n_groups = (uint32_t)csc_tile_groups(C, tile_cols);
    hipLaunchKernelGGL(tile_order_kernel, dim3(1), dim3(1024), 0, stream, n_tiles, tile_base, order);
    const dim3 g((n_groups + kXcd - 1) / kXcd * kXcd * kTileGroup), b(kPlaceThreads);
    const bool narrow = tile_cols == kNarrowTile;
    const auto kernel =
        vtype == FD_VAL_F32
            ? (narrow ? place_tile_kernel<FD_VAL_F32, kNarrowTile> : place_tile_kernel<FD_VAL_F32, kTileCols>)
        : vtype == FD_VAL_BF16
            ? (narrow ? place_tile_kernel<FD_VAL_BF16, kNarrowTile> : place_tile_kernel<FD_VAL_BF16, kTileCols>)
            : (narrow ? place_tile_kernel<FD_VAL_FP16, kNarrowTile> : place_tile_kernel<FD_VAL_FP16, kTileCols>);
    hipLaunchKernelGGL(kernel, g, b, 0, stream, R, C, n_tiles, tiles, rowptr, columns, values, scale, tile_base, order,
                       colptr, crow, cval);
    return hipGetLastError();
}

hipError_t launch_col_count(uint64_t nnz, const uint64_t* columns, uint32_t* count, hipStream_t stream) {
    if (nnz == 0) return hipSuccess;
    hipLaunchKernelGGL(col_count_kernel, dim3(blocks_for(nnz, 65536)), dim3(256), 0, stream, nnz, columns, count);
    return hipGetLastError();
}

hipError_t launch_col_scatter(uint64_t R, const uint64_t* rowptr, const uint64_t* columns, const void* vals,
                              int vbytes, const uint64_t* colptr, uint32_t* cursor, uint32_t* crow, void* cval,
                              hipStream_t stream) {
    if (R == 0) return hipSuccess;
    const dim3 g(blocks_for(R * 64, 0xFFFFFFFFu)), b(256);
    if (vbytes == 4)
        hipLaunchKernelGGL(col_scatter_kernel<float>, g, b, 0, stream, R, rowptr, columns, (const float*)vals, colptr,
                           cursor, crow, (float*)cval);
    else
        hipLaunchKernelGGL(col_scatter_kernel<uint16_t>, g, b, 0, stream, R, rowptr, columns, (const uint16_t*)vals,
                           colptr, cursor, crow, (uint16_t*)cval);
    return hipGetLastError();
}

hipError_t launch_col_sort(uint64_t C, const uint64_t* colptr, uint32_t* crow, void* cval, int vbytes,
                           hipStream_t stream) {
    if (C == 0) return hipSuccess;
    const dim3 g(blocks_for(C, 0xFFFFFFFFu)), b(256);
    if (vbytes == 4)
        hipLaunchKernelGGL(col_sort_kernel<float>, g, b, 0, stream, C, colptr, crow, (float*)cval);
    else
        hipLaunchKernelGGL(col_sort_kernel<uint16_t>, g, b, 0, stream, C, colptr, crow, (uint16_t*)cval);
    return hipGetLastError();
}

namespace {

// Whether one vector goes through the table of scales times x: it has to fit, there have to be entries to
// gather for (three for two columns; without, 256 rows on 128^3 voxels take 19.6 us with it and 18.8 without,
// 400 rows 26 and 29), and either two workgroups to a CU hide each other's tables or each has many entries
// for a row of its table (250 000 columns: 400 pencil rows 17 us with it and 19 without, 4000 rows of 300
// scattered entries 11 and 8).  Below 2^17 columns most CUs would idle: 4096 rows on 24^3 voxels 56 and 20.
bool worth_scaling(uint64_t C, uint64_t R, uint64_t nnz) {
    if (R > kScaledRows || nnz < C + C / 2) return false;
    return C >= (1ull << 19) || (C >= (1ull << 17) && nnz / R >= C / 128);
}

template <int VT, int V>
void launch_narrow(int G, const dim3& g, const dim3& b, hipStream_t stream, uint64_t C, const uint64_t* colptr,
                   const uint32_t* crow, const void* cval, const float* scale, const float* X, int k, uint64_t R,
                   uint64_t nnz, float* Y) {
    if constexpr (VT != FD_VAL_F32 && V == 1)
        if (G == 1 && worth_scaling(C, R, nnz)) {
            const dim3 few(blocks_for((C + kScaledGroups - 1) / kScaledGroups, 65536));
            hipLaunchKernelGGL((spmm_narrow_kernel<VT, 1, 1, true>), few, b, R * sizeof(float), stream, C, colptr, crow,
                               cval, scale, X, k, R, Y);
            return;
        }
    if constexpr (V == 1)
        if (k > 64) {
            const auto kernel =
                k > 128 ? spmm_narrow_kernel<VT, 1, 64, false, 4> : spmm_narrow_kernel<VT, 1, 64, false, 2>;
            hipLaunchKernelGGL(kernel, g, b, 0, stream, C, colptr, crow, cval, scale, X, k, R, Y);
            return;
        }
    switch (G) {
#define FD_NARROW(g_)                                                                                             \
    case g_:                                                                                                      \
        hipLaunchKernelGGL((spmm_narrow_kernel<VT, V, g_>), g, b, 0, stream, C, colptr, crow, cval, scale, X, k, \
                           R, Y);                                                                              \
        break
        FD_NARROW(1);
        FD_NARROW(2);
        FD_NARROW(4);
        FD_NARROW(8);
        FD_NARROW(16);
        FD_NARROW(32);
        default:
            FD_NARROW(64);
#undef FD_NARROW
    }
}

template <int VT>
hipError_t launch_spmm_typed(uint64_t C, const uint64_t* colptr, const uint32_t* crow, const void* cval,
                             const float* scale, const float* X, int k, uint64_t R, uint64_t nnz, float* Y, hipStream_t stream) {
    const dim3 b(256);
    // beyond 128 vectors a column's lanes are all along them and its entries are wave-uniform
    if (k % 4 == 0 && k > 128) {
        const dim3 g(blocks_for((C + 63) / 64 * 64, 4096));
        hipLaunchKernelGGL(spmm_wide_kernel<VT>, g, b, 0, stream, C, colptr, crow, cval, scale, X, k, Y);
        return hipGetLastError();
    }
    const dim3 g(blocks_for(C, 65536));
    const int V = k % 4 == 0 ? 4 : 1;
    int G = 1;
    while (G < 64 && G * V < k) G *= 2;
    if (V == 4)
        launch_narrow<VT, 4>(G, g, b, stream, C, colptr, crow, cval, scale, X, k, R, nnz, Y);
    else
        launch_narrow<VT, 1>(G, g, b, stream, C, colptr, crow, cval, scale, X, k, R, nnz, Y);
    return hipGetLastError();
}

}  // namespace

hipError_t launch_spmm(int vtype, uint64_t C, const uint64_t* colptr, const uint32_t* crow, const void* cval,
                       const float* scale, const float* X, int k, uint64_t R, uint64_t nnz, float* Y, hipStream_t stream) {
    if (C == 0 || k <= 0) return hipSuccess;
    if (vtype == FD_VAL_F32) return launch_spmm_typed<FD_VAL_F32>(C, colptr, crow, cval, scale, X, k, R, nnz, Y, stream);
    if (vtype == FD_VAL_BF16) return launch_spmm_typed<FD_VAL_BF16>(C, colptr, crow, cval, scale, X, k, R, nnz, Y, stream);
    return launch_spmm_typed<FD_VAL_FP16>(C, colptr, crow, cval, scale, X, k, R, nnz, Y, stream);
}

}  // namespace fdi
