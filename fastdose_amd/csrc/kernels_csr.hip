// kernels_csr.hip -- prefix scans and dense -> CSR conversion (gfx950).
//
// fd_dense_to_csr stands in for cusparseDenseToSparse in MatCSREnsemble::addMat
// (IMRTOpt/src/IMRTSparseMatEns.cu:78-161): row-major input, exact zeros dropped, ascending
// columns, 0-based 64-bit offsets.  Count pass (one wavefront per row segment) -> scan -> ordered fill
// (wavefront ballots keep the column order).
#include <algorithm>
#include <hip/hip_runtime.h>

#include "kernels.h"

namespace fdi {

namespace {

constexpr int kScanThreads = 1024;

// Exclusive scan of a value per thread of a workgroup of WAVES wavefronts, and the total.
template <int WAVES>
__device__ __forceinline__ uint64_t block_excl_scan_u64(uint64_t v, uint64_t* s_wave, uint64_t& total) {
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    uint64_t x = v;
#pragma unroll
    for (int o = 1; o < 64; o <<= 1) {
        const uint64_t y = __shfl_up(x, o, 64);
        if (lane >= o) x += y;
    }
    if (lane == 63) s_wave[wave] = x;
    __syncthreads();
    uint64_t before = 0;
    total = 0;
#pragma unroll
    for (int w = 0; w < WAVES; w++) {  // independent reads, unlike one thread's running sum
        const uint64_t t = s_wave[w];
        before += w < wave ? t : 0;
        total += t;
    }
    __syncthreads();
    return before + x - v;
}

// Thread's kScanItems consecutive elements from `at` on, and their exclusive sums from run on
constexpr int kScanItems = 16;
__device__ __forceinline__ uint64_t load_items(const uint32_t* __restrict__ count, uint64_t at, uint64_t N,
                                               uint32_t (&c)[kScanItems]) {
    uint64_t sum = 0;
    if (at + kScanItems <= N && (reinterpret_cast<uintptr_t>(count) & 15) == 0) {  // at is a multiple of 16
#pragma unroll
        for (int i = 0; i < kScanItems / 4; i++) {
            const uint4 q = reinterpret_cast<const uint4*>(count + at)[i];
            c[4 * i] = q.x;
            c[4 * i + 1] = q.y;
            c[4 * i + 2] = q.z;
            c[4 * i + 3] = q.w;
        }
    } else {
#pragma unroll
        for (int i = 0; i < kScanItems; i++) c[i] = at + i < N ? count[at + i] : 0u;
    }
#pragma unroll
    for (int i = 0; i < kScanItems; i++) sum += c[i];
    return sum;
}
__device__ __forceinline__ void store_items(uint64_t* __restrict__ off, uint64_t at, uint64_t N, uint64_t run,
                                            const uint32_t (&c)[kScanItems]) {
    if (at + kScanItems <= N && (reinterpret_cast<uintptr_t>(off) & 15) == 0) {
#pragma unroll
        for (int i = 0; i < kScanItems / 2; i++) {
            const uint64_t second = run + c[2 * i];
            reinterpret_cast<ulonglong2*>(off + at)[i] = make_ulonglong2(run, second);
            run = second + c[2 * i + 1];
        }
    } else {
#pragma unroll
        for (int i = 0; i < kScanItems; i++) {
            if (at + i < N) off[at + i] = run;
            run += c[i];
        }
    }
}

// Exclusive scan by one workgroup, kScanPass elements at a time.
constexpr uint64_t kScanPass = (uint64_t)kScanThreads * kScanItems;
__global__ __launch_bounds__(kScanThreads) void scan_u32_kernel(const uint32_t* __restrict__ count, uint64_t N,
                                                                uint64_t* __restrict__ off,
                                                                uint64_t* __restrict__ total) {
    __shared__ uint64_t s_wave[kScanThreads / 64];
    uint64_t carry = 0;
    for (uint64_t base = 0; base < N; base += kScanPass) {
        const uint64_t at = base + (uint64_t)threadIdx.x * kScanItems;
        uint32_t c[kScanItems];
        uint64_t sum;
        const uint64_t run = block_excl_scan_u64<kScanThreads / 64>(load_items(count, at, N, c), s_wave, sum);
        store_items(off, at, N, carry + run, c);
        carry += sum;
    }
    if (threadIdx.x == 0) total[0] = carry;
}

// Larger inputs in two kernels: the sums of tiles of 4096 elements, then every tile's scan from the sum
// of the tiles before it, which its workgroup adds up itself (up to kScanTiles of them; beyond, a third
// kernel scans the tile sums in between).
constexpr int kTileThreads = 256;
constexpr uint64_t kTile = (uint64_t)kTileThreads * kScanItems;
static_assert(kTile == kScanTile, "the scratch holds a sum per tile");
constexpr uint64_t kScanTiles = 4096;

__global__ __launch_bounds__(kTileThreads) void scan_tile_sums_kernel(const uint32_t* __restrict__ count, uint64_t N,
                                                                      uint64_t* __restrict__ sums) {
    __shared__ uint64_t s_wave[kTileThreads / 64];
    const uint64_t at = (uint64_t)blockIdx.x * kTile + (uint64_t)threadIdx.x * kScanItems;
    uint32_t c[kScanItems];
    uint64_t total;
    block_excl_scan_u64<kTileThreads / 64>(load_items(count, at, N, c), s_wave, total);
    if (threadIdx.x == 0) sums[blockIdx.x] = total;
}

// exclusive scan of the tile sums in place (one workgroup), grand total to total[0]
__global__ __launch_bounds__(1024) void scan_sums_kernel(uint64_t* __restrict__ sums, uint64_t nb,
                                                         uint64_t* __restrict__ total) {
    __shared__ uint64_t s_wave[1024 / 64];
    uint64_t carry = 0;
    for (uint64_t i0 = 0; i0 < nb; i0 += blockDim.x) {
        const uint64_t i = i0 + threadIdx.x;
        const uint64_t v = i < nb ? sums[i] : 0;
        uint64_t tot;
        const uint64_t ex = block_excl_scan_u64<1024 / 64>(v, s_wave, tot);
        if (i < nb) sums[i] = carry + ex;
        carry += tot;
    }
    if (threadIdx.x == 0) total[0] = carry;
}

// SCANNED: sums holds exclusive sums (and total is written already)
template <bool SCANNED>
__global__ __launch_bounds__(kTileThreads) void scan_tiles_kernel(const uint32_t* __restrict__ count, uint64_t N,
                                                                  const uint64_t* __restrict__ sums,
                                                                  uint64_t* __restrict__ off,
                                                                  uint64_t* __restrict__ total) {
    __shared__ uint64_t s_wave[kTileThreads / 64];
    const uint64_t at = (uint64_t)blockIdx.x * kTile + (uint64_t)threadIdx.x * kScanItems;
    uint32_t c[kScanItems];
    const uint64_t v = load_items(count, at, N, c);
    uint64_t before = 0, sum;
    if (SCANNED) {
        before = sums[blockIdx.x];
    } else {
        uint64_t mine = 0;
        for (uint32_t b = threadIdx.x; b < blockIdx.x; b += kTileThreads) mine += sums[b];
        block_excl_scan_u64<kTileThreads / 64>(mine, s_wave, before);
    }
    const uint64_t run = before + block_excl_scan_u64<kTileThreads / 64>(v, s_wave, sum);
    store_items(off, at, N, run, c);
    if (!SCANNED && blockIdx.x == gridDim.x - 1 && threadIdx.x == 0) total[0] = before + sum;
}

// Dense -> CSR works on segments: runs of consecutive elements of one row, one wavefront each.  A beam's
// dense rows are few and long (64 rows of 262 144 voxels), so a workgroup per row left three CUs of
// four idle and a serial loop in the others.  A segment needs no LDS and no barrier: lanes take
// consecutive elements, kDenseBatch loads in flight, and a ballot gives each nonzero its place.
// HBM-bound; at 64 x 262 144 the count goes from 0.26 to 0.015 ms and
// the fill from 0.53 to 0.013 ms (5 TB/s).
constexpr int kDenseSegment = 2048;
constexpr int kDenseBatch = 8;

// (row, first element, length) of this wavefront's segment; false beyond the last
__device__ __forceinline__ bool dense_segment(uint64_t rows, uint64_t cols, uint32_t n_seg, uint32_t seg_len,
                                              uint64_t& seg, uint64_t& row, uint64_t& first, uint32_t& len) {
    seg = (uint64_t)blockIdx.x * 4 + __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    row = seg / n_seg;
    if (row >= rows) return false;
    first = (seg - row * n_seg) * (uint64_t)seg_len;
    const uint64_t left = first < cols ? cols - first : 0;
    len = (uint32_t)(left < seg_len ? left : seg_len);
    return true;
}

__global__ __launch_bounds__(256) void dense_count_kernel(const float* __restrict__ dense, uint64_t rows,
                                                          uint64_t cols, uint32_t n_seg, uint32_t seg_len,
                                                          uint32_t* __restrict__ count) {
    uint64_t seg, row, first;
    uint32_t len;
    if (!dense_segment(rows, cols, n_seg, seg_len, seg, row, first, len)) return;
    const float* __restrict__ src = dense + row * cols + first;
    const uint32_t lane = threadIdx.x & 63;
    uint32_t c = 0;
    for (uint32_t j0 = 0; j0 < len; j0 += 64 * kDenseBatch) {
        float v[kDenseBatch];
#pragma unroll
        for (int u = 0; u < kDenseBatch; u++) {
            const uint32_t j = j0 + 64 * u + lane;
            v[u] = j < len ? src[j] : 0.0f;
        }
#pragma unroll
        for (int u = 0; u < kDenseBatch; u++) c += (uint32_t)__popcll(__ballot(v[u] != 0.0f));
    }
    if (lane == 0) count[seg] = c;
}

__global__ __launch_bounds__(256) void dense_fill_kernel(const float* __restrict__ dense, uint64_t rows,
                                                         uint64_t cols, uint32_t n_seg, uint32_t seg_len,
                                                         const uint64_t* __restrict__ seg_off,
                                                         uint64_t* __restrict__ columns,
                                                         float* __restrict__ values) {
    uint64_t seg, row, first;
    uint32_t len;
    if (!dense_segment(rows, cols, n_seg, seg_len, seg, row, first, len)) return;
    const float* __restrict__ src = dense + row * cols + first;
    const uint32_t lane = threadIdx.x & 63;
    uint64_t out = seg_off[seg];
    for (uint32_t j0 = 0; j0 < len; j0 += 64 * kDenseBatch) {
        float v[kDenseBatch];
#pragma unroll
        for (int u = 0; u < kDenseBatch; u++) {
            const uint32_t j = j0 + 64 * u + lane;
            v[u] = j < len ? src[j] : 0.0f;
        }
#pragma unroll
        for (int u = 0; u < kDenseBatch; u++) {
            const uint64_t mask = __ballot(v[u] != 0.0f);
            if (v[u] != 0.0f) {
                const uint64_t at = out + (uint32_t)__popcll(mask & ((1ull << lane) - 1ull));
                columns[at] = first + j0 + 64 * u + lane;
                values[at] = v[u];
            }
            out += (uint32_t)__popcll(mask);
        }
    }
}

__global__ void write_offsets_kernel(const uint64_t* __restrict__ seg_off, const uint64_t* __restrict__ total,
                                     uint64_t rows, uint32_t n_seg, uint64_t* __restrict__ offsets) {
    const uint64_t r = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (r < rows) offsets[r] = seg_off[r * n_seg];
    if (r == rows) offsets[rows] = total[0];
}

}  // namespace

hipError_t launch_scan_u32(const uint32_t* count, uint64_t N, uint64_t* off, uint64_t* total, uint64_t* scratch,
                           hipStream_t stream) {
    // one workgroup takes 5 us for up to a pass, and 7 for every further one; two kernels take 9
    if (N <= kScanPass) {
        hipLaunchKernelGGL(scan_u32_kernel, dim3(1), dim3(kScanThreads), 0, stream, count, N, off, total);
        return hipGetLastError();
    }
    const uint64_t nb = (N + kTile - 1) / kTile;
    hipLaunchKernelGGL(scan_tile_sums_kernel, dim3((unsigned)nb), dim3(kTileThreads), 0, stream, count, N, scratch);
    if (nb <= kScanTiles) {
        hipLaunchKernelGGL(scan_tiles_kernel<false>, dim3((unsigned)nb), dim3(kTileThreads), 0, stream, count, N,
                           scratch, off, total);
        return hipGetLastError();
    }
    hipLaunchKernelGGL(scan_sums_kernel, dim3(1), dim3(1024), 0, stream, scratch, nb, total);
    hipLaunchKernelGGL(scan_tiles_kernel<true>, dim3((unsigned)nb), dim3(kTileThreads), 0, stream, count, N, scratch,
                       off, total);
    return hipGetLastError();
}

DenseSplit dense_split(uint64_t rows, uint64_t cols, uint64_t max_segments) {
    DenseSplit s{1, kDenseSegment};
    if (rows == 0 || cols == 0) return s;
    const uint64_t want = (cols + kDenseSegment - 1) / kDenseSegment, most = std::max<uint64_t>(max_segments / rows, 1);
    s.per_row = (uint32_t)std::min(want, most);
    s.length = (uint32_t)std::max<uint64_t>((cols + s.per_row - 1) / s.per_row, kDenseSegment);
    return s;
}

hipError_t launch_dense_count(const float* dense, uint64_t rows, uint64_t cols, const DenseSplit& s, uint32_t* count,
                              hipStream_t stream) {
    if (rows == 0) return hipSuccess;
    hipLaunchKernelGGL(dense_count_kernel, dim3((unsigned)((rows * s.per_row + 3) / 4)), dim3(256), 0, stream, dense,
                       rows, cols, s.per_row, s.length, count);
    return hipGetLastError();
}

hipError_t launch_dense_fill(const float* dense, uint64_t rows, uint64_t cols, const DenseSplit& s,
                             const uint64_t* seg_off, uint64_t* columns, float* values, hipStream_t stream) {
    if (rows == 0) return hipSuccess;
    hipLaunchKernelGGL(dense_fill_kernel, dim3((unsigned)((rows * s.per_row + 3) / 4)), dim3(256), 0, stream, dense,
                       rows, cols, s.per_row, s.length, seg_off, columns, values);
    return hipGetLastError();
}

// Plain fill kernels: clearing through a kernel rather than a memset node keeps every stage
// capturable into a HIP graph.
template <typename T>
__global__ void fill_kernel(T* p, uint64_t n, T v) {
    for (uint64_t i = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x; i < n; i += (uint64_t)gridDim.x * blockDim.x)
        p[i] = v;
}

hipError_t launch_fill_u32(uint32_t* p, uint64_t n, uint32_t v, hipStream_t stream) {
    if (n == 0) return hipSuccess;
    const uint64_t blocks = std::min<uint64_t>((n + 255) / 256, 4096);
    hipLaunchKernelGGL(fill_kernel<uint32_t>, dim3((unsigned)blocks), dim3(256), 0, stream, p, n, v);
    return hipGetLastError();
}

hipError_t launch_fill_u64(uint64_t* p, uint64_t n, uint64_t v, hipStream_t stream) {
    if (n == 0) return hipSuccess;
    const uint64_t blocks = std::min<uint64_t>((n + 255) / 256, 4096);
    hipLaunchKernelGGL(fill_kernel<uint64_t>, dim3((unsigned)blocks), dim3(256), 0, stream, p, n, v);
    return hipGetLastError();
}

hipError_t launch_write_offsets(const uint64_t* seg_off, const uint64_t* total, uint64_t rows, uint32_t n_seg,
                                uint64_t* offsets, hipStream_t stream) {
    hipLaunchKernelGGL(write_offsets_kernel, dim3((unsigned)((rows + 1 + 255) / 256)), dim3(256), 0, stream,
                       seg_off, total, rows, n_seg, offsets);
    return hipGetLastError();
}

}  // namespace fdi
