// kernels_flags.hip -- beamlet / PTV intersection flags on the device (gfx950).
//
// d_beamletFlagInit (IMRTOpt/src/IMRTBeamBundle.cu:130-316): a beamlet of a bundle is active if
// any of its 3 x 3 lateral sample rays, at any of the central beam's long_dim depths, lands where
// the linearly filtered PTV mask is positive.  One wavefront per (beamlet, bundle): each lane keeps one
// of the nine rays and takes every seventh depth, and the wavefront stops after the seven depths with a
// hit (the flag is an OR, so neither order nor early exit changes it).  The point arithmetic is the host
// code's FP32 sequence (explicit fmaf, IEEE division, no contraction), so flags are bit-identical
// to fd_beamlet_flags_host.
//
// A plan's target fills a small part of the volume and most candidate beamlets miss it, which took the
// walk of every point with its eight texel reads.  A first kernel finds the mask's bounding box
// (reading the mask once; calls of a few beamlets take the volume for it, kBoxPoints); a beamlet then walks only the depths at which one of its nine rays can be
// inside it, and a point reads texels only if its base texel is.  What is left is the arithmetic of the
// points in the box around the target, so a lane computes its ray once and divides by multiplying with
// the reciprocal and correcting (Divisor).  180 beams of 400 beamlets on 200 x 200 x 160: 1.35 ms for
// every point, 0.13 ms for those in the box, 0.065 ms with the texels of a point read at once (serial
// reads with a branch each before: the loops took as many scalar instructions as vector ones).
#include <algorithm>
#include <hip/hip_runtime.h>

#include "kernels.h"

namespace fdi {
namespace {

constexpr int kFlagSS = 3;

// Bounding box of the mask's n nonzero texels: box[0..2] the smallest x, y, z, box[3..5] the bitwise
// complements of the largest (so that every entry is a minimum; ~0 in all of them, as before the call: an
// empty mask).  n < 2^31: its divisions take 32 bits.  Bound by reading the mask: 105 M texels, a quarter
// of them set, take 21 us of a call, and took 157 with every set texel's coordinates and an atomic per
// workgroup and word.
constexpr int kBoxThreads = 512;
constexpr uint64_t kBoxBlocks = 512;
__global__ __launch_bounds__(kBoxThreads) void mask_box_kernel(const uint8_t* __restrict__ mask, uint32_t X, uint32_t Y,
                                                               uint32_t n, uint32_t* __restrict__ box) {
    uint32_t lo[6] = {~0u, ~0u, ~0u, ~0u, ~0u, ~0u};
    // texels [i, j] of row r, both ends set
    auto add = [&](uint32_t r, uint32_t i, uint32_t j) {
        const uint32_t x0 = r * X, z = r / Y, y = r - z * Y;
        const uint32_t v[6] = {i - x0, y, z, ~(j - x0), ~y, ~z};
        for (int d = 0; d < 6; d++) lo[d] = min(lo[d], v[d]);
    };
    const uint32_t id = blockIdx.x * kBoxThreads + threadIdx.x, all = gridDim.x * kBoxThreads;
    // 16 texels at a time where the mask is aligned, single ones before and after
    const uint32_t head = min((uint32_t)(-(uintptr_t)mask & 15), n), quads = (n - head) / 16;
    for (uint32_t i = id; i < head; i += all)
        if (mask[i]) add(i / X, i, i);
    for (uint32_t q = id; q < quads; q += all) {
        const uint4 v = reinterpret_cast<const uint4*>(mask + head)[q];
        const uint64_t w[2] = {v.x | (uint64_t)v.y << 32, v.z | (uint64_t)v.w << 32};
        if ((w[0] | w[1]) == 0u) continue;
        // the first and the last of them bound the rest, unless the row ends in between
        const uint32_t at = head + 16 * q;
        const uint32_t i = at + (w[0] ? __builtin_ctzll(w[0]) >> 3 : 8 + (__builtin_ctzll(w[1]) >> 3));
        const uint32_t j = at + (w[1] ? 15 - (__builtin_clzll(w[1]) >> 3) : 7 - (__builtin_clzll(w[0]) >> 3));
        const uint32_t r = i / X;
        if (j - r * X < X) {
            add(r, i, j);
            continue;
        }
        for (int k = 0; k < 16; k++)
            if ((w[k >> 3] >> (8 * (k & 7))) & 255u) add((at + k) / X, at + k, at + k);
    }
    for (uint32_t i = head + 16 * quads + id; i < n; i += all)
        if (mask[i]) add(i / X, i, i);
    __shared__ uint32_t s_lo[6];
    if (threadIdx.x < 6) s_lo[threadIdx.x] = ~0u;
    __syncthreads();
    for (int d = 0; d < 6; d++) {
        for (int o = 32; o > 0; o >>= 1) lo[d] = min(lo[d], (uint32_t)__shfl_xor((int)lo[d], o, 64));
        if ((threadIdx.x & 63) == 0 && lo[d] != ~0u) atomicMin(&s_lo[d], lo[d]);
    }
    __syncthreads();
    // one line of six words: a workgroup that lowers none of them any more leaves it alone
    if (threadIdx.x < 6 && s_lo[threadIdx.x] < __hip_atomic_load(&box[threadIdx.x], __ATOMIC_RELAXED,
                                                                 __HIP_MEMORY_SCOPE_AGENT))
        atomicMin(&box[threadIdx.x], s_lo[threadIdx.x]);
}

// x / v as the IEEE division rounds it, in three instructions: with r = 1 / v rounded, x r corrected by
// its exact remainder times r is the rounded quotient (Markstein's theorem) unless v's significand is
// all ones or a step leaves the normal range; such divisors are divided by.  (Quotients out of range,
// infinities and NaN fail the box test either way; quotients below 2^-60 or so are rounded away by the
// half texel subtracted from them.)
struct Divisor {
    float v, r;
    bool plain;
    __device__ __forceinline__ explicit Divisor(float d) : v(d), r(1.0f / d) {
        plain = (__float_as_uint(d) & 0x7FFFFFu) != 0x7FFFFFu && d > 0x1p-40f && d < 0x1p40f;
    }
    __device__ __forceinline__ float of(float x) const {
        if (!plain) return x / v;
        const float q = x * r;
        return fmaf(fmaf(-q, v, x), r, q);
    }
};

// The box as signed texel bounds [lo, hi] (lo > hi when empty); without one, the whole volume.
struct MaskBox {
    int lo[3], hi[3];
};
__device__ __forceinline__ MaskBox read_box(const uint32_t* __restrict__ box, int X, int Y, int Z) {
    MaskBox b{{0, 0, 0}, {X - 1, Y - 1, Z - 1}};
    if (!box) return b;
    for (int d = 0; d < 3; d++) {
        const bool any = box[d] != ~0u;
        b.lo[d] = any ? (int)box[d] : 1;
        b.hi[d] = any ? (int)~box[3 + d] : 0;
    }
    return b;
}

// Linear-filtered binary mask > 0 at unnormalised texture coordinates (texel i spans [i, i+1),
// border 0): true iff a texel with nonzero weight is set.  The up to eight texels are read as four pairs
// along x, all in flight, at coordinates moved into the volume; what was moved or has no weight is
// masked off.
__device__ bool mask_hit_dev(const uint8_t* __restrict__ mask, int X, int Y, int Z, const MaskBox& box, float cx,
                             float cy, float cz) {
    const float t[3] = {cx - 0.5f, cy - 0.5f, cz - 0.5f};
    int base[3];
    bool two[3];  // the texel after the base texel has weight
#pragma unroll
    for (int d = 0; d < 3; d++) {
        const float f = floorf(t[d]);
        // texels base and base + 1 at most: one of them lies in the box
        if (!(f >= (float)(box.lo[d] - 1) && f <= (float)box.hi[d])) return false;
        base[d] = (int)f;
        two[d] = (t[d] - f) > 0.0f;
    }
    const int x = base[0];
    // the pair's bytes: texels x and x + 1, or the volume's first or last two where x is -1 or X - 1
    const int at = min(max(x, 0), max(X - 2, 0));
    uint32_t low = 0, high = 0;
#pragma unroll
    for (int k = 0; k < 4; k++) {
        const int y = base[1] + (k & 1), z = base[2] + (k >> 1);
        const bool row = y >= 0 && y < Y && z >= 0 && z < Z && (!(k & 1) || two[1]) && (!(k >> 1) || two[2]);
        const size_t o = (size_t)at + (size_t)X * ((size_t)min(max(y, 0), Y - 1) + (size_t)Y * min(max(z, 0), Z - 1));
        uint32_t w;
        if (X >= 2) {
            uint16_t pair;
            __builtin_memcpy(&pair, mask + o, 2);
            w = pair;
        } else {
            w = mask[o];
        }
        w = row ? w : 0u;
        low |= w & 255u;
        high |= w >> 8;
    }
    const uint32_t first = x < 0 ? 0u : (x > at ? high : low);
    const uint32_t second = x < 0 ? low : (x == at ? high : 0u);  // x = X - 1: none
    return first != 0u || (two[0] && second != 0u);
}

// BEV -> PVCS direction of sample ray r (j, k) of beamlet (bx, by), the host's FP32 sequence.
__device__ __forceinline__ void sample_ray(const FlagBeamDev& d, int bx, int by, int r, float p[3]) {
    const int j = r / kFlagSS, k = r - j * kFlagSS;
    const float dx = ((float)bx + (j + 0.5f) / (float)kFlagSS - (float)d.fx * 0.5f) * d.bs[0];
    const float dy = d.sad;
    const float dz = ((float)by + (k + 0.5f) / (float)kFlagSS - (float)d.fy * 0.5f) * d.bs[1];
    p[0] = fmaf(d.Ri[2], dz, fmaf(d.Ri[1], dy, d.Ri[0] * dx));
    p[1] = fmaf(d.Ri[5], dz, fmaf(d.Ri[4], dy, d.Ri[3] * dx));
    p[2] = fmaf(d.Ri[8], dz, fmaf(d.Ri[7], dy, d.Ri[6] * dx));
}

// 1 / x to about 1e-14 (the hardware's FP64 reciprocal and one Newton step).
__device__ __forceinline__ double reciprocal(double x) {
    const double r = __builtin_amdgcn_rcp(x);
    return fma(fma(-x, r, 1.0), r, r);
}

// Depth indices [i0, i1) of the ray with direction p at which a point (src + p depth / sad) / v can have
// its base texel within [lo - 1, hi] of the box: the ray's interval in FP64, widened by 0.05 texel plus
// 1e-5 of the coordinates' magnitude (the FP32 points are within a few 1e-7 of it) and by one index
// either way.  All depths for values too large to bound so.  Most beamlets end here, so there is one
// reciprocal per axis and no branch on the direction's sign (with divisions and branches the kernel took
// 2 % longer; FP64 multiply-adds run at the rate of FP32 ones).
__device__ __forceinline__ void ray_depths(const FlagBeamDev& d, const MaskBox& box, const float p[3],
                                           const float v[3], int& i0, int& i1) {
    double lo = 0.0, hi = 1e30;  // scale = depth / sad
    const double far_scale = fma((double)d.L, (double)d.ls, (double)d.lim_min) * reciprocal(d.sad);
    bool odd = !(far_scale < 1e9 && far_scale > 0.0 && d.ls > 0.0f);
#pragma unroll
    for (int a = 0; a < 3; a++) {
        const double s = d.src[a], q = p[a], u = v[a];
        odd |= !(fabs(s) < 1e9 && fabs(q) < 1e9 && u > 1e-9);
        const double m = u * 0.05 + 1e-5 * (fabs(s) + fabs(q) * far_scale);
        // base texel in [lo - 1, hi]: coordinate / v in [lo - 0.5, hi + 1.5)
        const double x0 = (box.lo[a] - 0.5) * u - m - s, x1 = (box.hi[a] + 1.5) * u + m - s;
        // a direction component below 1e-20 moves by less than the margin over the whole depth
        const bool still = fabs(q) < 1e-20;
        const double r = reciprocal(still ? 1.0 : q), t0 = x0 * r, t1 = x1 * r;
        lo = still ? lo : fmax(lo, fmin(t0, t1));
        hi = still ? (x0 > 0.0 || x1 < 0.0 ? -1.0 : hi) : fmin(hi, fmax(t0, t1));
    }
    i0 = 0;
    i1 = d.L;
    if (odd) return;
    const double L = d.L, r = reciprocal(d.ls);
    const double a0 = (lo * d.sad - d.lim_min) * r - 1.0, a1 = (hi * d.sad - d.lim_min) * r + 2.0;
    if (!(lo <= hi) || a0 >= L || a1 <= 0.0) {
        i1 = 0;
        return;
    }
    i0 = (int)fmax(a0, 0.0);
    i1 = (int)ceil(fmin(a1, L));
}

constexpr int kFlagWaves = 4;  // beamlets per workgroup
// Below kBoxPoints sample points, and one more per kBoxVoxels texels of the mask, the box is not looked for:
// finding it takes 4 us and 0.15 us per million texels, which beamlets that soon hit the target do not earn
// back (16 beamlets, all hits, on 200 x 200 x 160 31 us a call without and 41 with it; 400 beamlets 32 and
// 41, but 51 and 35 with a target eight texels wide).
constexpr uint64_t kBoxPoints = 200000, kBoxVoxels = 64;

__global__ __launch_bounds__(64 * kFlagWaves) void beamlet_flags_kernel(const FlagBeamDev* __restrict__ beams,
                                                                        const uint8_t* __restrict__ mask, int X,
                                                                        int Y, int Z, float vx, float vy, float vz,
                                                                        const uint32_t* __restrict__ mask_box,
                                                                        uint8_t* __restrict__ flags) {
    const FlagBeamDev& d = beams[blockIdx.y];
    const int lane = threadIdx.x & 63;
    const int idx = blockIdx.x * kFlagWaves + __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    if (idx >= d.fx * d.fy) return;
    const int bx = idx % d.fx, by = idx / d.fx;
    const MaskBox box = read_box(mask_box, X, Y, Z);
    const float v[3] = {vx, vy, vz};
    // my ray, and the depths at which it and the wavefront's nine rays can be inside the mask's box
    constexpr int kRays = kFlagSS * kFlagSS, kDepths = 64 / kRays;
    float p[3];
    sample_ray(d, bx, by, lane % kRays, p);
    int i0 = d.L, i1 = 0;
    if (box.lo[0] <= box.hi[0]) ray_depths(d, box, p, v, i0, i1);
    int first = i0 < i1 ? i0 : d.L, last = i0 < i1 ? i1 : 0;
    for (int o = 8; o > 0; o >>= 1) {  // lanes 0 ... 15 hold the nine rays
        first = min(first, __shfl_xor(first, o, 64));
        last = max(last, __shfl_xor(last, o, 64));
    }
    first = __builtin_amdgcn_readfirstlane(first);
    last = __builtin_amdgcn_readfirstlane(last);
    if (lane >= kRays * kDepths) i1 = 0;  // the 64th lane has no depth of its own
    const Divisor by_sad(d.sad), by_vx(vx), by_vy(vy), by_vz(vz);
    bool on = false;
    for (int i = first + lane / kRays; first < last && !on; i += kDepths, first += kDepths) {
        bool hit = false;
        if (i >= i0 && i < i1) {
            const float depth = d.lim_min + (float)i * d.ls;
            const float scale = by_sad.of(depth);
            hit = mask_hit_dev(mask, X, Y, Z, box, by_vx.of(fmaf(p[0], scale, d.src[0])),
                               by_vy.of(fmaf(p[1], scale, d.src[1])), by_vz.of(fmaf(p[2], scale, d.src[2])));
        }
        on = __any(hit);
    }
    if (lane == 0) flags[d.out_off + idx] = on ? 1 : 0;
}

}  // namespace

hipError_t launch_beamlet_flags(const FlagBeamDev* beams, int n, int max_pixels, uint64_t points, const uint8_t* mask,
                                const fd_volume& vol, uint32_t* box, uint8_t* flags, hipStream_t stream) {
    if (n <= 0 || max_pixels <= 0) return hipSuccess;
    const uint64_t voxels = (uint64_t)vol.dim[0] * vol.dim[1] * vol.dim[2];
    if (points < kBoxPoints + voxels / kBoxVoxels || voxels >= (1ull << 31)) {
        box = nullptr;
    } else {
        const uint64_t blocks = std::min(voxels / (16 * kBoxThreads) + 1, kBoxBlocks);
        hipLaunchKernelGGL(mask_box_kernel, dim3((unsigned)blocks), dim3(kBoxThreads), 0, stream, mask, vol.dim[0],
                           vol.dim[1], (uint32_t)voxels, box);
        hipError_t e = hipGetLastError();
        if (e != hipSuccess) return e;
    }
    dim3 grid((unsigned)((max_pixels + kFlagWaves - 1) / kFlagWaves), (unsigned)n), block(64 * kFlagWaves);
    hipLaunchKernelGGL(beamlet_flags_kernel, grid, block, 0, stream, beams, mask, (int)vol.dim[0], (int)vol.dim[1],
                       (int)vol.dim[2], vol.voxel_size[0], vol.voxel_size[1], vol.voxel_size[2], box, flags);
    return hipGetLastError();
}

}  // namespace fdi
