// kernels_flags.hip -- beamlet / PTV intersection flags on the device (gfx950).
//
// d_beamletFlagInit (IMRTOpt/src/IMRTBeamBundle.cu:130-316): a beamlet of a bundle is active if
// any of its 3 x 3 lateral sample rays, at any of the central beam's long_dim depths, lands where
// the linearly filtered PTV mask is positive.  One wavefront per (beamlet, bundle): lanes take the
// (depth, sample) points in the host loop's order 64 at a time and stop at the first chunk with a
// hit (the flag is an OR, so the early exit does not change it).  The point arithmetic is the host
// code's FP32 sequence (explicit fmaf, IEEE division, no contraction), so flags are bit-identical
// to fd_beamlet_flags_host.
//
// A plan's target fills a small part of the volume and most candidate beamlets miss it, which took the
// walk of every point with its eight texel reads.  A first kernel finds the mask's bounding box
// (reading the mask once); a beamlet then walks only the depths at which one of its nine rays can be
// inside it, and a point reads texels only if its base texel is.  180 beams of 400 beamlets on
// 200 x 200 x 160: 1.35 -> 0.13 ms.
#include <hip/hip_runtime.h>

#include "kernels.h"

namespace fdi {
namespace {

constexpr int kFlagSS = 3;

// Bounding box of the mask's nonzero texels: box[0..2] the smallest x, y, z, box[3..5] the bitwise
// complements of the largest (so that every entry is a minimum; ~0 in all of them: an empty mask).
__global__ __launch_bounds__(256) void mask_box_kernel(const uint8_t* __restrict__ mask, uint32_t X, uint32_t Y,
                                                       uint64_t n, uint32_t* __restrict__ box) {
    uint32_t lo[6] = {~0u, ~0u, ~0u, ~0u, ~0u, ~0u};
    auto add = [&](uint64_t i) {
        const uint64_t r = i / X;
        const uint32_t c[3] = {(uint32_t)(i - r * X), (uint32_t)(r % Y), (uint32_t)(r / Y)};
        for (int d = 0; d < 3; d++) {
            lo[d] = min(lo[d], c[d]);
            lo[3 + d] = min(lo[3 + d], ~c[d]);
        }
    };
    const uint64_t id = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x, all = (uint64_t)gridDim.x * blockDim.x;
    // 16 texels at a time where the mask is aligned, single ones before and after
    const uint64_t head = min((uint64_t)(-(uintptr_t)mask & 15), n), quads = (n - head) / 16;
    for (uint64_t i = id; i < head; i += all)
        if (mask[i]) add(i);
    for (uint64_t q = id; q < quads; q += all) {
        const uint4 v = reinterpret_cast<const uint4*>(mask + head)[q];
        if ((v.x | v.y | v.z | v.w) == 0u) continue;
        const uint32_t w[4] = {v.x, v.y, v.z, v.w};
        for (int k = 0; k < 16; k++)
            if ((w[k >> 2] >> (8 * (k & 3))) & 255u) add(head + 16 * q + k);
    }
    for (uint64_t i = head + 16 * quads + id; i < n; i += all)
        if (mask[i]) add(i);
    for (int d = 0; d < 6; d++) {
        for (int o = 32; o > 0; o >>= 1) lo[d] = min(lo[d], (uint32_t)__shfl_xor((int)lo[d], o, 64));
        if ((threadIdx.x & 63) == 0 && lo[d] != ~0u) atomicMin(&box[d], lo[d]);
    }
}

// The box as signed texel bounds [lo, hi] (lo > hi when empty).
struct MaskBox {
    int lo[3], hi[3];
};
__device__ __forceinline__ MaskBox read_box(const uint32_t* __restrict__ box) {
    MaskBox b;
    for (int d = 0; d < 3; d++) {
        const bool any = box[d] != ~0u;
        b.lo[d] = any ? (int)box[d] : 1;
        b.hi[d] = any ? (int)~box[3 + d] : 0;
    }
    return b;
}

// Linear-filtered binary mask > 0 at unnormalised texture coordinates (texel i spans [i, i+1),
// border 0): true iff a texel with nonzero weight is set.
__device__ bool mask_hit_dev(const uint8_t* __restrict__ mask, int X, int Y, int Z, const MaskBox& box, float cx,
                             float cy, float cz) {
    const float t[3] = {cx - 0.5f, cy - 0.5f, cz - 0.5f};
    int base[3], reach[3];
#pragma unroll
    for (int d = 0; d < 3; d++) {
        const float f = floorf(t[d]);
        // texels base and base + 1 at most: one of them lies in the box
        if (!(f >= (float)(box.lo[d] - 1) && f <= (float)box.hi[d])) return false;
        base[d] = (int)f;
        reach[d] = (t[d] - f) > 0.0f ? 2 : 1;
    }
    for (int k = 0; k < reach[2]; k++) {
        const int z = base[2] + k;
        if (z < 0 || z >= Z) continue;
        for (int j = 0; j < reach[1]; j++) {
            const int y = base[1] + j;
            if (y < 0 || y >= Y) continue;
            for (int i = 0; i < reach[0]; i++) {
                const int x = base[0] + i;
                if (x < 0 || x >= X) continue;
                if (mask[(size_t)x + (size_t)X * ((size_t)y + (size_t)Y * z)]) return true;
            }
        }
    }
    return false;
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

// Depth indices [i0, i1) of the ray with direction p at which a point (src + p depth / sad) / v can have
// its base texel within [lo - 1, hi] of the box: the ray's interval in FP64, widened by 0.05 texel plus
// 1e-5 of the coordinates' magnitude (the FP32 points are within a few 1e-7 of it) and by one index
// either way.  All depths for values too large to bound so.  (FP32 intervals take 5 % less time.)
__device__ __forceinline__ void ray_depths(const FlagBeamDev& d, const MaskBox& box, const float p[3],
                                           const float v[3], int& i0, int& i1) {
    double lo = 0.0, hi = 1e30;  // scale = depth / sad
    const double far_scale = ((double)d.lim_min + (double)d.L * d.ls) / d.sad;
    bool odd = !(far_scale < 1e9 && far_scale > 0.0);
    for (int a = 0; a < 3; a++) {
        const double s = d.src[a], q = p[a], u = v[a];
        odd |= !(fabs(s) < 1e9 && fabs(q) < 1e9 && u > 1e-9);
        const double m = u * 0.05 + 1e-5 * (fabs(s) + fabs(q) * far_scale);
        // base texel in [lo - 1, hi]: coordinate / v in [lo - 0.5, hi + 1.5)
        const double x0 = (box.lo[a] - 0.5) * u - m - s, x1 = (box.hi[a] + 1.5) * u + m - s;
        if (q > 0.0) {
            lo = fmax(lo, x0 / q);
            hi = fmin(hi, x1 / q);
        } else if (q < 0.0) {
            lo = fmax(lo, x1 / q);
            hi = fmin(hi, x0 / q);
        } else if (x0 > 0.0 || x1 < 0.0) {
            hi = -1.0;
        }
    }
    i0 = 0;
    i1 = d.L;
    if (odd) return;
    const double L = d.L, a0 = (lo * d.sad - d.lim_min) / d.ls - 1.0, a1 = (hi * d.sad - d.lim_min) / d.ls + 2.0;
    if (!(lo <= hi) || a0 >= L || a1 <= 0.0) {
        i1 = 0;
        return;
    }
    i0 = (int)fmax(a0, 0.0);
    i1 = (int)ceil(fmin(a1, L));
}

constexpr int kFlagWaves = 4;  // beamlets per workgroup

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
    const MaskBox box = read_box(mask_box);
    const float v[3] = {vx, vy, vz};
    // the depths at which one of the nine rays can be inside the mask's box
    int first = d.L, last = 0;
    if (lane < kFlagSS * kFlagSS && box.lo[0] <= box.hi[0]) {
        float p[3];
        int i0, i1;
        sample_ray(d, bx, by, lane, p);
        ray_depths(d, box, p, v, i0, i1);
        if (i0 < i1) {
            first = i0;
            last = i1;
        }
    }
    for (int o = 8; o > 0; o >>= 1) {  // lanes 0 ... 15 hold the nine rays
        first = min(first, __shfl_xor(first, o, 64));
        last = max(last, __shfl_xor(last, o, 64));
    }
    first = __builtin_amdgcn_readfirstlane(first);
    last = __builtin_amdgcn_readfirstlane(last);
    const int total = last * kFlagSS * kFlagSS;
    bool on = false;
    for (int t0 = first * kFlagSS * kFlagSS; t0 < total && !on; t0 += 64) {
        const int t = t0 + lane;
        bool hit = false;
        if (t < total) {
            const uint32_t i = (uint32_t)(t / (kFlagSS * kFlagSS));
            const float depth = d.lim_min + (float)i * d.ls;
            const float scale = depth / d.sad;
            float p[3];
            sample_ray(d, bx, by, t - (int)i * kFlagSS * kFlagSS, p);
            hit = mask_hit_dev(mask, X, Y, Z, box, fmaf(p[0], scale, d.src[0]) / vx,
                               fmaf(p[1], scale, d.src[1]) / vy, fmaf(p[2], scale, d.src[2]) / vz);
        }
        on = __any(hit);
    }
    if (lane == 0) flags[d.out_off + idx] = on ? 1 : 0;
}

}  // namespace

hipError_t launch_beamlet_flags(const FlagBeamDev* beams, int n, int max_pixels, const uint8_t* mask,
                                const fd_volume& vol, uint32_t* box, uint8_t* flags, hipStream_t stream) {
    if (n <= 0 || max_pixels <= 0) return hipSuccess;
    const uint64_t voxels = (uint64_t)vol.dim[0] * vol.dim[1] * vol.dim[2];
    hipError_t e = launch_fill_u32(box, 6, ~0u, stream);
    if (e != hipSuccess) return e;
    const uint64_t blocks = (voxels / 16 + 255) / 256 + 1;
    hipLaunchKernelGGL(mask_box_kernel, dim3((unsigned)(blocks < 1024 ? blocks : 1024)), dim3(256), 0, stream, mask,
                       vol.dim[0], vol.dim[1], voxels, box);
    dim3 grid((unsigned)((max_pixels + kFlagWaves - 1) / kFlagWaves), (unsigned)n), block(64 * kFlagWaves);
    hipLaunchKernelGGL(beamlet_flags_kernel, grid, block, 0, stream, beams, mask, (int)vol.dim[0], (int)vol.dim[1],
                       (int)vol.dim[2], vol.voxel_size[0], vol.voxel_size[1], vol.voxel_size[2], box, flags);
    return hipGetLastError();
}

}  // namespace fdi
