// tv.hip -- total-variation steps of ASD-POCS for gfx950.
//
// For a volume x, D its backward differences along z, y, x and |D|_eps = sqrt(eps + |D|^2), the
// gradient of sum |D|_eps at an interior voxel c (the vector of python/ASD_POCS.py:55-72) is
//   g(c) = (D_z + D_y + D_x)(c) / |D(c)|_eps
//          - D_z(c + e_z) / |D(c + e_z)|_eps - D_y(c + e_y) / |D(c + e_y)|_eps - D_x(c + e_x) / |D(c + e_x)|_eps,
// zero on the volume's border, and a step is x - step * g / norm with norm = ||g||_2, or 1 below eps
// (python/ASD_POCS.py:73-77, 188-192).  A batch holds independent volumes.
//
// A step is three launches: tv_pass_kernel<kTvNorm> sums g^2 per workgroup, tv_norm_kernel adds the
// sums up per volume, and tv_pass_kernel evaluates g again and applies it.  g is recomputed rather
// than stored: a pass reads the volume about twice from beyond L2 (its planes stay in the caches) and is
// bound by the vector memory path in front of them (seven reads per voxel: texture data unit busy 0.70-0.78,
// address unit 0.59-0.69 of the cycles, VALU issue 0.17-0.19 per SIMD-cycle), about as long as the 2 x 4
// bytes per voxel that storing and rereading g would add.
// Measured per step, 8 x 128^3: about 950 us as some 25 torch elementwise and reduction kernels, 82 us
// here (31 + 5 + 46).

#include <hip/hip_runtime.h>

#include <algorithm>
#include <cfloat>
#include <cmath>
#include <cstdint>

#include "ctrecon.h"

namespace {

constexpr int kTvX = 64, kTvY = 4;  // a workgroup's columns: a wavefront along x, four rows
constexpr int kTvZ = 16;            // planes a work-item walks

enum { kTvNorm, kTvGradient, kTvStep };

// 1 / sqrt(s) of a normal s: the hardware's estimate and one Newton step (0 where s has overflowed)
__device__ inline float tv_rsqrt(float s) {
    const float r = __builtin_amdgcn_rsqf(s);
    return s <= 3.4028235e38f ? fmaf(0.5f * r, fmaf(-s * r, r, 1.0f), r) : r;
}

// One work-item per (x, y) column and kTvZ planes.  Walking up in z, the planes' values and the
// ratio D_z / |D| of the plane above carry over, so a voxel costs seven reads and three roots: its
// successors' along x and y, and the next plane's own.
//   kTvNorm: sums[block] = sum of g^2;  kTvGradient: out = g / norm, 0 on the border;
//   kTvStep: out = x - step * g / norm (out must not be x).
template <int MODE>
__global__ void __launch_bounds__(kTvX * kTvY) tv_pass_kernel(const float* __restrict__ x, float* __restrict__ out,
                                                              double* __restrict__ sums, const float* __restrict__ norm,
                                                              const float* __restrict__ step, int nx, int ny, int nz,
                                                              int tiles_x, float eps) {
    const int ix = (blockIdx.x % tiles_x) * kTvX + (threadIdx.x & (kTvX - 1));
    const int iy = (blockIdx.x / tiles_x) * kTvY + threadIdx.x / kTvX;
    const int iz0 = blockIdx.y * kTvZ, iz1 = min(iz0 + kTvZ, nz);
    const size_t plane = (size_t)ny * nx, vol = plane * nz;
    const float* __restrict__ v = x + vol * blockIdx.z;
    float scale = 0.0f, width = 1.0f;
    if constexpr (MODE != kTvNorm) width = norm[blockIdx.z];
    if constexpr (MODE == kTvStep) scale = step[blockIdx.z];
    double sum = 0.0;
    const bool in_vol = ix < nx && iy < ny;
    if (ix >= 1 && ix < nx - 1 && iy >= 1 && iy < ny - 1) {
        const float* __restrict__ p = v + (size_t)iy * nx + ix;
        struct Plane {
            float c, l, r, d, u, rd, lu;  // own, x-1, x+1, y-1, y+1, (x+1, y-1), (x-1, y+1)
        };
        auto load = [&](int z) {
            const float* __restrict__ q = p + (size_t)z * plane;
            return Plane{q[0], q[-1], q[1], q[-nx], q[nx], q[1 - nx], q[nx - 1]};
        };
        const int za = max(iz0, 1), zb = min(iz1, nz - 1);  // interior planes of this chunk
        if (za < zb) {
            Plane low = load(za - 1), here = load(za);
            float dz = here.c - low.c, dy = here.c - here.d, dx = here.c - here.l;
            float inv = tv_rsqrt(eps + dz * dz + dy * dy + dx * dx);
            for (int z = za; z < zb; ++z) {
                const Plane high = load(z + 1);
                // |D| of the successors along x and y, and of the voxel above
                const float xz = here.r - low.r, xy = here.r - here.rd, xx = here.r - here.c;
                const float yz = here.u - low.u, yy = here.u - here.c, yx = here.u - here.lu;
                const float zz = high.c - here.c, zy = high.c - high.d, zx = high.c - high.l;
                const float inv_z = tv_rsqrt(eps + zz * zz + zy * zy + zx * zx);
                const float g = (dz + dy + dx) * inv - (zz * inv_z + yy * tv_rsqrt(eps + yz * yz + yy * yy + yx * yx) +
                                                        xx * tv_rsqrt(eps + xz * xz + xy * xy + xx * xx));
                if constexpr (MODE == kTvNorm)
                    sum += (double)(g * g);
                else if constexpr (MODE == kTvGradient)
                    out[vol * blockIdx.z + (size_t)z * plane + (size_t)iy * nx + ix] = g / width;
                else
                    out[vol * blockIdx.z + (size_t)z * plane + (size_t)iy * nx + ix] = here.c - scale * (g / width);
                low = here;
                here = high;
                dz = zz;
                dy = zy;
                dx = zx;
                inv = inv_z;
            }
        }
    }
    if constexpr (MODE != kTvNorm) {
        // the border
        if (in_vol)
            for (int z = iz0; z < iz1; ++z) {
                if (ix >= 1 && ix < nx - 1 && iy >= 1 && iy < ny - 1 && z >= 1 && z < nz - 1) continue;
                const size_t o = (size_t)z * plane + (size_t)iy * nx + ix;
                out[vol * blockIdx.z + o] = MODE == kTvStep ? v[o] : 0.0f;
            }
    } else {
        __shared__ double part[kTvX * kTvY / 64];
#pragma unroll
        for (int d = 32; d > 0; d >>= 1) sum += __shfl_down(sum, d);
        if ((threadIdx.x & 63) == 0) part[threadIdx.x >> 6] = sum;
        __syncthreads();
        if (threadIdx.x == 0) {
            double s = 0.0;
            for (int w = 0; w < kTvX * kTvY / 64; ++w) s += part[w];
            sums[((size_t)blockIdx.z * gridDim.y + blockIdx.y) * gridDim.x + blockIdx.x] = s;
        }
    }
}

// norm[b] = sqrt(sum of volume b's partial sums), or 1 where that is below eps
__global__ void __launch_bounds__(256) tv_norm_kernel(const double* __restrict__ sums, float* __restrict__ norm, int n,
                                                      float eps) {
    __shared__ double part[256];
    const double* __restrict__ s = sums + (size_t)blockIdx.x * n;
    double acc = 0.0;
    for (int i = threadIdx.x; i < n; i += 256) acc += s[i];
    part[threadIdx.x] = acc;
    for (int d = 128; d > 0; d >>= 1) {
        __syncthreads();
        if (threadIdx.x < d) part[threadIdx.x] += part[threadIdx.x + d];
    }
    if (threadIdx.x == 0) {
        const float r = (float)sqrt(part[0]);
        // on the bit patterns (r and eps are not negative), so that a NaN stays one
        norm[blockIdx.x] = __float_as_uint(r) < __float_as_uint(eps) ? 1.0f : r;
    }
}

struct TvLayout {
    int tiles_x, tiles, chunks;
    size_t norm_off, sums_off, vol_off, total;
};

// workspace: norms, partial sums and (for several steps) one batch of volumes
TvLayout tv_layout(int batch, int nx, int ny, int nz, int steps) {
    TvLayout l;
    l.tiles_x = (nx + kTvX - 1) / kTvX;
    l.tiles = l.tiles_x * ((ny + kTvY - 1) / kTvY);
    l.chunks = (nz + kTvZ - 1) / kTvZ;
    auto up = [](size_t n) { return (n + 255) / 256 * 256; };
    l.norm_off = 0;
    l.sums_off = up((size_t)batch * sizeof(float));
    l.vol_off = l.sums_off + up((size_t)batch * l.tiles * l.chunks * sizeof(double));
    l.total = l.vol_off + (steps > 1 ? (size_t)batch * nx * ny * nz * sizeof(float) : 0);
    return l;
}

bool tv_sizes_ok(int batch, int nx, int ny, int nz) {
    return batch > 0 && batch <= 65535 && nx >= 3 && ny >= 3 && nz >= 3 && nz <= 65535 * kTvZ &&
           (double)nx * ny * nz < 2147483647.0;
}

int tv_status() { return hipGetLastError() == hipSuccess ? CTR_OK : CTR_ERR_HIP; }

// norm[b] of the gradient of x
int tv_norms(const float* x, const TvLayout& l, char* ws, int batch, int nx, int ny, int nz, float eps, hipStream_t s) {
    double* sums = (double*)(ws + l.sums_off);
    hipLaunchKernelGGL(HIP_KERNEL_NAME(tv_pass_kernel<kTvNorm>), dim3(l.tiles, l.chunks, batch), dim3(kTvX * kTvY), 0, s, x,
                       (float*)nullptr, sums, (const float*)nullptr, (const float*)nullptr, nx, ny, nz, l.tiles_x, eps);
    const int st = tv_status();
    if (st) return st;
    hipLaunchKernelGGL(tv_norm_kernel, dim3(batch), dim3(256), 0, s, sums, (float*)(ws + l.norm_off), l.tiles * l.chunks,
                       eps);
    return tv_status();
}

}  // namespace

extern "C" {

size_t ctr_tv_workspace_bytes(int batch, int nx, int ny, int nz, int steps) {
    return tv_sizes_ok(batch, nx, ny, nz) ? tv_layout(batch, nx, ny, nz, steps).total : 0;
}

int ctr_tv_gradient(const float* x, float* grad, int batch, int nx, int ny, int nz, float eps, void* workspace,
                    size_t workspace_bytes, void* stream) {
    if (!x || !grad || !workspace || x == grad || !tv_sizes_ok(batch, nx, ny, nz) || !(eps >= FLT_MIN)) return CTR_ERR_INVALID;
    const TvLayout l = tv_layout(batch, nx, ny, nz, 1);
    if (workspace_bytes < l.total) return CTR_ERR_WORKSPACE;
    hipStream_t s = (hipStream_t)stream;
    char* ws = (char*)workspace;
    const int st = tv_norms(x, l, ws, batch, nx, ny, nz, eps, s);
    if (st) return st;
    hipLaunchKernelGGL(HIP_KERNEL_NAME(tv_pass_kernel<kTvGradient>), dim3(l.tiles, l.chunks, batch), dim3(kTvX * kTvY), 0,
                       s, x, grad, (double*)nullptr, (const float*)(ws + l.norm_off), (const float*)nullptr, nx, ny, nz,
                       l.tiles_x, eps);
    return tv_status();
}

int ctr_tv_descent(const float* x, float* out, const float* step, int batch, int nx, int ny, int nz, float eps, int steps,
                   void* workspace, size_t workspace_bytes, void* stream) {
    if (!x || !out || !step || !workspace || x == out || steps < 1 || !tv_sizes_ok(batch, nx, ny, nz) || !(eps >= FLT_MIN))
        return CTR_ERR_INVALID;
    const TvLayout l = tv_layout(batch, nx, ny, nz, steps);
    if (workspace_bytes < l.total) return CTR_ERR_WORKSPACE;
    hipStream_t s = (hipStream_t)stream;
    char* ws = (char*)workspace;
    float* other = (float*)(ws + l.vol_off);
    const float* from = x;
    for (int k = 0; k < steps; ++k) {
        // the last step writes `out`, the ones before it the two buffers in turn
        float* to = ((steps - 1 - k) & 1) ? other : out;
        int st = tv_norms(from, l, ws, batch, nx, ny, nz, eps, s);
        if (st) return st;
        hipLaunchKernelGGL(HIP_KERNEL_NAME(tv_pass_kernel<kTvStep>), dim3(l.tiles, l.chunks, batch), dim3(kTvX * kTvY), 0,
                           s, from, to, (double*)nullptr, (const float*)(ws + l.norm_off), step, nx, ny, nz, l.tiles_x,
                           eps);
        if ((st = tv_status())) return st;
        from = to;
    }
    return CTR_OK;
}

}  // extern "C"
