// iterate.hip -- the elementwise parts of a SART / ASD-POCS iteration for gfx950, one pass each.
//
// The iteration x <- x + relax B(w (p - A x)) / (B 1 + eps) (python/SART.py:44-59,
// python/ASD_POCS.py:170-186) has two elementwise parts, the weighted residual and the update.  As
// torch expressions they were about ten passes over the projections and five over the volume; each is
// one pass here, bound by HBM.  The operations and their order are the expressions', so the results are
// theirs bit for bit.  Three SART iterations at 256^3 x 60 views of 384 x 384: 5.58 -> 5.03 ms; an outer
// ASD-POCS iteration over eight 128^3 volumes: 9.40 -> 8.81 ms.

#include <hip/hip_runtime.h>

#include <cstdint>
#include <initializer_list>

#include "ctrecon.h"

namespace {

// W elements per thread (16-byte accesses where sizes and addresses allow); blockIdx.y is the volume of
// the batch, `a` and `b` belong to the geometry and serve every one.
template <int W>
struct Vec {
    typedef float type __attribute__((ext_vector_type(W)));
};
template <>
struct Vec<1> {
    struct type {
        float v;
        __device__ float& operator[](int) { return v; }
    };
};

// out = weighted ? a (ax - p) : (a == 0 ? 0 : (p - ax) / (a + eps))
template <int W>
__global__ void __launch_bounds__(256) residual_kernel(const float* __restrict__ p, const float* __restrict__ ax,
                                                       const float* __restrict__ a, float* __restrict__ out, size_t n,
                                                       int weighted, float eps) {
    typedef typename Vec<W>::type vec;
    const size_t i = ((size_t)blockIdx.x * 256 + threadIdx.x) * W, o = (size_t)blockIdx.y * n + i;
    if (i >= n) return;
    vec vp = *reinterpret_cast<const vec*>(p + o), vx = *reinterpret_cast<const vec*>(ax + o);
    vec va = *reinterpret_cast<const vec*>(a + i), r;
#pragma unroll
    for (int k = 0; k < W; ++k) {
        if (weighted)
            r[k] = va[k] * (vx[k] - vp[k]);
        else
            r[k] = va[k] == 0.0f ? 0.0f : (vp[k] - vx[k]) / (va[k] + eps);
    }
    *reinterpret_cast<vec*>(out + o) = r;
}

// out = x + (relax u) / (b + eps), u taken as 0 where b is 0 (masked), then negative values 0 (nonneg)
template <int W>
__global__ void __launch_bounds__(256) update_kernel(const float* __restrict__ x, const float* __restrict__ u,
                                                     const float* __restrict__ b, float* __restrict__ out, size_t n,
                                                     float relax, float eps, int masked, int nonneg) {
    typedef typename Vec<W>::type vec;
    const size_t i = ((size_t)blockIdx.x * 256 + threadIdx.x) * W, o = (size_t)blockIdx.y * n + i;
    if (i >= n) return;
    vec vx = *reinterpret_cast<const vec*>(x + o), vu = *reinterpret_cast<const vec*>(u + o);
    vec vb = *reinterpret_cast<const vec*>(b + i), r;
#pragma unroll
    for (int k = 0; k < W; ++k) {
        const float t = masked && vb[k] == 0.0f ? 0.0f : vu[k];
        float v = vx[k] + (relax * t) / (vb[k] + eps);
        // on the bit patterns, so that a NaN stays one: -0.0 .. -inf become 0
        const uint32_t bits = __float_as_uint(v);
        if (nonneg && bits >= 0x80000000u && bits <= 0xff800000u) v = 0.0f;
        r[k] = v;
    }
    *reinterpret_cast<vec*>(out + o) = r;
}

bool wide(size_t n, std::initializer_list<const void*> ptrs) {
    uintptr_t bits = n % 4 ? 1 : 0;
    for (const void* p : ptrs) bits |= reinterpret_cast<uintptr_t>(p) & 15;
    return bits == 0;
}

// a launch's x extent is at most 2^32 - 1 threads
bool sizes_ok(size_t n, int batch) { return n > 0 && n <= 0xffffff00u && batch > 0 && batch <= 65535; }

}  // namespace

extern "C" {

int ctr_residual(const float* p, const float* ax, const float* a, float* out, size_t n, int batch, int weighted, float eps,
                 void* stream) {
    if (!p || !ax || !a || !out || !sizes_ok(n, batch)) return CTR_ERR_INVALID;
    hipStream_t s = (hipStream_t)stream;
    if (wide(n, {p, ax, a, out}))
        hipLaunchKernelGGL(HIP_KERNEL_NAME(residual_kernel<4>), dim3((unsigned)((n / 4 + 255) / 256), batch), dim3(256), 0, s,
                           p, ax, a, out, n, weighted, eps);
    else
        hipLaunchKernelGGL(HIP_KERNEL_NAME(residual_kernel<1>), dim3((unsigned)((n + 255) / 256), batch), dim3(256), 0, s, p,
                           ax, a, out, n, weighted, eps);
    return hipGetLastError() == hipSuccess ? CTR_OK : CTR_ERR_HIP;
}

int ctr_update(const float* x, const float* u, const float* b, float* out, size_t n, int batch, float relax, float eps,
               int masked, int nonneg, void* stream) {
    if (!x || !u || !b || !out || !sizes_ok(n, batch)) return CTR_ERR_INVALID;
    hipStream_t s = (hipStream_t)stream;
    if (wide(n, {x, u, b, out}))
        hipLaunchKernelGGL(HIP_KERNEL_NAME(update_kernel<4>), dim3((unsigned)((n / 4 + 255) / 256), batch), dim3(256), 0, s, x,
                           u, b, out, n, relax, eps, masked, nonneg);
    else
        hipLaunchKernelGGL(HIP_KERNEL_NAME(update_kernel<1>), dim3((unsigned)((n + 255) / 256), batch), dim3(256), 0, s, x, u,
                           b, out, n, relax, eps, masked, nonneg);
    return hipGetLastError() == hipSuccess ? CTR_OK : CTR_ERR_HIP;
}

}  // extern "C"
