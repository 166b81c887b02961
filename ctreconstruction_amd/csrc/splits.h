// splits.h -- view splits: a backprojection of few voxel tiles shares each tile's views out to several
// workgroups, which sum into copies of the volume ("parts"); this adds the copies up.
#ifndef CTR_SPLITS_H
#define CTR_SPLITS_H

#include <hip/hip_runtime.h>

#include <cstdint>

#include "ctrecon.h"

namespace {

// vol = (accumulate ? vol : 0) + the splits' partial volumes, in split order (deterministic); blockIdx.y
// is the volume of a batch.
// One 16-byte load per split and thread where the volume's size and address allow it (W = 4).
template <int W>
__global__ void __launch_bounds__(256) sum_parts_kernel(const float* __restrict__ parts, float* __restrict__ vol,
                                                        size_t n, int splits, int accumulate) {
    typedef float vec __attribute__((ext_vector_type(W)));
    const size_t i = ((size_t)blockIdx.x * 256 + threadIdx.x) * W;
    if (i >= n) return;
    parts += (size_t)blockIdx.y * splits * n;
    vol += (size_t)blockIdx.y * n;
    vec sum = *reinterpret_cast<const vec*>(parts + i);
    for (int s = 1; s < splits; ++s) sum += *reinterpret_cast<const vec*>(parts + (size_t)s * n + i);
    vec* out = reinterpret_cast<vec*>(vol + i);
    *out = accumulate ? *out + sum : sum;
}

inline int sum_parts(const ctr_geometry* g, const float* parts, float* vol, int splits, int accumulate, hipStream_t s,
                     int batch = 1) {
    const size_t n = (size_t)g->nx * g->ny * g->nz;
    if (n % 4 == 0 && (reinterpret_cast<uintptr_t>(vol) & 15) == 0)
        hipLaunchKernelGGL(HIP_KERNEL_NAME(sum_parts_kernel<4>), dim3((unsigned)((n / 4 + 255) / 256), batch), dim3(256), 0, s,
                           parts, vol, n, splits, accumulate);
    else
        hipLaunchKernelGGL(HIP_KERNEL_NAME(sum_parts_kernel<1>), dim3((unsigned)((n + 255) / 256), batch), dim3(256), 0, s,
                           parts, vol, n, splits, accumulate);
    return hipGetLastError() == hipSuccess ? CTR_OK : CTR_ERR_HIP;
}

}  // namespace

#endif  // CTR_SPLITS_H
