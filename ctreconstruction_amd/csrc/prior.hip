// prior.hip -- gfx950 kernels of the learned 2.5D residual prior (no reference counterpart).
//
// 3x3 "same" convolutions over NHWC bfloat16 activations with bfloat16 weights [Cout][3][3][Cin]
// and FP32 accumulation:
//   conv3x3_fwd_kernel    implicit GEMM on MFMA (v_mfma_f32_16x16x32_bf16): M = pixels,
//                         N = Cout, K = 9*Cin; epilogue adds bias, optional ReLU, optional
//                         residual, stores bfloat16.  The input gradient of a convolution is
//                         the same kernel applied to the output gradient with the weights
//                         flipped in space and transposed in channels.
//   conv3x3_fwd_small_cin_kernel  the same for at most 4 input channels, input halo in LDS
//   conv3x3_fwd_persistent_kernel  the same for 64 input channels and 64 or at most 16 output
//                         channels: one workgroup per CU with all weights in LDS, walking pixel
//                         tiles with the next tile's input halo loaded while the current one is
//                         computed.
//   conv3x3_wgrad_kernel  weight and bias gradients on MFMA: 8 x 32 pixel tiles of the output
//                         gradient and their input halos staged in LDS and read transposed;
//                         grad_w = gout^T x_shift with K = pixels for all nine taps, FP32
//                         accumulation; partial sums per workgroup
//   conv3x3_wgrad_reduce  sums the partials in a fixed order (deterministic)
//   conv3x3_flip_kernel   weights of the input-gradient convolution

#include <hip/hip_runtime.h>

#include <algorithm>
#include <cstdint>

#include "ctrecon.h"

namespace {

typedef __bf16 bf16_t;
typedef bf16_t bf16x8 __attribute__((ext_vector_type(8)));
typedef bf16_t bf16x4 __attribute__((ext_vector_type(4)));
typedef float f32x4 __attribute__((ext_vector_type(4)));

constexpr int kConvWaves = 4;    // waves per workgroup
constexpr int kPxPerWave = 32;   // two 16-pixel MFMA row tiles per wave
constexpr int kMaxCout = 64;     // four 16-channel MFMA column tiles

__device__ inline bf16x8 zero8() {
    bf16x8 z;
#pragma unroll
    for (int e = 0; e < 8; ++e) z[e] = (bf16_t)0.0f;
    return z;
}

// MFMA operand layout (16 x 16 x 32, wave64): lane l supplies row (l % 16) of A and column
// (l % 16) of B, both with the 8 consecutive K elements 8*(l / 16) .. 8*(l / 16) + 7; it receives
// rows 4*(l / 16) .. +3 of column (l % 16) of D.
template <bool FAST>
__global__ void __launch_bounds__(256) conv3x3_fwd_kernel(
    const bf16_t* __restrict__ in, const bf16_t* __restrict__ w, const float* __restrict__ bias,
    const bf16_t* __restrict__ resid, bf16_t* __restrict__ out, int N, int H, int W, int Cin,
    int Cout, int relu, int vec) {
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    const int P = N * H * W;
    const int pbase = (blockIdx.x * kConvWaves + wave) * kPxPerWave;
    const int m = lane & 15, g = lane >> 4;
    const int K = 9 * Cin;
    const int ksteps = (K + 31) / 32;
    const int n_tiles = (Cout + 15) / 16;
    int py[2], px[2], pn[2];
    bool pv[2];
#pragma unroll
    for (int h = 0; h < 2; ++h) {
        const int p = pbase + h * 16 + m;
        pv[h] = p < P;
        const int pp = pv[h] ? p : 0;
        px[h] = pp % W;
        const int t = pp / W;
        py[h] = t % H;
        pn[h] = t / H;
    }
    f32x4 acc[2][4];
#pragma unroll
    for (int h = 0; h < 2; ++h)
#pragma unroll
        for (int t = 0; t < 4; ++t) acc[h][t] = f32x4{0.0f, 0.0f, 0.0f, 0.0f};

    for (int s = 0; s < ksteps; ++s) {
        const int k0 = s * 32 + g * 8;
        bf16x8 a[2], b[4];
        if constexpr (FAST) {
            // Cin % 32 == 0: the 8 K elements are 8 channels of one tap, 16-byte aligned
            const int tap = k0 / Cin, ci = k0 - tap * Cin;
            const int dy = tap / 3 - 1, dx = tap % 3 - 1;
#pragma unroll
            for (int h = 0; h < 2; ++h) {
                const int yy = py[h] + dy, xx = px[h] + dx;
                const bool ok = pv[h] && yy >= 0 && yy < H && xx >= 0 && xx < W;
                a[h] = ok ? *reinterpret_cast<const bf16x8*>(
                                in + ((size_t)(pn[h] * H + yy) * W + xx) * Cin + ci)
                          : zero8();
            }
#pragma unroll
            for (int t = 0; t < 4; ++t) {
                const int co = t * 16 + m;
                b[t] = (co < Cout) ? *reinterpret_cast<const bf16x8*>(w + (size_t)co * K + k0) : zero8();
            }
        } else {
#pragma unroll
            for (int h = 0; h < 2; ++h) a[h] = zero8();
#pragma unroll
            for (int t = 0; t < 4; ++t) b[t] = zero8();
#pragma unroll
            for (int e = 0; e < 8; ++e) {
                const int k = k0 + e;
                if (k >= K) break;
                const int tap = k / Cin, ci = k - tap * Cin;
                const int dy = tap / 3 - 1, dx = tap % 3 - 1;
#pragma unroll
                for (int h = 0; h < 2; ++h) {
                    const int yy = py[h] + dy, xx = px[h] + dx;
                    if (pv[h] && yy >= 0 && yy < H && xx >= 0 && xx < W)
                        a[h][e] = in[((size_t)(pn[h] * H + yy) * W + xx) * Cin + ci];
                }
#pragma unroll
                for (int t = 0; t < 4; ++t) {
                    const int co = t * 16 + m;
                    if (co < Cout) b[t][e] = w[(size_t)co * K + k];
                }
            }
        }
        // the weights are the row operand: lane (m, g) receives output channels
        // 16 t + 4 g .. +3 of pixel m, four adjacent values of one NHWC row
#pragma unroll
        for (int h = 0; h < 2; ++h)
#pragma unroll
            for (int t = 0; t < 4; ++t)
                if (t < n_tiles)  // uniform: column tiles past Cout are all zero
                    acc[h][t] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(b[t], a[h], acc[h][t], 0, 0, 0);
    }
#pragma unroll
    for (int t = 0; t < 4; ++t) {
        if (t >= n_tiles) continue;
        const int co0 = t * 16 + 4 * g;
        if (co0 >= Cout) continue;
#pragma unroll
        for (int h = 0; h < 2; ++h) {
            const int p = pbase + h * 16 + m;
            if (p >= P) continue;
            const size_t o = (size_t)p * Cout + co0;
            float v[4];
#pragma unroll
            for (int r = 0; r < 4; ++r) {
                v[r] = acc[h][t][r] + ((bias && co0 + r < Cout) ? bias[co0 + r] : 0.0f);
                if (relu) v[r] = fmaxf(v[r], 0.0f);
            }
            if (vec) {  // Cout % 4 == 0 and 8-byte aligned rows: four channels per access
                if (resid) {
                    const bf16x4 rv = *reinterpret_cast<const bf16x4*>(resid + o);
#pragma unroll
                    for (int r = 0; r < 4; ++r) v[r] += (float)rv[r];
                }
                bf16x4 q;
#pragma unroll
                for (int r = 0; r < 4; ++r) q[r] = (bf16_t)v[r];
                *reinterpret_cast<bf16x4*>(out + o) = q;
            } else {
#pragma unroll
                for (int r = 0; r < 4; ++r) {
                    if (co0 + r >= Cout) break;
                    float x = v[r];
                    if (resid) x += (float)resid[o + r];
                    out[o + r] = (bf16_t)x;
                }
            }
        }
    }
}

// Convolutions with at most 4 input channels (the network's first layer, 3 -> 64, and the input
// gradient of its last, 1 -> 64).  K = 9 taps x 4 channels (zero past Cin) in two MFMA K steps:
// taps 0-7, then tap 8.  A workgroup computes an 8 x 32 pixel tile from its (8+2) x (32+2) input
// halo in LDS (one 8-byte entry of 4 channels per pixel); lane (m, g) of wave w takes pixel m of
// the four 16-pixel row tiles of rows 2w, 2w+1 with K elements 8g .. 8g+7 (taps 2g and 2g+1 in
// the first step).  The workgroups are persistent: each builds the zero-padded weight operands
// in registers once and then walks tiles.
constexpr int kSTileH = 8, kSTileW = 32;
constexpr int kSHaloW = kSTileW + 2;
constexpr int kSHaloPix = (kSTileH + 2) * kSHaloW;

__global__ void __launch_bounds__(256) conv3x3_fwd_small_cin_kernel(
    const bf16_t* __restrict__ in, const bf16_t* __restrict__ w, const float* __restrict__ bias,
    const bf16_t* __restrict__ resid, bf16_t* __restrict__ out, int H, int W, int Cin, int Cout,
    int relu, int vec, int tiles_x, int tiles_y, int n_tiles) {
    __shared__ __attribute__((aligned(16))) bf16x4 halo[kSHaloPix];
    const int tid = threadIdx.x;
    const int lane = tid & 63, wave = tid >> 6;
    const int m = lane & 15, g = lane >> 4;
    const int n_ct = (Cout + 15) / 16;  // column tiles (uniform)
    // weights as the row operand: lane (m, g) of column tile t holds output channel 16 t + m,
    // K elements k = 32 s + 8 g + e of step s (tap k / 4, channel k % 4)
    bf16x8 b[2][4];
#pragma unroll
    for (int s = 0; s < 2; ++s)
#pragma unroll
        for (int t = 0; t < 4; ++t)
#pragma unroll
            for (int e = 0; e < 8; ++e) {
                const int k = 32 * s + 8 * g + e, tap = k >> 2, ci = k & 3, co = 16 * t + m;
                b[s][t][e] = (tap < 9 && ci < Cin && co < Cout) ? w[((size_t)co * 9 + tap) * Cin + ci] : (bf16_t)0.0f;
            }
    // lane (m, g) receives channels 16 t + 4 g .. +3 of its pixel: the bias starts them
    float bias_t[4][4];
#pragma unroll
    for (int t = 0; t < 4; ++t)
#pragma unroll
        for (int r = 0; r < 4; ++r) {
            const int co = 16 * t + 4 * g + r;
            bias_t[t][r] = (bias && co < Cout) ? bias[co] : 0.0f;
        }
    for (int tile = blockIdx.x; tile < n_tiles; tile += gridDim.x) {
        const int tx = tile % tiles_x, ty = (tile / tiles_x) % tiles_y, n = tile / (tiles_x * tiles_y);
        const int ty0 = ty * kSTileH, tx0 = tx * kSTileW;
        __syncthreads();  // the previous tile's halo is read
        for (int e = tid; e < kSHaloPix; e += 256) {
            const int yy = ty0 + e / kSHaloW - 1, xx = tx0 + e % kSHaloW - 1;
            bf16x4 v;
#pragma unroll
            for (int c = 0; c < 4; ++c) v[c] = (bf16_t)0.0f;
            if ((unsigned)yy < (unsigned)H && (unsigned)xx < (unsigned)W) {
                const bf16_t* src = in + ((size_t)(n * H + yy) * W + xx) * Cin;
#pragma unroll
                for (int c = 0; c < 4; ++c)
                    if (c < Cin) v[c] = src[c];
            }
            halo[e] = v;
        }
        __syncthreads();
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            const int row = 2 * wave + (i >> 1), col = 16 * (i & 1) + m;
            // halo entry of tap (dy, dx) for this pixel: (row + dy) * kSHaloW + col + dx
            const int t0 = 2 * g, t1 = 2 * g + 1;
            const bf16x4 p0 = halo[(row + t0 / 3) * kSHaloW + col + t0 % 3];
            const bf16x4 p1 = halo[(row + t1 / 3) * kSHaloW + col + t1 % 3];
            const bf16x4 p8 = halo[(row + 2) * kSHaloW + col + 2];
            bf16x8 a0, a1;
#pragma unroll
            for (int e = 0; e < 4; ++e) {
                a0[e] = p0[e];
                a0[4 + e] = p1[e];
                a1[e] = g == 0 ? p8[e] : (bf16_t)0.0f;
                a1[4 + e] = (bf16_t)0.0f;
            }
            const int yy = ty0 + row, xx = tx0 + col;
            const bool ok = yy < H && xx < W;
            const size_t o = ok ? ((size_t)(n * H + yy) * W + xx) * Cout : 0;
#pragma unroll
            for (int t = 0; t < 4; ++t) {
                if (t >= n_ct) break;
                f32x4 acc = f32x4{bias_t[t][0], bias_t[t][1], bias_t[t][2], bias_t[t][3]};
                acc = __builtin_amdgcn_mfma_f32_16x16x32_bf16(b[0][t], a0, acc, 0, 0, 0);
                acc = __builtin_amdgcn_mfma_f32_16x16x32_bf16(b[1][t], a1, acc, 0, 0, 0);
                const int co0 = 16 * t + 4 * g;
                if (!ok || co0 >= Cout) continue;
                float v[4];
#pragma unroll
                for (int r = 0; r < 4; ++r) v[r] = relu ? fmaxf(acc[r], 0.0f) : acc[r];
                if (vec) {  // Cout % 4 == 0 and 8-byte aligned rows
                    if (resid) {
                        const bf16x4 rv = *reinterpret_cast<const bf16x4*>(resid + o + co0);
#pragma unroll
                        for (int r = 0; r < 4; ++r) v[r] += (float)rv[r];
                    }
                    bf16x4 q;
#pragma unroll
                    for (int r = 0; r < 4; ++r) q[r] = (bf16_t)v[r];
                    *reinterpret_cast<bf16x4*>(out + o + co0) = q;
                } else {
#pragma unroll
                    for (int r = 0; r < 4; ++r) {
                        if (co0 + r >= Cout) break;
                        float x = v[r];
                        if (resid) x += (float)resid[o + co0 + r];
                        out[o + co0 + r] = (bf16_t)x;
                    }
                }
            }
        }
    }
}

// Persistent LDS variant for 64 input channels: the 64 -> 64 body of the network and its last
// layer (64 -> 1).  One 512-thread workgroup per CU keeps all nine taps of the weights in LDS
// (72 KB for 64 output channels) and walks 16 x 32 pixel
// tiles: the (16+2) x (32+2) input halo of the current tile sits in LDS (76.5 KB) while the
// next tile's halo is already loaded into registers.  Wave w computes rows 2w, 2w+1 of the
// tile: 4 MFMA row tiles (16 pixels) x 4 column tiles (16 channels), 16 MFMAs per 8 LDS
// operand reads in each K step of 32.  Rows of 8 16-byte chunks are stored with the chunk
// index XOR-ed by (row >> 1) & 7, so the operand reads of 16 consecutive pixels (or output
// channels) hit 16 different bank groups without padding.
constexpr int kPTileH = 16, kPTileW = 32;
constexpr int kPHaloW = kPTileW + 2;
constexpr int kPHaloPix = (kPTileH + 2) * kPHaloW;
constexpr int kPHaloChunks = kPHaloPix * 8;
constexpr int kPThreads = 512;
constexpr int kPPer = (kPHaloChunks + kPThreads - 1) / kPThreads;

__device__ inline int swz(int row, int chunk) { return chunk ^ ((row >> 1) & 7); }

// NT = 4 column tiles: 64 output channels, staged epilogue with 16-byte stores (and optional
// residual); NT = 1: up to 16 output channels (weights past Cout are zero), each lane stores its
// own channels (the network's last layer, 64 -> 1).
template <bool RELU, bool RESID, int NT>
__global__ void __launch_bounds__(kPThreads) conv3x3_fwd_persistent_kernel(
    const bf16_t* __restrict__ in, const bf16_t* __restrict__ w, const float* __restrict__ bias,
    const bf16_t* __restrict__ resid, bf16_t* __restrict__ out, int H, int W, int Cout, int tiles_x,
    int tiles_y, int n_tiles) {
    static_assert(NT == 4 || (NT == 1 && !RESID), "64 channels, or at most 16 without residual");
    constexpr int K = 9 * 64;
    constexpr int kCo = 16 * NT;  // output channels held in LDS (zero past Cout)
    __shared__ __attribute__((aligned(16))) bf16_t wl[kCo * 9 * 64];
    __shared__ __attribute__((aligned(16))) bf16_t halo[kPHaloPix * 64];
    const int tid = threadIdx.x;
    // all weights: row (co, tap) of 8 chunks
    for (int e = tid; e < kCo * 9 * 8; e += kPThreads) {
        const int c = e & 7, row = e >> 3;  // row = co * 9 + tap
        const int co = row / 9;
        *reinterpret_cast<bf16x8*>(&wl[(row * 8 + swz(co, c)) * 8]) =
            co < Cout ? *reinterpret_cast<const bf16x8*>(w + (size_t)co * K + (row - co * 9) * 64 + c * 8) : zero8();
    }
    // the halo chunks of this thread, the same for every tile: position in the halo relative to
    // the tile origin (hy, hx >= -1), element offset in the input, element offset in LDS
    int h_yx[kPPer], h_in[kPPer], h_lds[kPPer];
#pragma unroll
    for (int p = 0; p < kPPer; ++p) {
        const int e = tid + p * kPThreads;
        const int c = e & 7, pix = min(e >> 3, kPHaloPix - 1);
        const int hy = pix / kPHaloW - 1, hx = pix % kPHaloW - 1;
        h_yx[p] = ((hy + 1) << 16) | (hx + 1);
        h_in[p] = (hy * W + hx) * 64 + c * 8;
        h_lds[p] = (pix * 8 + swz(pix, c)) * 8;
    }
    bf16x8 pre[kPPer];
    auto fetch = [&](int tile) {
        const int tx = tile % tiles_x;
        const int ty = (tile / tiles_x) % tiles_y;
        const int n = tile / (tiles_x * tiles_y);
        const int ty0 = ty * kPTileH, tx0 = tx * kPTileW;
        const bf16_t* base = in + ((size_t)(n * H + ty0) * W + tx0) * 64;
#pragma unroll
        for (int p = 0; p < kPPer; ++p) {
            const int e = tid + p * kPThreads;
            const int yy = ty0 - 1 + (h_yx[p] >> 16), xx = tx0 - 1 + (h_yx[p] & 0xffff);
            bf16x8 v = zero8();
            if (e < kPHaloChunks && (unsigned)yy < (unsigned)H && (unsigned)xx < (unsigned)W)
                v = *reinterpret_cast<const bf16x8*>(base + h_in[p]);
            pre[p] = v;
        }
    };
    auto store = [&]() {
#pragma unroll
        for (int p = 0; p < kPPer; ++p) {
            const int e = tid + p * kPThreads;
            if (e < kPHaloChunks) *reinterpret_cast<bf16x8*>(&halo[h_lds[p]]) = pre[p];
        }
    };
    const int lane = tid & 63, wave = tid >> 6;
    const int m = lane & 15, g = lane >> 4;
    // the MFMAs take the weights as the row operand, so lane (m, g) holds output channels
    // 16 t + 4 g + r of pixel m: the bias of those channels starts every accumulator
    float bias_t[NT][4];
#pragma unroll
    for (int t = 0; t < NT; ++t)
#pragma unroll
        for (int r = 0; r < 4; ++r) {
            const int co = t * 16 + 4 * g + r;
            bias_t[t][r] = (bias && co < Cout) ? bias[co] : 0.0f;
        }
    int tile = blockIdx.x;
    if (tile < n_tiles) {
        fetch(tile);
        store();
    }
    __syncthreads();
    while (tile < n_tiles) {
        const int next = tile + (int)gridDim.x;
        f32x4 acc[4][NT];
#pragma unroll
        for (int i = 0; i < 4; ++i)
#pragma unroll
            for (int t = 0; t < NT; ++t) acc[i][t] = f32x4{bias_t[t][0], bias_t[t][1], bias_t[t][2], bias_t[t][3]};
        // the previous tile's stores have completed (their data registers are reused by the
        // accumulators); the next tile's halo is then in flight while this tile is computed
        __builtin_amdgcn_s_waitcnt(0);
        if (next < n_tiles) fetch(next);
#pragma unroll 1
        for (int tap = 0; tap < 9; ++tap) {
            const int dy = tap / 3, dx = tap % 3;
#pragma unroll
            for (int c0 = 0; c0 < 8; c0 += 4) {  // chunk offset of the K step (32 channels)
                const int ch = c0 + g;
                bf16x8 b[NT], a[4];
#pragma unroll
                for (int t = 0; t < NT; ++t) {
                    const int co = t * 16 + m;
                    b[t] = *reinterpret_cast<const bf16x8*>(&wl[((co * 9 + tap) * 8 + swz(co, ch)) * 8]);
                }
#pragma unroll
                for (int i = 0; i < 4; ++i) {
                    const int pix = (2 * wave + (i >> 1) + dy) * kPHaloW + 16 * (i & 1) + m + dx;
                    a[i] = *reinterpret_cast<const bf16x8*>(&halo[(pix * 8 + swz(pix, ch)) * 8]);
                }
#pragma unroll
                for (int i = 0; i < 4; ++i)
#pragma unroll
                    for (int t = 0; t < NT; ++t)
                        acc[i][t] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(b[t], a[i], acc[i][t], 0, 0, 0);
            }
        }
        if constexpr (NT == 1) {
            // lane (m, g) holds channels 4 g .. 4 g + 3 of pixel m of each row tile: stored
            // straight from the accumulators (at most 16 channels per pixel)
            const int tx = tile % tiles_x;
            const int ty = (tile / tiles_x) % tiles_y;
            const int n = tile / (tiles_x * tiles_y);
#pragma unroll
            for (int i = 0; i < 4; ++i) {
                const int yy = ty * kPTileH + 2 * wave + (i >> 1), xx = tx * kPTileW + 16 * (i & 1) + m;
                if (yy >= H || xx >= W) continue;
                const size_t o = ((size_t)(n * H + yy) * W + xx) * Cout;
#pragma unroll
                for (int r = 0; r < 4; ++r) {
                    const int co = 4 * g + r;
                    if (co < Cout) out[o + co] = (bf16_t)(RELU ? fmaxf(acc[i][0][r], 0.0f) : acc[i][0][r]);
                }
            }
        } else {
            const int tx = tile % tiles_x;
            const int ty = (tile / tiles_x) % tiles_y;
            const int n = tile / (tiles_x * tiles_y);
            // this thread's output chunks (pixel, 8 channels): their residual is loaded now, so
            // that it arrives while the results are staged
            constexpr int kChunks = kPTileH * kPTileW * 8 / kPThreads;
            bf16x8 rv[RESID ? kChunks : 1];
            size_t o[kChunks];
            bool ok[kChunks];
#pragma unroll
            for (int k = 0; k < kChunks; ++k) {
                const int e = tid + k * kPThreads;
                const int c = e & 7, p = e >> 3;
                const int yy = ty * kPTileH + p / kPTileW, xx = tx * kPTileW + p % kPTileW;
                ok[k] = yy < H && xx < W;
                o[k] = ((size_t)(n * H + min(yy, H - 1)) * W + min(xx, W - 1)) * 64 + c * 8;
                if constexpr (RESID) rv[k] = *reinterpret_cast<const bf16x8*>(resid + o[k]);
            }
            __syncthreads();  // every wave is done with this halo: reuse it to stage the results
            // (ReLU), as bfloat16, into stage[pixel][channel] (pixel = row * 32 + column, rows of 8
            // 16-byte chunks swizzled like the halo): four channels per 8-byte store
            bf16_t* stage = halo;
#pragma unroll
            for (int i = 0; i < 4; ++i) {
                const int p = (2 * wave + (i >> 1)) * kPTileW + 16 * (i & 1) + m;
#pragma unroll
                for (int t = 0; t < 4; ++t) {
                    const int co = t * 16 + 4 * g;
                    bf16x4 q;
#pragma unroll
                    for (int r = 0; r < 4; ++r) q[r] = (bf16_t)(RELU ? fmaxf(acc[i][t][r], 0.0f) : acc[i][t][r]);
                    *reinterpret_cast<bf16x4*>(&stage[(p * 8 + swz(p, co >> 3)) * 8 + (co & 7)]) = q;
                }
            }
            __syncthreads();
            // 16-byte chunks (pixel, 8 channels); residual added in FP32
#pragma unroll
            for (int k = 0; k < kChunks; ++k) {
                const int e = tid + k * kPThreads;
                const int c = e & 7, p = e >> 3;
                bf16x8 v = *reinterpret_cast<const bf16x8*>(&stage[(p * 8 + swz(p, c)) * 8]);
                if constexpr (RESID) {
#pragma unroll
                    for (int q = 0; q < 8; ++q) v[q] = (bf16_t)((float)v[q] + (float)rv[k][q]);
                }
                if (ok[k]) *reinterpret_cast<bf16x8*>(out + o[k]) = v;
            }
        }
        __syncthreads();  // every wave is done with this halo
        if (next < n_tiles) store();
        __syncthreads();
        tile = next;
    }
}

// Weight and bias gradients on MFMA: grad_w[tap][co][ci] = sum_p gout[p][co] x[p + tap][ci], nine
// 64 x 64 GEMMs with K = pixels that share their operands.  A 512-thread workgroup walks 8 x 32 pixel
// tiles: the output gradient's tile and the input's (8+2) x (32+2) halo are staged in LDS as they lie
// in memory ([pixel][channel], 16-byte stores) and the K-major operands come out of LDS transposed
// (ds_read_b64_tr_b16: the 16 lanes of a group read four pixels x 16 channels and lane i receives
// channel i of the four), so a tap is a pixel offset of the read and no transposed copy is written.
// Wave (ci tile w % 4, co half w / 4) holds all nine taps of its 32 x 16 block: per K step (32 pixels
// of a row) it reads two operands of gout and, since a halo row serves three output rows, three of x
// for 18 MFMAs.  The next tile is loaded into registers meanwhile.  The bias gradient is one more
// MFMA against ones.  16-channel blocks are XOR-ed with bits of the pixel's column, so that the eight
// pixels of a half-wave's read fall in distinct banks for every tap.  Partial sums per workgroup are
// added in a fixed order by conv3x3_wgrad_reduce.  With at most 16 input channels (SPLIT) there is one
// ci tile, and the four waves of a co half share out the tile's rows instead; each keeps its sums
// where the other ci tiles' would be.
// CUT: some tile reaches past the image.  Its pixels there have a zero output gradient, but those in the
// row below the image and the column right of it meet input inside the image at ky = 0 and kx = 0, and
// zero times an infinite activation is not zero: such rows are left out, such a column's input is
// cleared.  An instance of its own: in the common one that took 0.8 us of 33 at 16 x 128 x 128, whose
// tiles are whole (103 x 54 x 140, 3 -> 64 channels, with it: 92.9 -> 95.8 us).
// Bound by the staging: a tile's 75 KB take longer to arrive and be stored than its MFMAs (a
// workgroup per CU, 2.8 TB/s).  Measured at 16 x 128 x 128, 64 -> 64 channels: 27 us, 714 TFLOP/s
// (118 us with one workgroup per (pixel chunk, tap) that wrote transposed copies of both operands to
// LDS); at 103 x 54 x 140, 3 -> 64 channels 77 us (97 us without SPLIT, 450 us before).
constexpr int kGTileH = 8, kGTileW = 32;
constexpr int kGHaloW = kGTileW + 2, kGHaloPix = (kGTileH + 2) * kGHaloW;
constexpr int kGThreads = 512;
constexpr int kGGroups = 256;  // most workgroups: one per CU, and as many partial sums
constexpr int kGYPer = kGTileH * kGTileW * 8 / kGThreads;              // 16-byte chunks of gout per thread
constexpr int kGXPer = (kGHaloPix * 8 + kGThreads - 1) / kGThreads;    // and of the halo

// 16-channel block t of a pixel in tile column r sits in block t ^ gswz(r) of the pixel's row
__device__ inline int gswz(int r) { return ((r >> 1) & 1) | ((r >> 2) & 2); }

typedef short s16x4 __attribute__((ext_vector_type(4)));
typedef uint32_t u32x4 __attribute__((ext_vector_type(4)));

// operand of 16 channels x 8 pixels per lane group: two transposed reads, pixels 0-3 and 4-7
__device__ inline bf16x8 read_tr(const bf16_t* lo, const bf16_t* hi) {
    typedef __attribute__((address_space(3))) s16x4 lds4;
    const s16x4 a = __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds4*)lo);
    const s16x4 b = __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds4*)hi);
    typedef short s16x8 __attribute__((ext_vector_type(8)));
    return __builtin_bit_cast(bf16x8, __builtin_shufflevector(a, b, 0, 1, 2, 3, 4, 5, 6, 7));
}

template <bool SPLIT, bool CUT>
__global__ void __launch_bounds__(kGThreads) conv3x3_wgrad_kernel(
    const bf16_t* __restrict__ in, const bf16_t* __restrict__ gout, float* __restrict__ part_w,
    float* __restrict__ part_b, int H, int W, int Cin, int Cout, int tiles_x, int tiles_y, int n_tiles) {
    __shared__ __attribute__((aligned(16))) bf16_t ly[kGTileH * kGTileW * 64];
    __shared__ __attribute__((aligned(16))) bf16_t lx[kGHaloPix * 64];
    const int tid = threadIdx.x, lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int m = lane & 15, g = lane >> 4;
    constexpr int kRows = SPLIT ? kGTileH / 4 : kGTileH;  // tile rows of a wave, from row0
    const int slot = wave & 3, co_h = wave >> 2;
    const int ci_t = SPLIT ? 0 : slot, row0 = SPLIT ? slot * kRows : 0;
    const int n_ci = (Cin + 15) / 16, n_co = (Cout + 15) / 16;
    // blocks that hold no channel are neither staged nor multiplied
    const int co_tiles = ci_t < n_ci ? min(max(n_co - 2 * co_h, 0), 2) : 0;
    const bool vec_y = (Cout & 7) == 0, vec_x = (Cin & 7) == 0;
    auto load8 = [&](const bf16_t* base, int C, int c0, bool vec) {
        bf16x8 v = zero8();
        if (vec) {
            if (c0 < C) v = *reinterpret_cast<const bf16x8*>(base + c0);
        } else {
#pragma unroll
            for (int e = 0; e < 8; ++e)
                if (c0 + e < C) v[e] = base[c0 + e];
        }
        return v;
    };
    bf16x8 py[kGYPer], px[kGXPer];
    auto fetch = [&](int tile) {
        const int tx0 = (tile % tiles_x) * kGTileW, ty0 = ((tile / tiles_x) % tiles_y) * kGTileH;
        const size_t img = (size_t)(tile / (tiles_x * tiles_y)) * H * W;
#pragma unroll
        for (int p = 0; p < kGYPer; ++p) {
            const int e = tid + p * kGThreads, c = e & 7, pix = e >> 3;
            const int yy = ty0 + pix / kGTileW, xx = tx0 + pix % kGTileW;
            py[p] = (c < 2 * n_co && yy < H && xx < W) ? load8(gout + (img + (size_t)yy * W + xx) * Cout, Cout, 8 * c, vec_y)
                                                       : zero8();
        }
#pragma unroll
        for (int p = 0; p < kGXPer; ++p) {
            const int e = tid + p * kGThreads, c = e & 7, pix = e >> 3;
            const int yy = ty0 + pix / kGHaloW - 1, xx = tx0 + pix % kGHaloW - 1;
            px[p] = (pix < kGHaloPix && c < 2 * n_ci && (unsigned)yy < (unsigned)H && (unsigned)xx < (unsigned)W)
                        ? load8(in + (img + (size_t)yy * W + xx) * Cin, Cin, 8 * c, vec_x)
                        : zero8();
        }
    };
    auto store = [&]() {
#pragma unroll
        for (int p = 0; p < kGYPer; ++p) {
            const int e = tid + p * kGThreads, c = e & 7, pix = e >> 3;
            *reinterpret_cast<bf16x8*>(&ly[pix * 64 + (((c >> 1) ^ gswz(pix % kGTileW)) << 4) + (c & 1) * 8]) = py[p];
        }
#pragma unroll
        for (int p = 0; p < kGXPer; ++p) {
            const int e = tid + p * kGThreads, c = e & 7, pix = e >> 3;
            if (pix < kGHaloPix)
                *reinterpret_cast<bf16x8*>(&lx[pix * 64 + (((c >> 1) ^ gswz(pix % kGHaloW)) << 4) + (c & 1) * 8]) = px[p];
        }
    };
    // this lane's addresses in a tile row: pixel 8 g + m / 4 (+ 4, + dx), channels 4 (m % 4) .. +3
    int ay[2][2], ax[3][2];  // [co tile | dx][pixel half]
#pragma unroll
    for (int h = 0; h < 2; ++h) {
        const int r = 8 * g + (m >> 2) + 4 * h;
#pragma unroll
        for (int t = 0; t < 2; ++t) ay[t][h] = (row0 * kGTileW + r) * 64 + (((2 * co_h + t) ^ gswz(r)) << 4) + (m & 3) * 4;
#pragma unroll
        for (int d = 0; d < 3; ++d) ax[d][h] = (row0 * kGHaloW + r + d) * 64 + ((ci_t ^ gswz(r + d)) << 4) + (m & 3) * 4;
    }
    f32x4 acc[9][2], accb[2];
#pragma unroll
    for (int k = 0; k < 9; ++k)
#pragma unroll
        for (int t = 0; t < 2; ++t) acc[k][t] = f32x4{0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll
    for (int t = 0; t < 2; ++t) accb[t] = f32x4{0.0f, 0.0f, 0.0f, 0.0f};
    bf16x8 ones;
#pragma unroll
    for (int e = 0; e < 8; ++e) ones[e] = (bf16_t)1.0f;

    int tile = blockIdx.x;
    fetch(tile);
    while (tile < n_tiles) {
        int n_rows = kRows;
        u32x4 keep = {};
        if constexpr (CUT) {
            n_rows = min(H - ((tile / tiles_x) % tiles_y) * kGTileH - row0, kRows);
            const int past = W - (tile % tiles_x) * kGTileW;  // first tile column past the image
#pragma unroll
            for (int e = 0; e < 4; ++e)
                keep[e] = 8 * g + 2 * e == (past & ~1) ? ((past & 1) ? 0x0000ffffu : 0xffff0000u) : ~0u;
        }
        __syncthreads();  // every wave has read the previous tile
        store();
        __syncthreads();
        tile += gridDim.x;
        if (tile < n_tiles) fetch(tile);
        // x of halo row y at kx = d
        auto read_x = [&](int y, int d) {
            const bf16x8 v = read_tr(&lx[y * kGHaloW * 64 + ax[d][0]], &lx[y * kGHaloW * 64 + ax[d][1]]);
            return CUT && d == 0 ? __builtin_bit_cast(bf16x8, __builtin_bit_cast(u32x4, v) & keep) : v;
        };
        if (co_tiles) {
            bf16x8 b[3][3];  // [halo row % 3][dx]
#pragma unroll
            for (int y = 0; y < 2; ++y)
#pragma unroll
                for (int d = 0; d < 3; ++d) b[y][d] = read_x(y, d);
#pragma unroll
            for (int y = 0; y < kRows; ++y) {
                if (CUT && y >= n_rows) break;
                bf16x8 a[2];
#pragma unroll
                for (int t = 0; t < 2; ++t)
                    a[t] = read_tr(&ly[y * kGTileW * 64 + ay[t][0]], &ly[y * kGTileW * 64 + ay[t][1]]);
#pragma unroll
                for (int d = 0; d < 3; ++d) b[(y + 2) % 3][d] = read_x(y + 2, d);
#pragma unroll
                for (int dy = 0; dy < 3; ++dy)
#pragma unroll
                    for (int d = 0; d < 3; ++d)
#pragma unroll
                        for (int t = 0; t < 2; ++t)
                            acc[3 * dy + d][t] =
                                __builtin_amdgcn_mfma_f32_16x16x32_bf16(a[t], b[(y + dy) % 3][d], acc[3 * dy + d][t], 0, 0, 0);
                if (ci_t == 0)
#pragma unroll
                    for (int t = 0; t < 2; ++t) accb[t] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(a[t], ones, accb[t], 0, 0, 0);
            }
        }
    }
    // lane (m, g) holds rows (co) 4 g .. 4 g + 3 of column (ci) m of each 16 x 16 block
    float* pw = part_w + (size_t)blockIdx.x * 9 * kMaxCout * kMaxCout;
#pragma unroll
    for (int k = 0; k < 9; ++k)
#pragma unroll
        for (int t = 0; t < 2; ++t)
#pragma unroll
            for (int r = 0; r < 4; ++r)
                if (t < co_tiles)
                    pw[(k * kMaxCout + 32 * co_h + 16 * t + 4 * g + r) * kMaxCout + 16 * slot + m] = acc[k][t][r];
    if (ci_t == 0 && m == 0)
#pragma unroll
        for (int t = 0; t < 2; ++t)
#pragma unroll
            for (int r = 0; r < 4; ++r)
                part_b[((size_t)blockIdx.x * 4 + slot) * kMaxCout + 32 * co_h + 16 * t + 4 * g + r] = accb[t][r];
}

// grad_w[co][tap][ci] = sum over the workgroups' partial sums (fixed order); grad_b[co] likewise.
// One workgroup per (co, tap) row and a quarter of the partial sums per wave, so that the reads of a
// partial sum's row are one 256-byte run; with slots = 4 that row holds the sums of the four row
// shares, 16 channels each.  7 us for 256 partial sums at 64 -> 64 channels (60 us for 128 with a
// thread per output and the partial sums one after the other).
__global__ void __launch_bounds__(256) conv3x3_wgrad_reduce(const float* __restrict__ part_w, const float* __restrict__ part_b,
                                                            float* __restrict__ grad_w, float* __restrict__ grad_b, int n_parts,
                                                            int Cin, int Cout, int slots) {
    __shared__ float sums[4][64];
    const int ci = threadIdx.x & 63, w = threadIdx.x >> 6;
    const int row = blockIdx.x;  // co * 9 + tap, and Cout * 9 for the bias
    const bool bias = row == Cout * 9;
    const int co = row / 9, tap = row - 9 * co;
    const float* src = bias ? part_b + ci : part_w + ((size_t)tap * kMaxCout + co) * kMaxCout + ci;
    const size_t step = bias ? 4 * kMaxCout : 9 * kMaxCout * kMaxCout;
    const int n = bias ? Cout : Cin;
    const int per = (n_parts + 3) / 4, c1 = min((w + 1) * per, n_parts);
    float s = 0.0f;
    if (ci < n || (!bias && slots > 1)) {
#pragma unroll 8
        for (int c = w * per; c < c1; ++c) s += src[(size_t)c * step];
        for (int k = 1; bias && k < slots; ++k)
#pragma unroll 8
            for (int c = w * per; c < c1; ++c) s += src[(size_t)c * step + k * kMaxCout];
    }
    sums[w][ci] = s;
    __syncthreads();
    if (w || ci >= n) return;
    float total = (sums[0][ci] + sums[1][ci]) + (sums[2][ci] + sums[3][ci]);
    for (int k = 1; !bias && k < slots; ++k)
        total += (sums[0][16 * k + ci] + sums[1][16 * k + ci]) + (sums[2][16 * k + ci] + sums[3][16 * k + ci]);
    if (bias)
        grad_b[ci] = total;
    else
        grad_w[(size_t)row * Cin + ci] = total;
}

// Weights of the input-gradient convolution: out[ci][2 - ky][2 - kx][co] = w[co][ky][kx][ci]
__global__ void __launch_bounds__(256) conv3x3_flip_kernel(const bf16_t* __restrict__ w, bf16_t* __restrict__ out, int Cin,
                                                           int Cout) {
    const int i = blockIdx.x * 256 + threadIdx.x;  // index into out
    if (i >= Cin * 9 * Cout) return;
    const int co = i % Cout, tap = (i / Cout) % 9, ci = i / (9 * Cout);
    out[i] = w[(co * 9 + 8 - tap) * Cin + ci];
}

// tiles and workgroups of a weight gradient: as many tiles for each workgroup, at most one per CU
struct WgradGrid {
    int tiles_x, tiles_y;
    long long tiles;
    int groups;
};

WgradGrid wgrad_grid(int n, int h, int w) {
    WgradGrid r;
    r.tiles_x = (w + kGTileW - 1) / kGTileW;
    r.tiles_y = (h + kGTileH - 1) / kGTileH;
    r.tiles = (long long)n * r.tiles_x * r.tiles_y;
    const long long each = (r.tiles + kGGroups - 1) / kGGroups;
    r.groups = (int)((r.tiles + each - 1) / each);
    return r;
}

}  // namespace

extern "C" {

int ctr_conv3x3_bf16_forward(const void* in, const void* weight, const float* bias,
                             const void* residual, void* out, int n, int h, int w, int cin, int cout,
                             int relu, void* stream) {
    if (!in || !weight || !out) return CTR_ERR_INVALID;
    if (n <= 0 || h <= 0 || w <= 0 || cin <= 0 || cout <= 0 || cout > kMaxCout) return CTR_ERR_INVALID;
    const long long P = (long long)n * h * w;
    if (P * (cin > cout ? cin : cout) >= 2147483647LL) return CTR_ERR_INVALID;
    const long long blocks = (P + kConvWaves * kPxPerWave - 1) / (kConvWaves * kPxPerWave);
    hipStream_t s = (hipStream_t)stream;
    const bf16_t* x = (const bf16_t*)in;
    const bf16_t* wt = (const bf16_t*)weight;
    const bf16_t* r = (const bf16_t*)residual;
    bf16_t* y = (bf16_t*)out;
    // the generic kernel stores four channels at a time when rows allow it
    const int vec = (cout % 4 == 0) && ((reinterpret_cast<uintptr_t>(out) | reinterpret_cast<uintptr_t>(residual)) & 7) == 0;
    if (cin == 64 && (cout == 64 || (cout <= 16 && !r))) {
        const int tiles_x = (w + kPTileW - 1) / kPTileW, tiles_y = (h + kPTileH - 1) / kPTileH;
        const long long n_tiles = (long long)n * tiles_x * tiles_y;
        if (n_tiles >= 2147483647LL) return CTR_ERR_INVALID;
        int dev = 0, n_cu = 0;
        if (hipGetDevice(&dev) != hipSuccess ||
            hipDeviceGetAttribute(&n_cu, hipDeviceAttributeMultiprocessorCount, dev) != hipSuccess)
            return CTR_ERR_HIP;
        const int grid = (int)std::min<long long>(n_tiles, std::max(n_cu, 1));
        auto launch = [&](auto kern) {
            hipLaunchKernelGGL(kern, dim3(grid), dim3(kPThreads), 0, s, x, wt, bias, r, y, h, w, cout, tiles_x,
                               tiles_y, (int)n_tiles);
        };
        if (cout <= 16)
            relu ? launch(conv3x3_fwd_persistent_kernel<true, false, 1>) : launch(conv3x3_fwd_persistent_kernel<false, false, 1>);
        else if (relu)
            r ? launch(conv3x3_fwd_persistent_kernel<true, true, 4>) : launch(conv3x3_fwd_persistent_kernel<true, false, 4>);
        else
            r ? launch(conv3x3_fwd_persistent_kernel<false, true, 4>) : launch(conv3x3_fwd_persistent_kernel<false, false, 4>);
    } else if (cin <= 4) {
        const int tiles_x = (w + kSTileW - 1) / kSTileW, tiles_y = (h + kSTileH - 1) / kSTileH;
        const long long n_tiles = (long long)n * tiles_x * tiles_y;
        if (n_tiles >= 2147483647LL) return CTR_ERR_INVALID;
        int dev = 0, n_cu = 0;
        if (hipGetDevice(&dev) != hipSuccess ||
            hipDeviceGetAttribute(&n_cu, hipDeviceAttributeMultiprocessorCount, dev) != hipSuccess)
            return CTR_ERR_HIP;
        // persistent: eight workgroups per CU walk the tiles
        const int grid = (int)std::min<long long>(n_tiles, 8LL * std::max(n_cu, 1));
        hipLaunchKernelGGL(conv3x3_fwd_small_cin_kernel, dim3(grid), dim3(256), 0, s, x, wt, bias, r, y,
                           h, w, cin, cout, relu, vec, tiles_x, tiles_y, (int)n_tiles);
    } else if (cin % 32 == 0) {
        hipLaunchKernelGGL(HIP_KERNEL_NAME(conv3x3_fwd_kernel<true>), dim3((unsigned)blocks), dim3(256),
                           0, s, x, wt, bias, r, y, n, h, w, cin, cout, relu, vec);
    } else {
        hipLaunchKernelGGL(HIP_KERNEL_NAME(conv3x3_fwd_kernel<false>), dim3((unsigned)blocks), dim3(256),
                           0, s, x, wt, bias, r, y, n, h, w, cin, cout, relu, vec);
    }
    return hipGetLastError() == hipSuccess ? CTR_OK : CTR_ERR_HIP;
}

size_t ctr_conv3x3_bf16_wgrad_workspace_bytes(int n, int h, int w, int cin, int cout) {
    (void)cin;
    (void)cout;
    if (n <= 0 || h <= 0 || w <= 0) return 0;
    return (size_t)wgrad_grid(n, h, w).groups * (9 * kMaxCout * kMaxCout + 4 * kMaxCout) * sizeof(float);
}

int ctr_conv3x3_bf16_wgrad(const void* in, const void* grad_out, float* grad_weight, float* grad_bias,
                           int n, int h, int w, int cin, int cout, void* workspace,
                           size_t workspace_bytes, void* stream) {
    if (!in || !grad_out || !grad_weight || !workspace) return CTR_ERR_INVALID;
    if (n <= 0 || h <= 0 || w <= 0 || cin <= 0 || cout <= 0 || cin > kMaxCout || cout > kMaxCout)
        return CTR_ERR_INVALID;
    const long long P = (long long)n * h * w;
    if (P * kMaxCout >= 2147483647LL) return CTR_ERR_INVALID;
    if (workspace_bytes < ctr_conv3x3_bf16_wgrad_workspace_bytes(n, h, w, cin, cout)) return CTR_ERR_WORKSPACE;
    const WgradGrid wg = wgrad_grid(n, h, w);
    if (wg.tiles >= 2147483647LL - kGGroups) return CTR_ERR_INVALID;
    float* part_w = (float*)workspace;
    float* part_b = part_w + (size_t)wg.groups * 9 * kMaxCout * kMaxCout;
    hipStream_t s = (hipStream_t)stream;
    auto launch = [&](auto kernel) {
        hipLaunchKernelGGL(kernel, dim3(wg.groups), dim3(kGThreads), 0, s, (const bf16_t*)in, (const bf16_t*)grad_out,
                           part_w, part_b, h, w, cin, cout, wg.tiles_x, wg.tiles_y, (int)wg.tiles);
    };
    const bool split = cin <= 16, cut = h % kGTileH != 0 || w % kGTileW != 0;
    if (cut)
        split ? launch(conv3x3_wgrad_kernel<true, true>) : launch(conv3x3_wgrad_kernel<false, true>);
    else
        split ? launch(conv3x3_wgrad_kernel<true, false>) : launch(conv3x3_wgrad_kernel<false, false>);
    if (hipGetLastError() != hipSuccess) return CTR_ERR_HIP;
    hipLaunchKernelGGL(conv3x3_wgrad_reduce, dim3(cout * 9 + (grad_bias ? 1 : 0)), dim3(256), 0, s, part_w, part_b,
                       grad_weight, grad_bias, wg.groups, cin, cout, split ? 4 : 1);
    return hipGetLastError() == hipSuccess ? CTR_OK : CTR_ERR_HIP;
}

// flipped weights of the input-gradient convolution, then the weight gradient's workspace
static size_t flipped_bytes(int cin, int cout) { return ((size_t)cin * 9 * cout * sizeof(bf16_t) + 255) / 256 * 256; }

size_t ctr_conv3x3_bf16_backward_workspace_bytes(int n, int h, int w, int cin, int cout) {
    if (n <= 0 || h <= 0 || w <= 0 || cin <= 0 || cout <= 0 || cin > kMaxCout || cout > kMaxCout) return 0;
    return flipped_bytes(cin, cout) + ctr_conv3x3_bf16_wgrad_workspace_bytes(n, h, w, cin, cout);
}

int ctr_conv3x3_bf16_backward(const void* in, const void* weight, const void* grad_out, void* grad_in, float* grad_weight,
                              float* grad_bias, int n, int h, int w, int cin, int cout, void* workspace,
                              size_t workspace_bytes, void* stream) {
    if (!in || !grad_out || !grad_weight || !workspace || (grad_in && !weight)) return CTR_ERR_INVALID;
    if (n <= 0 || h <= 0 || w <= 0 || cin <= 0 || cout <= 0 || cin > kMaxCout || cout > kMaxCout) return CTR_ERR_INVALID;
    if ((long long)n * h * w * kMaxCout >= 2147483647LL) return CTR_ERR_INVALID;
    if (workspace_bytes < ctr_conv3x3_bf16_backward_workspace_bytes(n, h, w, cin, cout)) return CTR_ERR_WORKSPACE;
    const size_t flipped = flipped_bytes(cin, cout);
    if (grad_in) {
        bf16_t* wf = (bf16_t*)workspace;
        hipLaunchKernelGGL(conv3x3_flip_kernel, dim3((cin * 9 * cout + 255) / 256), dim3(256), 0, (hipStream_t)stream,
                           (const bf16_t*)weight, wf, cin, cout);
        if (hipGetLastError() != hipSuccess) return CTR_ERR_HIP;
        const int st = ctr_conv3x3_bf16_forward(grad_out, wf, nullptr, nullptr, grad_in, n, h, w, cout, cin, 0, stream);
        if (st != CTR_OK) return st;
    }
    return ctr_conv3x3_bf16_wgrad(in, grad_out, grad_weight, grad_bias, n, h, w, cin, cout, (char*)workspace + flipped,
                                  workspace_bytes - flipped, stream);
}

}  // extern "C"
