// The prefill GEMM's split x, written per token row by a workgroup of 256
// threads.  Shared by the GEMM's own split kernel (gemm.hip) and by decoder
// kernels that produce a GEMM input and write it split straight away
// (decoder.hip), so both give the same halves.
//
// Layout (token-major): xs [npad][nb][64 halves] = per block the 32 scaled
// elements' fp16 hi then lo, in the k order of the GEMM's weight fragments;
// bsum [npad][nb] = per block the f32 sum of the scaled elements (Q4_1's
// offset term); scale [npad] = the token's power-of-two scale s_n, chosen so that
// max|x_n| / s_n lies in [2^13, 2^14).
#pragma once

#include <hip/hip_runtime.h>

#include <cstddef>

namespace mlq {
namespace {

// An item is the eight elements of one fragment slot run: item i is slots
// 8 g .. 8 g + 7 of block i / 4, g = i % 4, so it leaves as one 16-byte hi and one
// 16-byte lo store, the four items of a block side by side.  (Sixteen consecutive
// elements per thread, the earlier split, left in 8-byte pieces 16 bytes apart:
// 512 x 4096 in the order of Q4_1's fragments 8.7 us, now 8.2.)
// Thread t holds items t + 256 c, c < kXsCache, so rows of up to 16 384 elements
// are split from registers.
constexpr int kXsCache = 8;

// First element of item i's two runs of four.
template <int QT>
__device__ __forceinline__ int xs_first(int i) {
    return 32 * (i >> 2) + (QT == 1 ? 8 : 4) * (i & 3);
}
template <int QT>
__device__ __forceinline__ constexpr int xs_second() {
    return QT == 1 ? 4 : 16;  // from the first run
}

typedef _Float16 xs_h8 __attribute__((ext_vector_type(8)));

// max |x| over the workgroup (every thread gets it); `red` is 4 floats of LDS.
__device__ __forceinline__ float xsplit_row_max(float mx, float* red) {
#pragma unroll
    for (int o = 32; o > 0; o >>= 1) mx = fmaxf(mx, __shfl_xor(mx, o, 64));
    if ((threadIdx.x & 63) == 0) red[threadIdx.x >> 6] = mx;
    __syncthreads();
    return fmaxf(fmaxf(red[0], red[1]), fmaxf(red[2], red[3]));
}

// Power-of-two scale of a row with max |x| = mx: inv = 1 / s, sc = s.
__device__ __forceinline__ void xsplit_scale(float mx, float& inv, float& sc) {
    inv = 1.0f;
    sc = 1.0f;
    if (mx > 0.0f && mx <= 3.0e38f) {
        int ex = 0;
        (void)frexpf(mx, &ex);  // mx in [2^(ex-1), 2^ex)
        const int e = min(126, max(-126, 14 - ex));
        inv = ldexpf(1.0f, e);
        sc = ldexpf(1.0f, -e);
    }
}

// Scales, splits and stores item i of token row n (v: its two runs).  Called by
// every lane (a block's four items are on adjacent lanes); items past the row
// store nothing.
template <int QT>
__device__ __forceinline__ void xsplit_emit_item(int n, int nb, int i, float (&v)[8], float inv,
                                                 _Float16* __restrict__ xs, float* __restrict__ bsum) {
#pragma unroll
    for (int k = 0; k < 8; ++k) v[k] *= inv;
    float sum = ((v[0] + v[1]) + (v[2] + v[3])) + ((v[4] + v[5]) + (v[6] + v[7]));
    auto add_lane = [](float s, int other) { return s + __builtin_bit_cast(float, other); };
    sum = add_lane(sum, __builtin_amdgcn_mov_dpp(__builtin_bit_cast(int, sum), 0xB1, 0xF, 0xF, true));  // lane ^ 1
    sum = add_lane(sum, __builtin_amdgcn_mov_dpp(__builtin_bit_cast(int, sum), 0x4E, 0xF, 0xF, true));  // lane ^ 2
    if (i >= 4 * nb) return;
    const int g = i & 3;
    const size_t b = static_cast<size_t>(n) * nb + (i >> 2);
    if (g == 0) bsum[b] = sum;
    xs_h8 hi, lo;
#pragma unroll
    for (int j = 0; j < 8; ++j) {
        // Q4 fragments take each run as elements 0, 2, 1, 3.
        const int k = QT == 1 ? j : (j & 4) + (((j & 1) << 1) | ((j >> 1) & 1));
        const _Float16 h = static_cast<_Float16>(v[k]);
        hi[j] = h;
        lo[j] = static_cast<_Float16>(v[k] - static_cast<float>(h));
    }
    _Float16* dst = xs + b * 64 + 8 * g;
    *reinterpret_cast<xs_h8*>(dst) = hi;
    *reinterpret_cast<xs_h8*>(dst + 32) = lo;
}

// The whole split of token row n from the values the workgroup holds (thread
// t: items t + 256 c in v[c], zeros past the row; 4 nb <= 256 C): the row's
// maximum, its scale (stored by thread 0) and every item.
template <int QT, int C>
__device__ __forceinline__ void xsplit_emit_row(int n, int nb, float (&v)[C][8], _Float16* __restrict__ xs,
                                                float* __restrict__ bsum, float* __restrict__ scale, float* red) {
    float mx = 0.0f;
#pragma unroll
    for (int c = 0; c < C; ++c)
#pragma unroll
        for (int i = 0; i < 8; ++i) mx = fmaxf(mx, fabsf(v[c][i]));
    mx = xsplit_row_max(mx, red);
    float inv, sc;
    xsplit_scale(mx, inv, sc);
    if (threadIdx.x == 0) scale[n] = sc;
    const int iters = (4 * nb + 255) / 256;  // uniform across the workgroup
#pragma unroll
    for (int c = 0; c < C; ++c)
        if (c < iters) xsplit_emit_item<QT>(n, nb, static_cast<int>(threadIdx.x) + 256 * c, v[c], inv, xs, bsum);
}

// One float4 of `p` into v[k .. k + 3].
__device__ __forceinline__ void xs_put4(float (&v)[8], int k, const float* p) {
    const float4 f = *reinterpret_cast<const float4*>(p);
    v[k] = f.x, v[k + 1] = f.y, v[k + 2] = f.z, v[k + 3] = f.w;
}

}  // namespace
}  // namespace mlq
