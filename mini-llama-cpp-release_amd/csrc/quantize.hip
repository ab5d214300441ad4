// Device-side weight quantizer (f32 -> Q8_0 / Q4_0 / Q4_1 blocks) and the
// synthetic normal generator used by benchmarks.
//
// The quantizers produce the same bytes as the reference's host routines:
//   quantize_to_q8_0  src/quant.cpp:112-170
//   quantize_to_q4_0  src/quant.cpp:207-270
//   Q4_1              tests/test_cuda_quant.cpp:129-180 (the only Q4_1 quantizer
//                     the reference has; its parity tests use it)
// Every step is an IEEE f32 operation with one rounding (|v|, max, a / 127,
// 1 / d, v * inv, its sum with 8, (v - m) * inv) or integer work, so the device result
// matches the host bit for bit: hipcc divides with correct rounding (no fast-math),
// roundf rounds half away from zero like std::round, and nothing is contracted into an
// fma (contract(off) below): Q4_0's v * inv + 8 as one would move codes whose product
// rounds onto a tie, 1e-7 of them for f32 normal weights, 1e-4 for bf16 ones, 8e-4 for
// integers up to 100.  The scale is encoded with the reference's binary16 rule (round half
// up in magnitude at the first dropped bit, overflow and NaN to Inf,
// src/quant.cpp:19-55), not the hardware cvt.
//
// Four lanes quantize one block; a lane reads two float4s where every row is 16-byte
// aligned, element by element otherwise.

#include "mlq_kernels.h"

#include <hip/hip_runtime.h>

#include <cstdint>

namespace mlq {
namespace {

__device__ __forceinline__ uint32_t f32_bits(float v) { return __builtin_bit_cast(uint32_t, v); }

// f32 -> binary16 with the reference's rounding (see header comment).
__device__ uint16_t half_round_up(float value) {
    const uint32_t u = f32_bits(value);
    const uint32_t sign = (u >> 16) & 0x8000u;
    const int e = static_cast<int>((u >> 23) & 0xffu) - 112;
    const uint32_t frac = u & 0x7fffffu;
    if (e >= 31) return static_cast<uint16_t>(sign | 0x7c00u);
    if (e <= 0) {
        if (e < -10) return static_cast<uint16_t>(sign);
        uint32_t sig = (frac | 0x800000u) >> (1 - e);
        sig += (sig & 0x1000u) << 1;  // +0x2000 when the first dropped bit is set
        return static_cast<uint16_t>(sign | (sig >> 13));
    }
    uint32_t sig = frac + ((frac & 0x1000u) << 1);
    int eh = e;
    if (sig & 0x800000u) {
        sig = 0;
        if (++eh >= 31) return static_cast<uint16_t>(sign | 0x7c00u);
    }
    return static_cast<uint16_t>(sign | (static_cast<uint32_t>(eh) << 10) | (sig >> 13));
}

__device__ __forceinline__ float half_value(uint16_t h) {
    return (float)__builtin_bit_cast(_Float16, h);  // exact (v_cvt_f32_f16)
}

__device__ __forceinline__ int round_int(float v) { return static_cast<int>(roundf(v)); }

template <int QT> struct QB;
template <> struct QB<1> { static constexpr int BB = 34; };
template <> struct QB<2> { static constexpr int BB = 18; };
template <> struct QB<3> { static constexpr int BB = 20; };

// The other lane of the quad that differs in bit 0 (CTRL 0xB1) or bit 1 (0x4E).
template <int CTRL>
__device__ __forceinline__ float quad_peer(float v) {
    return __builtin_bit_cast(
        float, __builtin_amdgcn_mov_dpp(__builtin_bit_cast(int, v), CTRL, 0xf, 0xf, true));
}

// Largest of a quad's values (none is NaN).
__device__ __forceinline__ float quad_max(float v) {
    float o = quad_peer<0xB1>(v);
    v = (v < o) ? o : v;
    o = quad_peer<0x4E>(v);
    return (v < o) ? o : v;
}

// Smallest of a quad's values (none is NaN); of equal ones the lowest lane's, as a
// scan in element order keeps it (it decides the sign of a zero).
__device__ __forceinline__ float quad_first_min(float v, int l) {
    float o = quad_peer<0xB1>(v);
    v = (l & 1) ? ((v < o) ? v : o) : ((o < v) ? o : v);
    o = quad_peer<0x4E>(v);
    return (l & 2) ? ((v < o) ? v : o) : ((o < v) ? o : v);
}

constexpr int kQuantThreads = 256;
constexpr int kQuantPasses = 2;
constexpr int kQuantBlocks = kQuantThreads / 4 * kQuantPasses;  // blocks per workgroup

// How a lane finds its elements: rows of whole blocks back to back (no division),
// rows whose float4s are aligned and whole or absent, any rows.
enum Rows { kWhole, kVector, kElement };

// Bound: HBM (4 * row_len read, blocks written).  Four lanes take a block, lane l its
// elements 4l..4l+3 and 16+4l..16+4l+3: both are one float4, a Q4 byte's two nibbles
// are in one lane, and the block's extremes fold in two quad permutes.  The packed
// blocks of the workgroup (kQuantBlocks of them, a multiple of 16 bytes) gather in LDS
// and leave in 16-byte stores.  One thread per block
// (128-byte strides between lanes, 16-bit stores) / this, us: 11008 x 4096 Q8_0 46.3 /
// 41.2 (5.5 TB/s, four fifths of it reads; a copy, half writes, runs at 5.1), Q4_0 39.2 / 38.2, Q4_1 40.4 / 40.4; 10000 x 2500 Q8_0
// 29.0 / 26.3; 16000 x 2051 Q4_0 69.7 / 58.7; 3000 x 896 Q4_0 5.2 / 4.1.
template <int QT, Rows ROWS>
__global__ __launch_bounds__(kQuantThreads) void quantize_kernel(const float* __restrict__ src,
                                                                 long long total, int row_len,
                                                                 uint8_t* __restrict__ dst,
                                                                 bool wide) {
#pragma clang fp contract(off)
    constexpr int BB = QB<QT>::BB;
    static_assert(kQuantBlocks * BB % 16 == 0, "a workgroup's blocks start 16-byte aligned");
    __shared__ alignas(16) uint16_t packed[kQuantBlocks * BB / 2];
    const int t = threadIdx.x;
    const int l = t & 3;
    const long long first = static_cast<long long>(blockIdx.x) * kQuantBlocks;
    const int here = static_cast<int>(min(static_cast<long long>(kQuantBlocks), total - first));

    float v[kQuantPasses][8];  // elements 4l.., then 16 + 4l..
    int len[kQuantPasses];
#pragma unroll
    for (int s = 0; s < kQuantPasses; ++s) {
        // lanes past the last block repeat it (their result is not stored)
        const int local = min(s * (kQuantThreads / 4) + (t >> 2), here - 1);
        if (ROWS == kWhole) {
            const float4* p = reinterpret_cast<const float4*>(src + (first + local) * kQK);
            len[s] = kQK;
            const float4 a = p[l];
            const float4 b = p[4 + l];
            v[s][0] = a.x, v[s][1] = a.y, v[s][2] = a.z, v[s][3] = a.w;
            v[s][4] = b.x, v[s][5] = b.y, v[s][6] = b.z, v[s][7] = b.w;
        } else {
            const unsigned nb = (static_cast<unsigned>(row_len) + kQK - 1) / kQK;
            const unsigned at = static_cast<unsigned>(first % nb) + local;
            const float* p = src + static_cast<size_t>(first / nb + at / nb) * row_len + at % nb * kQK;
            len[s] = min(kQK, row_len - static_cast<int>(at % nb) * kQK);
#pragma unroll
            for (int h = 0; h < 2; ++h) {
                const int e = 16 * h + 4 * l;
                if (ROWS == kVector) {
                    float4 f = make_float4(0.0f, 0.0f, 0.0f, 0.0f);
                    if (e < len[s]) f = *reinterpret_cast<const float4*>(p + e);
                    v[s][4 * h] = f.x, v[s][4 * h + 1] = f.y, v[s][4 * h + 2] = f.z, v[s][4 * h + 3] = f.w;
                } else {
#pragma unroll
                    for (int c = 0; c < 4; ++c) v[s][4 * h + c] = (e + c < len[s]) ? p[e + c] : 0.0f;
                }
            }
        }
    }

#pragma unroll
    for (int s = 0; s < kQuantPasses; ++s) {
        uint16_t* out = packed + (s * (kQuantThreads / 4) + (t >> 2)) * (BB / 2);
        if (QT == 1 || QT == 2) {
            float amax = 0.0f;  // elements past the row are 0
#pragma unroll
            for (int i = 0; i < 8; ++i) {
                const float a = fabsf(v[s][i]);
                amax = (a > amax) ? a : amax;
            }
            amax = quad_max(amax);
            const bool some = amax > 0.0f;  // else the block is all zero bytes
            const uint16_t dh = some ? half_round_up(amax / (QT == 1 ? 127.0f : 7.0f)) : 0;
            const float dq = half_value(dh);
            const float inv = (dq == 0.0f) ? 0.0f : 1.0f / dq;
            if (l == 0) out[0] = dh;
            if (QT == 1) {
                int q[8];
#pragma unroll
                for (int i = 0; i < 8; ++i) {
                    q[i] = round_int(v[s][i] * inv);
                    q[i] = some ? max(-127, min(127, q[i])) & 0xff : 0;
                }
#pragma unroll
                for (int h = 0; h < 2; ++h) {
                    out[1 + 8 * h + 2 * l] = static_cast<uint16_t>(q[4 * h] | (q[4 * h + 1] << 8));
                    out[2 + 8 * h + 2 * l] = static_cast<uint16_t>(q[4 * h + 2] | (q[4 * h + 3] << 8));
                }
            } else {
                int q[4];
#pragma unroll
                for (int j = 0; j < 4; ++j) {
                    const int qlo = max(0, min(15, round_int(v[s][j] * inv + 8.0f)));
                    const int qhi = max(0, min(15, round_int(v[s][4 + j] * inv + 8.0f)));
                    q[j] = some ? qlo | (qhi << 4) : 0;
                }
                out[1 + 2 * l] = static_cast<uint16_t>(q[0] | (q[1] << 8));
                out[2 + 2 * l] = static_cast<uint16_t>(q[2] | (q[3] << 8));
            }
        } else {
            // std::min / std::max semantics in element order: the first of equal
            // values stays, NaN never enters.
            float lo[2] = {__builtin_inff(), __builtin_inff()};
            float hi = -__builtin_inff();
#pragma unroll
            for (int i = 0; i < 8; ++i) {
                if (16 * (i >> 2) + 4 * l + (i & 3) < len[s]) {
                    lo[i >> 2] = (v[s][i] < lo[i >> 2]) ? v[s][i] : lo[i >> 2];
                    hi = (hi < v[s][i]) ? v[s][i] : hi;
                }
            }
            lo[0] = quad_first_min(lo[0], l);
            lo[1] = quad_first_min(lo[1], l);
            const float mn = (lo[1] < lo[0]) ? lo[1] : lo[0];
            const float range = quad_max(hi) - mn;
            const bool some = range > 0.0f;
            const uint16_t dh = some ? half_round_up(range / 15.0f) : 0;
            const uint16_t mh = half_round_up((!some && mn == __builtin_inff()) ? 0.0f : mn);
            const float dq = half_value(dh);
            const float mq = half_value(mh);
            const float inv = (dq == 0.0f) ? 0.0f : 1.0f / dq;
            if (l == 0) {
                out[0] = dh;
                out[1] = mh;
            }
            int q[4];
#pragma unroll
            for (int j = 0; j < 4; ++j) {
                int q0 = (4 * l + j < len[s]) ? round_int((v[s][j] - mq) * inv) : 0;
                int q1 = (16 + 4 * l + j < len[s]) ? round_int((v[s][4 + j] - mq) * inv) : 0;
                q0 = max(0, min(15, q0));
                q1 = max(0, min(15, q1));
                q[j] = some ? q0 | (q1 << 4) : 0;
            }
            out[2 + 2 * l] = static_cast<uint16_t>(q[0] | (q[1] << 8));
            out[3 + 2 * l] = static_cast<uint16_t>(q[2] | (q[3] << 8));
        }
    }
    __syncthreads();

    // `wide`: dst is 16-byte aligned; else, and for the last workgroup's remainder, 16-bit halves.
    uint8_t* base = dst + static_cast<size_t>(first) * BB;
    const int bytes = here * BB;
    const int units = wide ? bytes / 16 : 0;
    for (int u = t; u < units; u += kQuantThreads) {
        reinterpret_cast<uint4*>(base)[u] = reinterpret_cast<const uint4*>(packed)[u];
    }
    for (int h = units * 8 + t; h < bytes / 2; h += kQuantThreads) {
        reinterpret_cast<uint16_t*>(base)[h] = packed[h];
    }
}

// splitmix64 (Steele, Lea, Flood 2014) on the element pair index, Box-Muller
// on the two 32-bit halves' top 24 bits.
__device__ __forceinline__ uint64_t splitmix64(uint64_t z) {
    z += 0x9e3779b97f4a7c15ull;
    z = (z ^ (z >> 30)) * 0xbf58476d1ce4e5b9ull;
    z = (z ^ (z >> 27)) * 0x94d049bb133111ebull;
    return z ^ (z >> 31);
}

__global__ __launch_bounds__(256) void fill_normal_kernel(float* __restrict__ dst, size_t n,
                                                          uint64_t seed, float mean,
                                                          float stddev) {
    const size_t pair = static_cast<size_t>(blockIdx.x) * blockDim.x + threadIdx.x;
    const size_t i0 = pair * 2;
    if (i0 >= n) return;
    const uint64_t h = splitmix64(seed ^ splitmix64(pair));
    const float u1 = (static_cast<float>(static_cast<uint32_t>(h >> 40)) + 1.0f) * (1.0f / 16777217.0f);
    const float u2 = static_cast<float>(static_cast<uint32_t>(h >> 8) & 0xffffffu) * (1.0f / 16777216.0f);
    const float rad = sqrtf(-2.0f * logf(u1));
    float s, c;
    sincosf(6.283185307179586f * u2, &s, &c);
    dst[i0] = mean + stddev * rad * c;
    if (i0 + 1 < n) dst[i0 + 1] = mean + stddev * rad * s;
}

template <int QT>
hipError_t launch_q(const float* src, int rows, int row_len, void* dst, hipStream_t stream) {
    const long long n = static_cast<long long>(rows) * ((static_cast<long long>(row_len) + kQK - 1) / kQK);
    const dim3 grid(static_cast<unsigned>((n + kQuantBlocks - 1) / kQuantBlocks));
    uint8_t* out = static_cast<uint8_t*>(dst);
    const bool wide = (reinterpret_cast<uintptr_t>(dst) & 15u) == 0;
    // A float4 needs its 16-byte alignment: the source's and, in every row, the length's.
    const bool vec = (reinterpret_cast<uintptr_t>(src) & 15u) == 0 && row_len % 4 == 0;
    if (vec && row_len % kQK == 0) {
        quantize_kernel<QT, kWhole><<<grid, kQuantThreads, 0, stream>>>(src, n, row_len, out, wide);
    } else if (vec) {
        quantize_kernel<QT, kVector><<<grid, kQuantThreads, 0, stream>>>(src, n, row_len, out, wide);
    } else {
        quantize_kernel<QT, kElement><<<grid, kQuantThreads, 0, stream>>>(src, n, row_len, out, wide);
    }
    return hipGetLastError();
}

}  // namespace

hipError_t launch_quantize(int qtype, const float* src, int rows, int row_len, void* dst,
                           hipStream_t stream) {
    switch (qtype) {
        case 1: return launch_q<1>(src, rows, row_len, dst, stream);
        case 2: return launch_q<2>(src, rows, row_len, dst, stream);
        case 3: return launch_q<3>(src, rows, row_len, dst, stream);
        default: return hipErrorInvalidValue;
    }
}

hipError_t launch_fill_normal(float* dst, size_t n, uint64_t seed, float mean, float stddev,
                              hipStream_t stream) {
    const size_t pairs = (n + 1) / 2;
    const size_t grid = (pairs + 255) / 256;
    hipLaunchKernelGGL(fill_normal_kernel, dim3(static_cast<unsigned>(grid)), dim3(256), 0, stream,
                       dst, n, seed, mean, stddev);
    return hipGetLastError();
}

}  // namespace mlq
