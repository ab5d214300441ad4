// Device forward ops behind the reference's op-by-op device interfaces
// (include/mini_llama/cuda_ops.h, cuda_attention.h, cuda_matmul.h): RMSNorm,
// SiLU, elementwise product and sum, softmax, embedding row lookup, RoPE
// (normal and NeoX pairing), single-token attention over a KV cache and an
// F32 matrix product.  Each op reads and writes device buffers the caller
// owns and is launched on the caller's stream; nothing here allocates.
//
// These are the small kernels of a decode step that the quantized linears
// surround.  They move kilobytes per call and are launch-bound, so each is one
// grid-stride or one-workgroup kernel: a single launch per op (the reference
// uses two or three: a separate sum / max pass and a normalisation pass).
// Arithmetic follows the reference's CPU ops (src/ops.cpp:19-79, 109-176) in
// f32, with the sums taken as wavefront trees instead of a serial loop.

#include "mlq_kernels.h"

#include <hip/hip_runtime.h>

#include <algorithm>
#include <cmath>
#include <cstdint>

namespace mlq {
namespace {

constexpr int kOpThreads = 256;
constexpr int kReduceThreads = 1024;
constexpr int kAttnWaves = 4;
constexpr int kMatTile = 16;
constexpr int kCoherent = 16;  // sc1: write through / read from the point of coherence (agent scope)

typedef uint32_t u32x4 __attribute__((ext_vector_type(4)));

__device__ __forceinline__ float wave_sum(float v) {
#pragma unroll
    for (int o = 32; o > 0; o >>= 1) v += __shfl_xor(v, o, 64);
    return v;
}

__device__ __forceinline__ float wave_max(float v) {
#pragma unroll
    for (int o = 32; o > 0; o >>= 1) v = fmaxf(v, __shfl_xor(v, o, 64));
    return v;
}

// Sum (MAX = false) or maximum over the workgroup; the result in every thread.
template <bool MAX>
__device__ __forceinline__ float block_reduce(float v) {
    __shared__ float part[kReduceThreads / 64];
    v = MAX ? wave_max(v) : wave_sum(v);
    __syncthreads();  // `part` may still be read by an earlier call
    if ((threadIdx.x & 63) == 0) part[threadIdx.x >> 6] = v;
    __syncthreads();
    float t = part[0];
    const int waves = static_cast<int>(blockDim.x >> 6);
    for (int i = 1; i < waves; ++i) t = MAX ? fmaxf(t, part[i]) : t + part[i];
    return t;
}

// y = x * (1 / sqrt(mean(x^2) + eps)) * w  (src/ops.cpp:19-41), one workgroup.
__global__ __launch_bounds__(kReduceThreads) void op_rmsnorm_kernel(const float* __restrict__ x,
                                                                   const float* __restrict__ w, int n, float eps,
                                                                   float* __restrict__ y) {
    float ss = 0.0f;
    for (int i = threadIdx.x; i < n; i += blockDim.x) ss += x[i] * x[i];
    ss = block_reduce<false>(ss);
    const float scale = 1.0f / sqrtf(ss / static_cast<float>(n) + eps);
    for (int i = threadIdx.x; i < n; i += blockDim.x) y[i] = x[i] * scale * w[i];
}

// Elementwise ops over n elements (grid-stride).
enum class Ew { Silu, Mul, Add };

template <Ew OP>
__global__ __launch_bounds__(kOpThreads) void op_elementwise_kernel(const float* __restrict__ a,
                                                                   const float* __restrict__ b, size_t n,
                                                                   float* __restrict__ y) {
    const size_t stride = static_cast<size_t>(gridDim.x) * blockDim.x;
    for (size_t i = static_cast<size_t>(blockIdx.x) * blockDim.x + threadIdx.x; i < n; i += stride) {
        const float v = a[i];
        if (OP == Ew::Silu) y[i] = v / (1.0f + expf(-v));  // src/ops.cpp:72-79
        if (OP == Ew::Mul) y[i] = v * b[i];
        if (OP == Ew::Add) y[i] = v + b[i];
    }
}

// Softmax of one vector (src/ops.cpp:43-70), one workgroup: maximum, then
// exp(x - max) and its sum, then the division.
__global__ __launch_bounds__(kReduceThreads) void op_softmax_kernel(const float* __restrict__ x, int n,
                                                                   float* __restrict__ y) {
    float m = -INFINITY;
    for (int i = threadIdx.x; i < n; i += blockDim.x) m = fmaxf(m, x[i]);
    m = block_reduce<true>(m);
    float s = 0.0f;
    for (int i = threadIdx.x; i < n; i += blockDim.x) {
        const float e = expf(x[i] - m);
        y[i] = e;
        s += e;
    }
    s = block_reduce<false>(s);
    for (int i = threadIdx.x; i < n; i += blockDim.x) y[i] = y[i] / s;
}

__global__ __launch_bounds__(kOpThreads) void op_embedding_kernel(const float* __restrict__ table, int dim,
                                                                 int token, float* __restrict__ y) {
    const float* row = table + static_cast<size_t>(token) * dim;
    for (int i = blockIdx.x * blockDim.x + threadIdx.x; i < dim; i += gridDim.x * blockDim.x) y[i] = row[i];
}

// RoPE of x [n_heads][head_dim] at position pos, one thread per rotated pair
// (src/ops.cpp:109-141): normal pairs (2i, 2i + 1), NeoX pairs (i, i + hd/2);
// the frequency of pair i is theta^(-2i / hd) in both.
__global__ __launch_bounds__(kOpThreads) void op_rope_kernel(float* __restrict__ x, int n_heads, int hd, int pos,
                                                            float theta, int neox) {
    const int half = hd / 2;
    const int idx = blockIdx.x * blockDim.x + threadIdx.x;
    if (idx >= n_heads * half) return;
    const int h = idx / half;
    const int i = idx % half;
    const float freq = 1.0f / powf(theta, static_cast<float>(2 * i) / static_cast<float>(hd));
    const float ang = static_cast<float>(pos) * freq;
    const float c = cosf(ang);
    const float s = sinf(ang);
    float* base = x + static_cast<size_t>(h) * hd;
    const int i0 = neox ? i : 2 * i;
    const int i1 = neox ? i + half : 2 * i + 1;
    const float x0 = base[i0];
    const float x1 = base[i1];
    base[i0] = x0 * c - x1 * s;
    base[i1] = x0 * s + x1 * c;
}

// Single-token attention of query head blockIdx.x over cache positions
// 0..pos of one layer (the math of src/forward.cpp:530-600: scores q.k *
// scale, softmax over the positions, probability-weighted sum of v).  The
// cache is [layer][max_seq][n_kv_heads][hd] f32, as CudaKVCache lays it out
// (src/cuda_kv_cache.cpp).  Four waves take every fourth position each and
// keep a running maximum, normaliser and weighted v sum (online softmax, so
// no score buffer is needed for any context length); the waves' states are
// merged through LDS.  Lane l holds elements l, l + 64, ... of the head.  Head
// sizes or pointers that 16-byte loads do not fit run this one.
template <int PER>
__global__ __launch_bounds__(64 * kAttnWaves) void op_attention_decode_kernel(
    const float* __restrict__ q, const float* __restrict__ keys, const float* __restrict__ values, int layer,
    int max_seq, int n_heads, int n_kv_heads, int hd, int pos, float scale, float* __restrict__ out) {
    __shared__ float st_m[kAttnWaves], st_l[kAttnWaves];
    __shared__ float st_acc[kAttnWaves][64 * PER];
    const int h = blockIdx.x;
    const int kvh = h / (n_heads / n_kv_heads);
    const int wave = threadIdx.x >> 6;
    const int lane = threadIdx.x & 63;
    const size_t row = static_cast<size_t>(n_kv_heads) * hd;
    const size_t base = static_cast<size_t>(layer) * max_seq * row + static_cast<size_t>(kvh) * hd;
    float qv[PER], acc[PER];
#pragma unroll
    for (int j = 0; j < PER; ++j) {
        const int e = lane + 64 * j;
        qv[j] = e < hd ? q[static_cast<size_t>(h) * hd + e] : 0.0f;
        acc[j] = 0.0f;
    }
    float m = -INFINITY, l = 0.0f;
    for (int t = wave; t <= pos; t += kAttnWaves) {
        const float* kt = keys + base + static_cast<size_t>(t) * row;
        const float* vt = values + base + static_cast<size_t>(t) * row;
        float d = 0.0f;
#pragma unroll
        for (int j = 0; j < PER; ++j) {
            const int e = lane + 64 * j;
            if (e < hd) d += qv[j] * kt[e];
        }
        const float s = wave_sum(d) * scale;
        const float mn = fmaxf(m, s);
        const float c = expf(m - mn);  // 0 on the wave's first position (m = -inf)
        const float p = expf(s - mn);
        l = l * c + p;
#pragma unroll
        for (int j = 0; j < PER; ++j) {
            const int e = lane + 64 * j;
            acc[j] = acc[j] * c + (e < hd ? p * vt[e] : 0.0f);
        }
        m = mn;
    }
    if (lane == 0) {
        st_m[wave] = m;
        st_l[wave] = l;
    }
#pragma unroll
    for (int j = 0; j < PER; ++j) st_acc[wave][lane + 64 * j] = acc[j];
    __syncthreads();
    // Merge: position 0 exists, so wave 0's maximum is finite and so is M.
    float M = st_m[0];
    for (int w = 1; w < kAttnWaves; ++w) M = fmaxf(M, st_m[w]);
    float L = 0.0f, f[kAttnWaves];
    for (int w = 0; w < kAttnWaves; ++w) {
        f[w] = st_l[w] > 0.0f ? expf(st_m[w] - M) : 0.0f;
        L += st_l[w] * f[w];
    }
    for (int e = threadIdx.x; e < hd; e += blockDim.x) {
        float v = 0.0f;
        for (int w = 0; w < kAttnWaves; ++w) v += st_acc[w][e] * f[w];
        out[static_cast<size_t>(h) * hd + e] = v / L;
    }
}

// Combines v with the lanes a DPP pattern names, or with the other 16 / 32 lanes.
template <int CTRL>
__device__ __forceinline__ float dpp(float v) {
    return __builtin_bit_cast(float, __builtin_amdgcn_mov_dpp(__builtin_bit_cast(int, v), CTRL, 0xF, 0xF, true));
}
struct OpSum {
    static __device__ __forceinline__ float of(float a, float b) { return a + b; }
};
struct OpMax {
    static __device__ __forceinline__ float of(float a, float b) { return fmaxf(a, b); }
};
template <class OP>
__device__ __forceinline__ float other16(float v) {
    const unsigned u = __builtin_bit_cast(unsigned, v);
    const auto r = __builtin_amdgcn_permlane16_swap(u, u, false, false);
    return OP::of(__builtin_bit_cast(float, static_cast<unsigned>(r[0])), __builtin_bit_cast(float, static_cast<unsigned>(r[1])));
}
template <class OP>
__device__ __forceinline__ float other32(float v) {
    const unsigned u = __builtin_bit_cast(unsigned, v);
    const auto r = __builtin_amdgcn_permlane32_swap(u, u, false, false);
    return OP::of(__builtin_bit_cast(float, static_cast<unsigned>(r[0])), __builtin_bit_cast(float, static_cast<unsigned>(r[1])));
}
// Over each run of LPR lanes; over the lanes of equal lane % LPR.  All VALU: the
// shuffles through LDS they replace cost 5 us of the launch at 4 heads a group.
template <int LPR>
__device__ __forceinline__ float run_sum(float v) {
    if (LPR >= 2) v += dpp<0xB1>(v);    // quad_perm [1, 0, 3, 2]
    if (LPR >= 4) v += dpp<0x4E>(v);    // quad_perm [2, 3, 0, 1]
    if (LPR >= 8) v += dpp<0x141>(v);   // row_half_mirror
    if (LPR >= 16) v += dpp<0x140>(v);  // row_mirror
    if (LPR >= 32) v = other16<OpSum>(v);
    if (LPR >= 64) v = other32<OpSum>(v);
    return v;
}
template <int LPR, class OP>
__device__ __forceinline__ float cross_runs(float v) {
    static_assert(LPR >= 4, "rotations of 8 and 4 lanes");
    if (LPR <= 8) v = OP::of(v, dpp<0x128>(v));  // row_ror:8
    if (LPR <= 4) v = OP::of(v, dpp<0x124>(v));  // row_ror:4
    if (LPR <= 16) v = other16<OP>(v);
    if (LPR <= 32) v = other32<OP>(v);
    return v;
}

// The softmax runs in base 2 (scores times log2(e) in the scale): one v_exp_f32 a
// weight, and the rounding of a score is what it was in base e.
__device__ __forceinline__ float exp2_of(float v) { return __builtin_amdgcn_exp2f(v); }
// A maximum to subtract: 0 while there are only -inf scores (their weights are 0).
__device__ __forceinline__ float finite_max(float m) { return m == -INFINITY ? 0.0f : m; }

// The same attention with the positions spread over the chip: workgroup
// (hg, split) takes up to G query heads of one KV head and the positions
// [split * per_split, ...) of it.  LPR lanes share a cache row (4 C floats of it
// each, C 16-byte loads LPR * 16 bytes apart), so a wave takes 64 / LPR rows at
// once; every row is used by all G heads from registers (q and the weighted v
// sums live there), and two rows per lane are in flight.  Each lane group keeps
// its own online softmax; the groups meet in the wave (DPP), the waves in
// LDS, the splits through `part`: each stores (max, sum, weighted v) per head and
// counts in, and the last of a head group merges them in a fixed order.
//
// Bound: HBM (the cache is read once) plus the split's tail (two dependent trips
// to memory).  The one-workgroup-per-head kernel above read 24.6 MB (32 heads, 8 KV
// heads of 128, 3000 positions) with 128 waves and one row in flight each: 1010 us;
// this one takes 15 us (launch and tail about 8, the read at 5 TB/s about 5).
template <int LPR, int C, int G>
__global__ __launch_bounds__(G == 1 ? 1024 : 256) void op_attention_split_kernel(const float* __restrict__ q, const float* __restrict__ keys,
                                          const float* __restrict__ values, int layer, int max_seq, int n_heads,
                                          int n_kv_heads, int hd, int pos, float scale2, float* __restrict__ out,
                                          int per_split, float* __restrict__ part, unsigned* __restrict__ count,
                                          uint32_t* done, uint32_t seq) {
    constexpr int R = 64 / LPR;    // rows of a wave
    constexpr int P = 2;           // rows of a lane in flight
    constexpr int E = 4 * C * LPR;  // head elements covered (>= hd)
    constexpr int ROW = E + 4;      // a state: the weighted v sum, maximum, sum, padding
    extern __shared__ __attribute__((aligned(16))) float sm[];  // [wave][G][ROW], weights; the merge's own
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6, waves = static_cast<int>(blockDim.x >> 6);
    const int li = lane % LPR, rg = lane / LPR;
    const int group = n_heads / n_kv_heads;
    const int chunks = (group + G - 1) / G;
    const int kvh = blockIdx.x / chunks;
    const int h0 = kvh * group + (blockIdx.x % chunks) * G;
    const int nh = min(G, (kvh + 1) * group - h0);
    const int split = blockIdx.y, splits = gridDim.y;
    const int t0 = split * per_split, t1 = min(pos + 1, t0 + per_split);
    const size_t row = static_cast<size_t>(n_kv_heads) * hd;
    const size_t base = static_cast<size_t>(layer) * max_seq * row + static_cast<size_t>(kvh) * hd;

    const float4 zero4{0.0f, 0.0f, 0.0f, 0.0f};
    // Loads are unconditional (lanes past the head re-read its last elements and
    // drop them): under a branch each would be waited for before the next.
    int eo[C];
    bool eok[C];
#pragma unroll
    for (int c = 0; c < C; ++c) {
        eo[c] = min((c * LPR + li) * 4, hd - 4);
        eok[c] = (c * LPR + li) * 4 < hd;
    }
    float4 qv[G][C], acc[G][C];
    float m[G], l[G];
#pragma unroll
    for (int g = 0; g < G; ++g) {
        m[g] = -INFINITY;
        l[g] = 0.0f;
#pragma unroll
        for (int c = 0; c < C; ++c) {
            qv[g][c] = *reinterpret_cast<const float4*>(q + static_cast<size_t>(h0 + min(g, nh - 1)) * hd + eo[c]);
            if (!eok[c]) qv[g][c] = zero4;
            acc[g][c] = zero4;
        }
    }
    const int stride = waves * R;
    for (int tb = t0; tb < t1; tb += P * stride) {
        float4 kr[P][C], vr[P][C];
#pragma unroll
        for (int p = 0; p < P; ++p) {
            const int t = min(tb + p * stride + wave * R + rg, t1 - 1);  // rows past the end: not used below
            const float* kt = keys + base + static_cast<size_t>(t) * row;
            const float* vt = values + base + static_cast<size_t>(t) * row;
#pragma unroll
            for (int c = 0; c < C; ++c) {
                kr[p][c] = *reinterpret_cast<const float4*>(kt + eo[c]);
                vr[p][c] = *reinterpret_cast<const float4*>(vt + eo[c]);
            }
        }
        float s[P][G];
#pragma unroll
        for (int p = 0; p < P; ++p) {
            const bool valid = tb + p * stride + wave * R + rg < t1;
#pragma unroll
            for (int c = 0; c < C; ++c) {
                if (!eok[c]) kr[p][c] = zero4;
                if (!valid || !eok[c]) vr[p][c] = zero4;  // weight 0 must meet no infinity
            }
#pragma unroll
            for (int g = 0; g < G; ++g) {
                float d = 0.0f;
#pragma unroll
                for (int c = 0; c < C; ++c) {
                    d = __builtin_fmaf(qv[g][c].x, kr[p][c].x, d);
                    d = __builtin_fmaf(qv[g][c].y, kr[p][c].y, d);
                    d = __builtin_fmaf(qv[g][c].z, kr[p][c].z, d);
                    d = __builtin_fmaf(qv[g][c].w, kr[p][c].w, d);
                }
                d = run_sum<LPR>(d) * scale2;
                s[p][g] = valid ? d : -INFINITY;
            }
        }
#pragma unroll
        for (int g = 0; g < G; ++g) {
            float mn = m[g];
#pragma unroll
            for (int p = 0; p < P; ++p) mn = fmaxf(mn, s[p][g]);
            const float ref = finite_max(mn);
            const float f = exp2_of(m[g] - ref);
            m[g] = mn;
            l[g] *= f;
            float w[P];
#pragma unroll
            for (int p = 0; p < P; ++p) {
                w[p] = exp2_of(s[p][g] - ref);
                l[g] += w[p];
            }
#pragma unroll
            for (int c = 0; c < C; ++c) {
                acc[g][c].x *= f, acc[g][c].y *= f, acc[g][c].z *= f, acc[g][c].w *= f;
#pragma unroll
                for (int p = 0; p < P; ++p) {
                    acc[g][c].x = __builtin_fmaf(w[p], vr[p][c].x, acc[g][c].x);
                    acc[g][c].y = __builtin_fmaf(w[p], vr[p][c].y, acc[g][c].y);
                    acc[g][c].z = __builtin_fmaf(w[p], vr[p][c].z, acc[g][c].z);
                    acc[g][c].w = __builtin_fmaf(w[p], vr[p][c].w, acc[g][c].w);
                }
            }
        }
    }
    // The wave's lane groups, then the waves through LDS.
#pragma unroll
    for (int g = 0; g < G; ++g) {
        const float mw = cross_runs<LPR, OpMax>(m[g]);
        const float f = exp2_of(m[g] - finite_max(mw));
        const float lw = cross_runs<LPR, OpSum>(l[g] * f);
#pragma unroll
        for (int c = 0; c < C; ++c) {
            acc[g][c].x = cross_runs<LPR, OpSum>(acc[g][c].x * f);
            acc[g][c].y = cross_runs<LPR, OpSum>(acc[g][c].y * f);
            acc[g][c].z = cross_runs<LPR, OpSum>(acc[g][c].z * f);
            acc[g][c].w = cross_runs<LPR, OpSum>(acc[g][c].w * f);
        }
        float* st = sm + (wave * G + g) * ROW;
        if (rg == 0) {
#pragma unroll
            for (int c = 0; c < C; ++c) *reinterpret_cast<float4*>(st + (c * LPR + li) * 4) = acc[g][c];
            if (li == 0) st[E] = mw, st[E + 1] = lw;
        }
    }
    __syncthreads();
    float* const wt = sm + waves * G * ROW;  // [G][waves] weights of the waves, then [G][2]: max, sum
    float* const ml = wt + G * waves;
    if (static_cast<int>(threadIdx.x) < nh) {
        const int g = threadIdx.x;
        float M = -INFINITY, L = 0.0f;
        for (int w = 0; w < waves; ++w) M = fmaxf(M, sm[(w * G + g) * ROW + E]);
        for (int w = 0; w < waves; ++w) {
            const float f = exp2_of(sm[(w * G + g) * ROW + E] - finite_max(M));
            wt[g * waves + w] = f;
            L += sm[(w * G + g) * ROW + E + 1] * f;
        }
        ml[2 * g] = M, ml[2 * g + 1] = L;
    }
    __syncthreads();
    const int n4 = hd / 4;
    const __amdgpu_buffer_rsrc_t prs = __builtin_amdgcn_make_buffer_rsrc(
        part, static_cast<short>(0), splits == 1 ? 0 : static_cast<int>(gridDim.x) * G * splits * ROW * 4, 0x00020000);
    const uint32_t mine = (blockIdx.x * G * splits) * ROW * 4;  // [g][split][ROW] of this head group
    for (int i = threadIdx.x; i < nh * n4; i += blockDim.x) {
        const int g = i / n4, e = i % n4 * 4;
        float4 v = zero4;
        for (int w = 0; w < waves; ++w) {
            const float4 x = *reinterpret_cast<const float4*>(sm + (w * G + g) * ROW + e);
            const float f = wt[g * waves + w];
            v.x = __builtin_fmaf(x.x, f, v.x), v.y = __builtin_fmaf(x.y, f, v.y);
            v.z = __builtin_fmaf(x.z, f, v.z), v.w = __builtin_fmaf(x.w, f, v.w);
        }
        if (splits == 1) {
            const float L = ml[2 * g + 1];
            float* o = out + static_cast<size_t>(h0 + g) * hd + e;
            o[0] = v.x / L, o[1] = v.y / L, o[2] = v.z / L, o[3] = v.w / L;
        } else {
            __builtin_amdgcn_raw_buffer_store_b128(__builtin_bit_cast(u32x4, v), prs, mine + ((g * splits + split) * ROW + e) * 4,
                                                   0, kCoherent);
        }
    }
    if (splits == 1) return;
    if (static_cast<int>(threadIdx.x) < nh) {
        const u32x4 v{__builtin_bit_cast(uint32_t, ml[2 * threadIdx.x]), __builtin_bit_cast(uint32_t, ml[2 * threadIdx.x + 1]),
                      0u, 0u};
        __builtin_amdgcn_raw_buffer_store_b128(v, prs, mine + ((threadIdx.x * splits + split) * ROW + E) * 4, 0, kCoherent);
    }
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");  // this wave's part of the state is in memory
    __shared__ unsigned last;
    __syncthreads();
    if (threadIdx.x == 0) {
        const unsigned before = __hip_atomic_fetch_add(count + blockIdx.x, 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        last = before == static_cast<unsigned>(splits) - 1 ? 1u : 0u;
    }
    __syncthreads();
    if (last == 0u) return;
    // Every thread sums one float4 of a head over its share of the splits, 16
    // loads in flight (each batch is one trip to memory).
    auto load4 = [&](int g, int s, int e) {
        return __builtin_bit_cast(
            float4, __builtin_amdgcn_raw_buffer_load_b128(prs, mine + ((g * splits + s) * ROW + e) * 4, 0, kCoherent));
    };
    constexpr int B = 16;
    const int items = nh * n4;
    const int ways = items >= static_cast<int>(blockDim.x) ? 1 : static_cast<int>(blockDim.x) / items;
    float4* const red = reinterpret_cast<float4*>(sm + G * 64);  // [way][items]
    float4 x[B];
    auto load_batch = [&](int i, int s0) {
        const int it = i % items;
#pragma unroll
        for (int u = 0; u < B; ++u) x[u] = load4(it / n4, min(s0 + u * ways, splits - 1), it % n4 * 4);
    };
    // The first batch flies with the (max, sum) words.
    if (static_cast<int>(threadIdx.x) < items * ways) load_batch(threadIdx.x, static_cast<int>(threadIdx.x) / items);
    for (int g = wave; g < nh; g += waves) {
        float ms = -INFINITY, ls = 0.0f;  // splits <= 64: one a lane
        if (lane < splits) {
            const float4 v = load4(g, lane, E);
            ms = v.x, ls = v.y;
        }
        const float M = wave_max(ms);
        const float f = exp2_of(ms - finite_max(M));
        const float L = wave_sum(lane < splits ? ls * f : 0.0f);
        if (lane < splits) sm[g * 64 + lane] = f / L;
    }
    __syncthreads();
    for (int i = threadIdx.x; i < items * ways; i += blockDim.x) {
        const int way = i / items, it = i % items;
        const int g = it / n4, e = it % n4 * 4;
        float4 v = zero4;
        for (int s0 = way; s0 < splits; s0 += B * ways) {
            if (i != static_cast<int>(threadIdx.x) || s0 != way) load_batch(i, s0);
#pragma unroll
            for (int u = 0; u < B; ++u) {
                if (s0 + u * ways >= splits) continue;
                const float f = sm[g * 64 + s0 + u * ways];
                v.x = __builtin_fmaf(x[u].x, f, v.x), v.y = __builtin_fmaf(x[u].y, f, v.y);
                v.z = __builtin_fmaf(x[u].z, f, v.z), v.w = __builtin_fmaf(x[u].w, f, v.w);
            }
        }
        if (ways == 1) {
            float* o = out + static_cast<size_t>(h0 + g) * hd + e;
            o[0] = v.x, o[1] = v.y, o[2] = v.z, o[3] = v.w;
        } else {
            red[i] = v;
        }
    }
    if (ways > 1) {
        __syncthreads();
        for (int i = threadIdx.x; i < items; i += blockDim.x) {
            float4 v = red[i];
            for (int w = 1; w < ways; ++w) {
                const float4 x = red[w * items + i];
                v.x += x.x, v.y += x.y, v.z += x.z, v.w += x.w;
            }
            float* o = out + static_cast<size_t>(h0 + i / n4) * hd + i % n4 * 4;
            o[0] = v.x, o[1] = v.y, o[2] = v.z, o[3] = v.w;
        }
    }
    if (threadIdx.x == 0) __hip_atomic_store(count + blockIdx.x, 0u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    if (done != nullptr) {
        __syncthreads();                                  // every wave has used its part of the states
        asm volatile("s_waitcnt vmcnt(0)" ::: "memory");  // the counter is back at zero
        if (threadIdx.x == 0) __hip_atomic_store(done + blockIdx.x, seq, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_SYSTEM);
    }
}

// C[M][N] = A[M][K] * op(B) in f32, op(B)[k][n] = B[k * N + n], or
// B[n * K + k] when B is stored transposed (a linear's W [N][K]).  16 x 16
// output tiles with the operands staged through LDS, K in steps of 16.
__global__ __launch_bounds__(kMatTile * kMatTile) void op_matmul_f32_kernel(const float* __restrict__ A,
                                                                           const float* __restrict__ B, int M,
                                                                           int K, int N, int bt,
                                                                           float* __restrict__ C) {
    __shared__ float ta[kMatTile][kMatTile + 1];
    __shared__ float tb[kMatTile][kMatTile + 1];
    const int tx = threadIdx.x % kMatTile;
    const int ty = threadIdx.x / kMatTile;
    const int m = blockIdx.y * kMatTile + ty;
    const int n = blockIdx.x * kMatTile + tx;
    float acc = 0.0f;
    for (int k0 = 0; k0 < K; k0 += kMatTile) {
        const int ka = k0 + tx;
        ta[ty][tx] = (m < M && ka < K) ? A[static_cast<size_t>(m) * K + ka] : 0.0f;
        const int kb = k0 + ty;
        const int nb = blockIdx.x * kMatTile + tx;
        float bv = 0.0f;
        if (kb < K && nb < N) bv = bt ? B[static_cast<size_t>(nb) * K + kb] : B[static_cast<size_t>(kb) * N + nb];
        tb[ty][tx] = bv;
        __syncthreads();
#pragma unroll
        for (int kk = 0; kk < kMatTile; ++kk) acc += ta[ty][kk] * tb[kk][tx];
        __syncthreads();
    }
    if (m < M && n < N) C[static_cast<size_t>(m) * N + n] = acc;
}

unsigned ew_grid(size_t n) {
    const size_t g = (n + kOpThreads - 1) / kOpThreads;
    return static_cast<unsigned>(g < 4096 ? (g > 0 ? g : 1) : 4096);
}

unsigned reduce_threads(int n) {
    // One wave for short vectors (the tiny model's 32 elements), up to 1024.
    unsigned t = 64;
    while (t < kReduceThreads && static_cast<int>(t) < n) t <<= 1;
    return t;
}

}  // namespace

hipError_t launch_op_rmsnorm(const float* x, const float* w, int n, float eps, float* y, hipStream_t s) {
    hipLaunchKernelGGL(op_rmsnorm_kernel, dim3(1), dim3(reduce_threads(n)), 0, s, x, w, n, eps, y);
    return hipGetLastError();
}

hipError_t launch_op_elementwise(int op, const float* a, const float* b, size_t n, float* y, hipStream_t s) {
    switch (op) {
        case kOpSilu:
            hipLaunchKernelGGL(op_elementwise_kernel<Ew::Silu>, dim3(ew_grid(n)), dim3(kOpThreads), 0, s, a, b, n, y);
            break;
        case kOpMul:
            hipLaunchKernelGGL(op_elementwise_kernel<Ew::Mul>, dim3(ew_grid(n)), dim3(kOpThreads), 0, s, a, b, n, y);
            break;
        case kOpAdd:
            hipLaunchKernelGGL(op_elementwise_kernel<Ew::Add>, dim3(ew_grid(n)), dim3(kOpThreads), 0, s, a, b, n, y);
            break;
        default:
            return hipErrorInvalidValue;
    }
    return hipGetLastError();
}

hipError_t launch_op_softmax(const float* x, int n, float* y, hipStream_t s) {
    hipLaunchKernelGGL(op_softmax_kernel, dim3(1), dim3(reduce_threads(n)), 0, s, x, n, y);
    return hipGetLastError();
}

hipError_t launch_op_embedding(const float* table, int dim, int token, float* y, hipStream_t s) {
    hipLaunchKernelGGL(op_embedding_kernel, dim3(ew_grid(static_cast<size_t>(dim))), dim3(kOpThreads), 0, s, table,
                       dim, token, y);
    return hipGetLastError();
}

hipError_t launch_op_rope(float* x, int n_heads, int head_dim, int pos, float theta, bool neox, hipStream_t s) {
    const int pairs = n_heads * (head_dim / 2);
    hipLaunchKernelGGL(op_rope_kernel, dim3((pairs + kOpThreads - 1) / kOpThreads), dim3(kOpThreads), 0, s, x,
                       n_heads, head_dim, pos, theta, neox ? 1 : 0);
    return hipGetLastError();
}

// The split kernel for G heads a workgroup: per head size, LPR lanes x C loads.
template <int G, int C>
static void launch_attention_split(dim3 grid, int waves, const float* q, const float* keys, const float* values,
                                   int layer, int max_seq, int n_heads, int n_kv_heads, int hd, int pos, float scale,
                                   float* out, int per_split, const OpAttnScratch& scratch, hipStream_t s) {
    unsigned* const count = static_cast<unsigned*>(scratch.mem);
    float* const part = scratch.mem != nullptr ? reinterpret_cast<float*>(count + kOpAttnScratchGroups) : nullptr;
    auto go = [&](auto kernel, int E) {
        const size_t lds = std::max(static_cast<size_t>(waves) * G * (E + 4) + G * (waves + 2),
                                    static_cast<size_t>(G) * 64 + 64 * waves * 4) * sizeof(float);
        hipLaunchKernelGGL(kernel, grid, dim3(64 * waves), lds, s, q, keys, values, layer, max_seq, n_heads, n_kv_heads,
                           hd, pos, scale * 1.44269504f, out, per_split, part, count, scratch.done, scratch.seq);
    };
    constexpr int F = 64 / (4 * C);  // lanes of a 64-element row
    if (hd <= 64) {
        go(op_attention_split_kernel<F, C, G>, 64);
    } else if (hd <= 128) {
        go(op_attention_split_kernel<2 * F, C, G>, 128);
    } else if (hd <= 256) {
        go(op_attention_split_kernel<4 * F, C, G>, 256);
    } else if constexpr (G < 8) {  // groups of 8 take heads of up to 256
        go(op_attention_split_kernel<8 * F, C, G>, 512);
    }
}

// 16-byte loads fit the head and the pointers.
static bool attention_vectors(const float* q, const float* keys, const float* values, int head_dim) {
    const uintptr_t p = reinterpret_cast<uintptr_t>(q) | reinterpret_cast<uintptr_t>(keys) | reinterpret_cast<uintptr_t>(values);
    return head_dim % 4 == 0 && (p & 15u) == 0;
}

// Head elements that the lane layout of a head size covers.
static int attention_elements(int head_dim) { return head_dim <= 64 ? 64 : head_dim <= 128 ? 128 : head_dim <= 256 ? 256 : 512; }

// Positions split over workgroups where they outweigh the split's tail (about 5 us):
// past 49 152 elements of a head (us, unsplit / split: 32 heads of 128 at 250 positions
// 7.5 / 9.7, at 500 14.1 / 12.0; 14 heads of 64 at 1000 9.2 / 12.2, at 3000 34 / 14.7).
// Workgroups of one head take 64 KB of cache, those of a group 128 KB, within 128 .. 768
// (32 / 32 heads of 128, 3000 positions: 43.5 / 28.5 / 24.4 / 26.3 us with 256 / 512 /
// 768 / 1024 workgroups; 32 / 8 heads: 14.9 / 15.8 / 18.4 with 128 / 256 / 512), and at
// least 32 positions.
OpAttnPlan op_attention_plan(const float* q, const float* keys, const float* values, int n_heads, int n_kv_heads,
                             int head_dim, int pos) {
    const int n = pos + 1;
    OpAttnPlan p{1, n_heads, 1, n};
    if (head_dim > kOpAttnMaxHeadDim || !attention_vectors(q, keys, values, head_dim)) return p;
    if (static_cast<long long>(n) * head_dim <= 49152) return p;
    const int group = n_heads / n_kv_heads;
    const int G = group > 4 && head_dim <= 256 ? 8 : group >= 3 ? 4 : group;
    const int groups = n_kv_heads * ((group + G - 1) / G);
    if (groups > kOpAttnScratchGroups) return p;
    const size_t bytes = static_cast<size_t>(n) * n_kv_heads * head_dim * 8;
    const int target = static_cast<int>(std::min<size_t>(768, std::max<size_t>(128, bytes >> (G == 1 ? 16 : 17))));
    const size_t room = kOpAttnScratchBytes - kOpAttnScratchGroups * sizeof(unsigned);
    const size_t state = static_cast<size_t>(groups) * G * (attention_elements(head_dim) + 4) * sizeof(float);
    const int splits = std::min({64, (target + groups - 1) / groups, n / 32, static_cast<int>(room / state)});
    if (splits <= 1) return p;
    const int per = (n + splits - 1) / splits;
    return OpAttnPlan{G, groups, (n + per - 1) / per, per};
}

hipError_t launch_op_attention_decode(const float* q, const float* keys, const float* values, int layer,
                                      int max_seq, int n_heads, int n_kv_heads, int head_dim, int pos,
                                      float* out, const OpAttnPlan& plan, const OpAttnScratch& scratch,
                                      hipStream_t s) {
    const float scale = 1.0f / std::sqrt(static_cast<float>(head_dim));
    if (head_dim > kOpAttnMaxHeadDim) return hipErrorInvalidValue;
    if (attention_vectors(q, keys, values, head_dim)) {
        auto go = [&](auto launch, dim3 grid, int waves, int per, const OpAttnScratch& mem) {
            launch(grid, waves, q, keys, values, layer, max_seq, n_heads, n_kv_heads, head_dim, pos, scale, out, per, mem, s);
        };
        const dim3 grid(plan.groups, plan.splits);
        if (plan.splits == 1 || scratch.mem == nullptr) {
            // One workgroup per head, as many waves as have rows.
            const int rows = std::max(1, 64 / (attention_elements(head_dim) / 16));
            const int waves = std::max(1, std::min(16, (pos + 2 * rows) / (2 * rows)));
            go(launch_attention_split<1, 4>, dim3(n_heads, 1), waves, pos + 1, OpAttnScratch{});
        } else if (plan.G == 1) {
            go(launch_attention_split<1, 4>, grid, 4, plan.per, scratch);
        } else if (plan.G == 2) {
            go(launch_attention_split<2, 4>, grid, 4, plan.per, scratch);
        } else if (plan.G == 4) {
            go(launch_attention_split<4, 4>, grid, 4, plan.per, scratch);
        } else {
            go(launch_attention_split<8, 2>, grid, 4, plan.per, scratch);
        }
        return hipGetLastError();
    }
    auto go = [&](auto kernel) {
        hipLaunchKernelGGL(kernel, dim3(n_heads), dim3(64 * kAttnWaves), 0, s, q, keys, values, layer, max_seq,
                           n_heads, n_kv_heads, head_dim, pos, scale, out);
    };
    if (head_dim <= 64) {
        go(op_attention_decode_kernel<1>);
    } else if (head_dim <= 128) {
        go(op_attention_decode_kernel<2>);
    } else if (head_dim <= 256) {
        go(op_attention_decode_kernel<4>);
    } else {
        go(op_attention_decode_kernel<kOpAttnMaxHeadDim / 64>);
    }
    return hipGetLastError();
}

hipError_t launch_op_matmul_f32(const float* a, const float* b, int m, int k, int n, bool b_transposed, float* c,
                                hipStream_t s) {
    const dim3 grid((n + kMatTile - 1) / kMatTile, (m + kMatTile - 1) / kMatTile);
    hipLaunchKernelGGL(op_matmul_f32_kernel, grid, dim3(kMatTile * kMatTile), 0, s, a, b, m, k, n,
                       b_transposed ? 1 : 0, c);
    return hipGetLastError();
}

}  // namespace mlq
