// Large-tile MFMA kernel of the batched GEMM (included by gemm.hip, whose
// choose_plan says which calls it takes and whose header gives the arithmetic: x split once into
// fp16 hi + lo per token, weights as exact fp16 integers, one block of 32 k folded
// into the f32 sums at a time with its scale).
//
// Bound: waits and issue order.  A block of a 32 x 32 tile costs 4
// v_mfma_f32_32x32x16_f16 (128 cycles of a SIMD's matrix core; the hi / lo split
// doubles the useful work) and 16 scale fmas, plus the decode of its weights (10 VALU
// per 8 codes), which only a wide tile spreads out.  Counters at 4096 x 4096 Q4_0, 512
// tokens: matrix cores 32 % busy, VALU 32 %, neither 50 %; LDS 26 %, 47 % of that in
// bank conflicts; waves wait 30 % of their cycles and 34 % for issue.  The same mix of
// MFMA, fma and decode instructions without any memory access takes 29 us.
//
// Split: a workgroup owns BM = 128 rows x BN = 64 tokens and eight waves (two per
// SIMD).  Wave (wm, ks) computes a 64 x 64 tile of block ks of every step of four
// blocks, so each decoded weight fragment meets two token tiles and each x fragment
// two row tiles, and nobody needs a K split across workgroups to fill a SIMD; the
// four partial tiles meet in LDS once at the end.  (32 x 64 or 64 x 32 per wave with
// 16 waves: 43-47 us against 41.5 at 4096 x 4096 Q4_0, 512 tokens; 64 x 128 or
// 128 x 64 with one wave per SIMD: 47-49; larger tiles spill.)
//
// Pipeline: x and weight bytes go straight to LDS (buffer_load ... lds, no
// registers), three stages deep, the copies spread over the step's tiles (issued
// together they held every wave at the start of the step: 47 -> 41.5 us).  The next
// block is read from LDS and decoded while the current one is on the matrix cores;
// a tile's scale fmas run under the next tile's MFMAs.  One barrier per step.
// Q4_1's offset term m * sum(x') is an f32 product on the matrix cores, one
// v_mfma_f32_32x32x1_2b_f32 (K = 1, both token tiles) per row tile and block: the
// sums stay f32 and an infinite m meets no padding.  64 cycles for two tiles, what
// two fp16 instructions on the sums' halves took (call, us, halves / f32: 4096 x 4096
// at 512 tokens 51.4 / 51.3, q/k/v at 2048 533 / 536, gate/up at 300 170.6 / 171.4;
// at the other places of a step up to 2.7 % slower).
// Measured (kernel alone, cold weights, us; the 128 x 32-token kernel it replaced in
// brackets): 4096 x 4096, 512 tokens Q4_0 43.0 (59.8), Q8_0 48.9 (68.6), Q4_1 51.0
// (69.7); 11008 x 4096 Q4_0 122.6 (163.0).
#pragma once

#include "mlq_kernels.h"

#include <hip/hip_runtime.h>

#include <cstdint>
#include <type_traits>

namespace mlq {
namespace {

typedef _Float16 f16x8 __attribute__((ext_vector_type(8)));
typedef _Float16 h2_t __attribute__((ext_vector_type(2)));
typedef float f32x4 __attribute__((ext_vector_type(4)));
typedef float f32x16 __attribute__((ext_vector_type(16)));
typedef float f32x32 __attribute__((ext_vector_type(32)));
typedef uint32_t u32x4 __attribute__((ext_vector_type(4)));

constexpr int kTileBlocks = 4;  // blocks of K per step

template <int QT> struct TileFmt;
template <> struct TileFmt<1> { static constexpr int BB = 34, ND = 5; };  // ND: code dwords a lane reads
template <> struct TileFmt<2> { static constexpr int BB = 18, ND = 3; };
template <> struct TileFmt<3> { static constexpr int BB = 20, ND = 2; };

template <int QT, int WM, int WN, int NWM, int NWN, int KS, int ST>
struct Tile {
    static constexpr int BM = 32 * WM * NWM;
    static constexpr int BN = 32 * WN * NWN;
    static constexpr int waves = NWM * NWN * KS;
    static constexpr int threads = 64 * waves;
    static constexpr int WBYTES = kTileBlocks * TileFmt<QT>::BB;  // bytes of one row's chunk
    static constexpr int WROW = (WBYTES + 15) / 16 * 16;          // its LDS row: whole 16-byte units
    static constexpr int x_bytes = kTileBlocks * BN * 128;
    static constexpr int s_bytes = QT == 3 ? (kTileBlocks * BN * 4 + 1023) / 1024 * 1024 : 0;
    static constexpr int w_bytes = BM * WROW;
    static constexpr int x_inst = x_bytes / 1024;   // 16 bytes per lane
    static constexpr int s_inst = s_bytes / 1024;
    static constexpr int w_inst = w_bytes / 1024;
    static constexpr int XI = (x_inst + waves - 1) / waves;
    static constexpr int SI = (s_inst + waves - 1) / waves;
    static constexpr int WI = (w_inst + waves - 1) / waves;
    static constexpr int stage = x_bytes + s_bytes + w_bytes;
    static constexpr int G = WM * WN * 4;  // f32x4 groups of a wave's tile
    static constexpr int GK = G / KS;      // groups a wave sums and stores
    static constexpr int loop_bytes = ST * stage + 16;  // + the dwords read past the last row's codes
    // Rounds of the K groups' reduction through LDS (at most 128 KB each).
    static constexpr int RR = KS == 1 ? 1 : (BM * BN * 4 * KS + 131071) / 131072;
    static constexpr int red_bytes = KS > 1 ? BM * BN * 4 * KS / RR : 0;
    static constexpr int lds = loop_bytes > red_bytes ? loop_bytes : red_bytes;
    static_assert(x_bytes % 1024 == 0 && s_bytes % 1024 == 0 && w_bytes % 1024 == 0, "whole copies");
    static_assert(G % (KS * RR) == 0 && kTileBlocks % KS == 0, "K split of a step");
};

struct TileArgs {
    const uint8_t* W[3];
    float* y[3];
    int M[3];
    int tile1, tile2;       // first row tile of weights 1 and 2 (row_tiles when absent)
    const _Float16* xs;     // split x [npad][nb][64]
    const float* bsum;      // Q4_1: block sums [npad][nb]
    const float* xscale;    // [npad]
    float* part;
    uint32_t part_bytes;
    unsigned* tile_count;
    int N, nb, row_tiles, tok_tiles, splits, chunks_per_split;
    int xcd_br, xcd_row_outer;
};

// 64 lanes copy 16 bytes each from buffer rs at voff + soff to LDS bytes
// lds + 16 * lane; asynchronous, counted by vmcnt.
__device__ __forceinline__ void lds_copy16(u32x4 rs, uint32_t voff, uint32_t soff, uint32_t lds) {
    asm volatile("s_mov_b32 m0, %0\n\ts_nop 0\n\tbuffer_load_dwordx4 %1, %2, %3 offen lds"
                 :
                 : "s"(lds), "v"(voff), "s"(rs), "s"(soff)
                 : "memory");
}
__device__ __forceinline__ u32x4 tile_rsrc(const void* base, uint32_t bytes) {
    const uint64_t p = reinterpret_cast<uint64_t>(base);
    u32x4 r{static_cast<uint32_t>(p), static_cast<uint32_t>(p >> 32) & 0xffffu, bytes, 0x00020000u};
#pragma unroll
    for (int i = 0; i < 4; ++i) r[i] = __builtin_amdgcn_readfirstlane(r[i]);
    return r;
}

// x of a step in LDS: [block][token][128 bytes], a block's hi then lo halves.
// Position of 16-byte unit u of token t's 128 bytes within them: spreads the
// same unit of 8 or 16 consecutive tokens over the LDS banks.
__device__ __forceinline__ int x_swizzle(int t) { return (t ^ (t >> 3)) & 7; }

__device__ __forceinline__ uint32_t bias_sub(uint32_t v, uint32_t neg_bias2) {
    const h2_t r = __builtin_bit_cast(h2_t, v) + __builtin_bit_cast(h2_t, neg_bias2);
    return __builtin_bit_cast(uint32_t, r);
}

// Q8_0 byte dwords (qs bytes 8g..8g+7) -> 8 fp16 codes.
__device__ __forceinline__ f16x8 bytes_to_f16(uint32_t a, uint32_t b, uint32_t neg_bias2) {
    const uint32_t ax = a ^ 0x80808080u;
    const uint32_t bx = b ^ 0x80808080u;
    const uint32_t mb = 0x64646464u;
    const u32x4 r{bias_sub(__builtin_amdgcn_perm(mb, ax, 0x04010400u), neg_bias2),
                  bias_sub(__builtin_amdgcn_perm(mb, ax, 0x04030402u), neg_bias2),
                  bias_sub(__builtin_amdgcn_perm(mb, bx, 0x04010400u), neg_bias2),
                  bias_sub(__builtin_amdgcn_perm(mb, bx, 0x04030402u), neg_bias2)};
    return __builtin_bit_cast(f16x8, r);
}

// Q4 code dword (bytes 4g .. 4g + 3 of qs) -> q - OFF as fp16, the low nibbles of
// bytes 0, 2, 1, 3, then the high ones.  0x6400 | n is 1024 + n; the high nibbles
// stay in place (1024 + 16 n) and one fma scales them.
template <int OFF>
__device__ __forceinline__ f16x8 nibbles_f16(uint32_t q, uint32_t mask, uint32_t mask4, uint32_t magic) {
    const uint32_t p = q >> 8;
    const h2_t off{static_cast<_Float16>(-1024.0f - OFF), static_cast<_Float16>(-1024.0f - OFF)};
    const h2_t s16{static_cast<_Float16>(0.0625f), static_cast<_Float16>(0.0625f)};
    const h2_t off16{static_cast<_Float16>(-64.0f - OFF), static_cast<_Float16>(-64.0f - OFF)};
    const h2_t a = __builtin_bit_cast(h2_t, (q & mask) | magic) + off;
    const h2_t b = __builtin_bit_cast(h2_t, (p & mask) | magic) + off;
    const h2_t c = __builtin_elementwise_fma(__builtin_bit_cast(h2_t, (q & mask4) | magic), s16, off16);
    const h2_t d = __builtin_elementwise_fma(__builtin_bit_cast(h2_t, (p & mask4) | magic), s16, off16);
    return f16x8{a.x, a.y, b.x, b.y, c.x, c.y, d.x, d.y};
}

template <int QT, int WM, int WN, int NWM, int NWN, int KS, int ST>
__global__ __launch_bounds__(64 * NWM * NWN * KS, (NWM * NWN * KS + 3) / 4) void gemm_tile_kernel(const TileArgs a) {
    using T = Tile<QT, WM, WN, NWM, NWN, KS, ST>;
    constexpr int BB = TileFmt<QT>::BB, ND = TileFmt<QT>::ND, BN = T::BN;
    constexpr int JB = kTileBlocks / KS;  // blocks of a step that one wave computes
    extern __shared__ __attribute__((aligned(16))) char smem[];
    const uint32_t lds0 = static_cast<uint32_t>(
        reinterpret_cast<uintptr_t>((__attribute__((address_space(3))) char*)smem));

    const int lane = threadIdx.x & 63;
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int wm = wave % NWM, wn = (wave / NWM) % NWN, ks = wave / (NWM * NWN);
    const int l32 = lane & 31, h = lane >> 5;

    const int wg = blockIdx.x;
    const int split = wg % a.splits;
    int tile = wg / a.splits;
    if (a.xcd_br > 0) {
        const int bt_n = 8 / a.xcd_br;
        const int rows_b = a.row_tiles / a.xcd_br, toks_b = a.tok_tiles / bt_n;
        const int xcd = wg % 8, j = wg / 8;
        const int rl = a.xcd_row_outer ? j / toks_b : j % rows_b;
        const int tl = a.xcd_row_outer ? j % toks_b : j / rows_b;
        tile = ((xcd % bt_n) * toks_b + tl) * a.row_tiles + (xcd / bt_n) * rows_b + rl;
    }
    const int rt = tile % a.row_tiles;
    const int gi = (rt >= a.tile1 ? 1 : 0) + (rt >= a.tile2 ? 1 : 0);
    const uint8_t* const Wg = gi == 0 ? a.W[0] : gi == 1 ? a.W[1] : a.W[2];
    float* const yg = gi == 0 ? a.y[0] : gi == 1 ? a.y[1] : a.y[2];
    const int M = gi == 0 ? a.M[0] : gi == 1 ? a.M[1] : a.M[2];
    const int m_base = (rt - (gi == 0 ? 0 : gi == 1 ? a.tile1 : a.tile2)) * T::BM;
    const int n_base = (tile / a.row_tiles) * BN;
    const int nb = a.nb;
    const int c0 = split * a.chunks_per_split;
    const int nchunk = min(nb / kTileBlocks, c0 + a.chunks_per_split) - c0;

    const uint32_t row_bytes = static_cast<uint32_t>(nb) * BB;
    const u32x4 wrs0 = tile_rsrc(Wg + static_cast<size_t>(m_base) * row_bytes,
                                static_cast<uint32_t>(min(T::BM, M - m_base)) * row_bytes);
    const u32x4 xrs0 = tile_rsrc(a.xs + static_cast<size_t>(n_base) * nb * 64, static_cast<uint32_t>(BN) * nb * 128);
    const u32x4 srs0 = tile_rsrc(QT == 3 ? a.bsum + static_cast<size_t>(n_base) * nb : nullptr,
                                QT == 3 ? static_cast<uint32_t>(BN) * nb * 4 : 0);

    uint32_t xoff[T::XI], woff[T::WI], soff[T::SI > 0 ? T::SI : 1];
    uint32_t xlds[T::XI], wlds[T::WI], slds[T::SI > 0 ? T::SI : 1];
#pragma unroll
    for (int i = 0; i < T::XI; ++i) {
        const int q = min(wave + i * T::waves, T::x_inst - 1);
        const int j = q / (BN / 8);
        const int t = (q % (BN / 8)) * 8 + (lane >> 3);
        xoff[i] = (static_cast<uint32_t>(t) * nb + j) * 128 + ((lane & 7) ^ x_swizzle(t)) * 16;
        xlds[i] = lds0 + q * 1024;
    }
#pragma unroll
    for (int i = 0; i < T::SI; ++i) {
        const int q = min(wave + i * T::waves, T::s_inst - 1);
        soff[i] = static_cast<uint32_t>(q * 64 + lane) * nb * 4;  // tokens past BN: past the range
        slds[i] = lds0 + T::x_bytes + q * 1024;
    }
#pragma unroll
    for (int i = 0; i < T::WI; ++i) {
        const int q = min(wave + i * T::waves, T::w_inst - 1);
        const int u = q * 64 + lane;
        woff[i] = static_cast<uint32_t>(u / (T::WROW / 16)) * row_bytes + (u % (T::WROW / 16)) * 16;
        wlds[i] = lds0 + T::x_bytes + T::s_bytes + q * 1024;
    }
    // Requests part `part` of `parts` of chunk c into the stage at st.
    auto issue = [&](int c, uint32_t st, int part, int parts) {
        const uint32_t cc = static_cast<uint32_t>(c0 + c);
        u32x4 wrs = wrs0, xrs = xrs0, srs = srs0;
        if (c >= nchunk) wrs[2] = xrs[2] = srs[2] = 0;
        constexpr int CNT = T::XI + T::WI + T::SI;
#pragma unroll
        for (int q = 0; q < CNT; ++q) {
            if (q * parts / CNT != part) continue;
            const int x = q - T::WI, u = x - T::XI;
            if (q < T::WI) lds_copy16(wrs, woff[q], cc * T::WBYTES, wlds[q] + st);
            if (x >= 0 && x < T::XI) lds_copy16(xrs, xoff[x < 0 ? 0 : x], cc * (kTileBlocks * 128), xlds[x < 0 ? 0 : x] + st);
            if (u >= 0) lds_copy16(srs, soff[u < 0 ? 0 : u], cc * (kTileBlocks * 4), slds[u < 0 ? 0 : u] + st);
        }
    };

    uint32_t mask = 0x000F000Fu, mask4 = 0x00F000F0u, magic = 0x64006400u;
    asm volatile("" : "+v"(mask), "+v"(mask4), "+v"(magic));

    // The sums of (row tile, token tile); Q4_1 keeps a row tile's two token tiles in one
    // vector, as the block sums' product writes them.
    static_assert(QT != 3 || WN == 2, "the block sums' product takes both token tiles");
    using Acc = std::conditional_t<QT == 3, f32x32, f32x16>;
    constexpr int AT = QT == 3 ? WN : 1;  // token tiles of one vector, 16 elements each
    Acc acc[WM][WN / AT];
#pragma unroll
    for (int r = 0; r < WM; ++r)
#pragma unroll
        for (int t = 0; t < WN / AT; ++t) acc[r][t] = Acc{};
    const f32x16 zero{};

    // A step's operands of this wave: its blocks' decoded weights, scales and x.
    struct Frag {
        f16x8 w[WM][2];
        _Float16 d[WM];
        f16x8 hi[WN][2], lo[WN][2];
        uint32_t dm[QT == 3 ? WM : 1];  // Q4_1: d and m as stored
        float s;                        // Q4_1: block sum of token l32 of token tile h
    };
    const int sw = x_swizzle(l32);
    uint32_t xu[2][2];
#pragma unroll
    for (int s = 0; s < 2; ++s) {
        xu[s][0] = (wn * WN * 32 + l32) * 128 + (((2 * h + s) ^ sw) * 16);
        xu[s][1] = (wn * WN * 32 + l32) * 128 + (((4 + 2 * h + s) ^ sw) * 16);
    }
    const uint32_t wrow0 = T::x_bytes + T::s_bytes + (wm * WM * 32 + l32) * T::WROW;
    auto read_x = [&](uint32_t st, int j, int t, Frag& f) {
        const char* xt = smem + st + j * (BN * 128) + t * 4096;
#pragma unroll
        for (int s = 0; s < 2; ++s) {
            f.hi[t][s] = *reinterpret_cast<const f16x8*>(xt + xu[s][0]);
            f.lo[t][s] = *reinterpret_cast<const f16x8*>(xt + xu[s][1]);
        }
        if (QT == 3 && t == 0)
            f.s = *reinterpret_cast<const float*>(smem + st + T::x_bytes + (wn * WN * 32 + lane) * 16 + j * 4);
    };
    auto read_w = [&](uint32_t st, int j, int r, uint32_t (&raw)[ND], Frag& f) {
        const char* row = smem + st + wrow0 + r * (32 * T::WROW);
        const uint32_t* pw = reinterpret_cast<const uint32_t*>(row);
        if (QT == 3) {
            f.dm[r] = pw[5 * j];
#pragma unroll
            for (int i = 0; i < ND; ++i) raw[i] = pw[5 * j + 1 + 2 * h + i];
            return;
        }
        f.d[r] = *reinterpret_cast<const _Float16*>(row + j * BB);
        // Even blocks' codes start two bytes into a dword, odd blocks' on one.
        const int first = QT == 2 ? 9 * (j >> 1) + 5 * (j & 1) + 2 * h : 17 * (j >> 1) + 9 * (j & 1) + 4 * h;
#pragma unroll
        for (int i = 0; i < ND; ++i) raw[i] = pw[first + i];
    };
    auto decode_w = [&](int j, int r, const uint32_t (&raw)[ND], Frag& f) {
        const uint32_t sh = (j & 1) ? 0 : 16;
        uint32_t q[ND];
#pragma unroll
        for (int i = 0; i + 1 < ND; ++i) q[i] = __builtin_amdgcn_alignbit(raw[i + 1], raw[i], sh);
        if (QT == 3) {
            f.d[r] = __builtin_bit_cast(h2_t, f.dm[r]).x;
            f.w[r][0] = nibbles_f16<0>(raw[0], mask, mask4, magic);
            f.w[r][1] = nibbles_f16<0>(raw[1], mask, mask4, magic);
        } else if (QT == 1) {
            f.w[r][0] = bytes_to_f16(q[0], q[1], 0xE480E480u);
            f.w[r][1] = bytes_to_f16(q[2], q[3], 0xE480E480u);
        } else {
            f.w[r][0] = nibbles_f16<8>(q[0], mask, mask4, magic);
            f.w[r][1] = nibbles_f16<8>(q[1], mask, mask4, magic);
        }
    };

    constexpr int CNT = T::XI + T::WI + T::SI;
    static_assert(ST * CNT < 64, "vmcnt range");
    static_assert(JB == 1, "one block per wave and step");
    uint32_t st_c = 0;  // stage of the current chunk
    auto next_stage = [&](uint32_t st) { return st + T::stage == ST * T::stage ? 0 : st + T::stage; };
    f32x16 C[2];
    float dprev;
    const int j = ks;
    // One step: chunk c is in `cur`, chunk c + 1 in LDS.
    auto step = [&](int c, Frag& cur, Frag& nxt) {
        asm volatile("s_waitcnt vmcnt(%0) lgkmcnt(0)\n\ts_barrier" ::"n"((ST - 2) * CNT) : "memory");
        const uint32_t st_n = next_stage(st_c);
        uint32_t raw[WM][ND];
        constexpr int NT = WM * WN;
#pragma unroll
        for (int k = 0; k < NT; ++k) {
            const int t = k / WM, r = k % WM;
            f32x16 v = __builtin_amdgcn_mfma_f32_32x32x16_f16(cur.hi[t][0], cur.w[r][0], zero, 0, 0, 0);
            v = __builtin_amdgcn_mfma_f32_32x32x16_f16(cur.hi[t][1], cur.w[r][1], v, 0, 0, 0);
            v = __builtin_amdgcn_mfma_f32_32x32x16_f16(cur.lo[t][0], cur.w[r][0], v, 0, 0, 0);
            v = __builtin_amdgcn_mfma_f32_32x32x16_f16(cur.lo[t][1], cur.w[r][1], v, 0, 0, 0);
            if (k == 0) {
#pragma unroll
                for (int q = 0; q < WM; ++q) read_w(st_n, j, q, raw[q], nxt);
            }
            issue(c + ST, st_c, k, NT);
            if (r == WM - 1) read_x(st_n, j, t, nxt);
            const int kp = (k + NT - 1) % NT;  // the tile before
            Acc& ap = acc[kp % WM][kp / WM / AT];
            const int p0 = 16 * (kp / WM % AT);
#pragma unroll
            for (int i = 0; i < 16; ++i) ap[p0 + i] = __builtin_fmaf(dprev, C[(k + 1) & 1][i], ap[p0 + i]);
            if constexpr (QT == 3) {
                // + m * sum(x'), one k: both token tiles of a row tile (lanes 0-31 and
                // 32-63 of the sums), between that row tile's two rounds of scale fmas.
                if (k >= 1 && k <= WM) {
                    const float m = static_cast<float>(__builtin_bit_cast(h2_t, cur.dm[kp % WM]).y);
                    ap = __builtin_amdgcn_mfma_f32_32x32x1f32(cur.s, m, ap, 0, 0, 0);
                }
            }
            C[k & 1] = v;
            dprev = static_cast<float>(cur.d[r]);
            if (NT - k <= WM) decode_w(j, k + WM - NT, raw[k + WM - NT], nxt);
            __builtin_amdgcn_sched_barrier(0);
        }
        st_c = st_n;
    };

    // Stage s holds chunk c with c % ST == s.  A step computes chunk c from
    // registers; chunk c + 1 is read from LDS into the other set of registers and
    // decoded meanwhile, and chunk c + ST is requested into the stage of chunk c,
    // which every wave has read by the step's barrier.  Chunks past the last are
    // copied from an empty range: zeros.
    {
        Frag A, B;
        C[0] = C[1] = f32x16{};
        dprev = 0.0f;
#pragma unroll
        for (int k = 0; k < ST; ++k) issue(k, k * T::stage, 0, 1);
        asm volatile("s_waitcnt vmcnt(%0)\n\ts_barrier" ::"n"((ST - 1) * CNT) : "memory");
        uint32_t raw[WM][ND];
#pragma unroll
        for (int r = 0; r < WM; ++r) read_w(0, j, r, raw[r], A);
#pragma unroll
        for (int t = 0; t < WN; ++t) read_x(0, j, t, A);
#pragma unroll
        for (int r = 0; r < WM; ++r) decode_w(j, r, raw[r], A);
        for (int c = 0; c < nchunk; c += 2) {
            step(c, A, B);
            step(c + 1, B, A);
        }
        Acc& ap = acc[WM - 1][(WN - 1) / AT];
        constexpr int p0 = 16 * ((WN - 1) % AT);
#pragma unroll
        for (int i = 0; i < 16; ++i) ap[p0 + i] = __builtin_fmaf(dprev, C[(WM * WN - 1) & 1][i], ap[p0 + i]);
        asm volatile("s_waitcnt vmcnt(0) lgkmcnt(0)" ::: "memory");  // no copy may land in the reduction below
    }

    // Add the K groups' tiles in group order: group k of the waves of one tile
    // sums and stores its share of the f32x4 groups.
    constexpr int GR = T::G / T::RR, GKR = T::GK / T::RR;
    auto group_of = [&](int q) { return (q / GKR) * GR + ks * GKR + q % GKR; };
    auto acc4 = [&](int g) {
        const int t = g / 4 % WN;
        const Acc& v = acc[g / 4 / WN][t / AT];
        const int i = 16 * (t % AT) + 4 * (g % 4);
        return f32x4{v[i], v[i + 1], v[i + 2], v[i + 3]};
    };
    f32x4 own[T::GK];
    if (KS > 1) {
        f32x4* red = reinterpret_cast<f32x4*>(smem) + (wn * NWM + wm) * GR * 64 + lane;
        constexpr int kstride = NWM * NWN * GR * 64;
#pragma unroll
        for (int u = 0; u < T::RR; ++u) {
            __syncthreads();
#pragma unroll
            for (int g = 0; g < GR; ++g) red[ks * kstride + g * 64] = acc4(u * GR + g);
            __syncthreads();
#pragma unroll
            for (int q = 0; q < GKR; ++q) {
                f32x4 s = red[(ks * GKR + q) * 64];
#pragma unroll
                for (int k = 1; k < KS; ++k) s += red[k * kstride + (ks * GKR + q) * 64];
                own[u * GKR + q] = s;
            }
        }
    } else {
#pragma unroll
        for (int g = 0; g < T::G; ++g) own[g] = acc4(g);
    }

    if (a.splits > 1) {
        // Partial tile [tile][split][group][thread], written through; the workgroup
        // that completes the tile's count adds the splits in order.
        const uint32_t tile_base = static_cast<uint32_t>(tile) * a.splits * (T::GK * T::threads * 16);
        const __amdgpu_buffer_rsrc_t prs = __builtin_amdgcn_make_buffer_rsrc(a.part, static_cast<short>(0),
                                                                             static_cast<int>(a.part_bytes), 0x00020000);
#pragma unroll
        for (int q = 0; q < T::GK; ++q)
            __builtin_amdgcn_raw_buffer_store_b128(__builtin_bit_cast(u32x4, own[q]), prs,
                                                   tile_base + ((split * T::GK + q) * T::threads + threadIdx.x) * 16, 0,
                                                   16);
        asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
        __shared__ unsigned last;
        __syncthreads();
        if (threadIdx.x == 0) {
            const unsigned done =
                __hip_atomic_fetch_add(a.tile_count + tile, 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
            last = done == static_cast<unsigned>(a.splits) - 1 ? 1u : 0u;
        }
        __syncthreads();
        if (last == 0u) return;
#pragma unroll
        for (int q = 0; q < T::GK; ++q) own[q] = f32x4{};
        constexpr int kBatch = T::GK <= 2 ? 8 : 4;
        for (int s0 = 0; s0 < a.splits; s0 += kBatch) {
            f32x4 v[kBatch][T::GK];
#pragma unroll
            for (int b = 0; b < kBatch; ++b) {
                const int s = min(s0 + b, a.splits - 1);
#pragma unroll
                for (int q = 0; q < T::GK; ++q)
                    v[b][q] = __builtin_bit_cast(
                        f32x4, __builtin_amdgcn_raw_buffer_load_b128(
                                   prs, tile_base + ((s * T::GK + q) * T::threads + threadIdx.x) * 16, 0, 16));
            }
#pragma unroll
            for (int b = 0; b < kBatch; ++b)
                if (s0 + b < a.splits) {
#pragma unroll
                    for (int q = 0; q < T::GK; ++q) own[q] += v[b][q];
                }
        }
        if (threadIdx.x == 0) __hip_atomic_store(a.tile_count + tile, 0u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    }
#pragma unroll
    for (int q = 0; q < T::GK; ++q) {
        const int g = group_of(q);
        const int rtile = g / 4 / WN, ttile = g / 4 % WN;
        const int row = m_base + (wm * WM + rtile) * 32 + l32;
        const int n0 = n_base + (wn * WN + ttile) * 32 + 8 * (g % 4) + 4 * h;
#pragma unroll
        for (int i = 0; i < 4; ++i)
            if (n0 + i < a.N && row < M) yg[static_cast<size_t>(n0 + i) * M + row] = own[q][i] * a.xscale[n0 + i];
    }
}

}  // namespace
}  // namespace mlq
