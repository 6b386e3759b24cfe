// Dequant-GEMM for prompt chunks and pieces of 33 tokens and more on the matrix cores
// (gfx950): the products of gemm.hip (y[t][r] = sum_k deq(W_r)[k] x[t][k],
// src/xiaoju-pipe/core/xj_cpu.c:36-54) for hundreds of tokens per launch, so
// that a weight is read once per 128 tokens and decoded once per 64 (by each of
// the two wavefronts that share its rows).
//
// What bounds it: two f16 MFMAs per product (Q6_K: three), i.e. the matrix
// cores; the weights' bytes are read once per token group through the caches.
// The arithmetic is gemm.hip's: the activations of a token's 256-element block
// as v * 2^-e = hi + lo (two f16 planes), the weights as small integers exact
// in f16, every product exact, a block accumulated in fp32, then added as
//   Q4_K: 2^e (d S - dmin M), S = sum sc_j q (hi + lo), M = sum m_j sx_j with
//         the group sums sx_j of hi + lo as two f16 planes of their own (one
//         MFMA per tile and block)
//   Q6_K: 2^e d S, sc (q - 32) = F + R with F rounded to f16 and R exact:
//         S = F hi + R hi + F lo
//
// Work split. A 512-thread work-group computes 256 rows x 128 tokens at a
// time, a wavefront 64 x 64 of it as 2 x 2 tiles of v_mfma_f32_32x32x16_f16
// (tokens as rows of the tile, weight rows as its columns: a lane's outputs
// share one weight row, so d and dmin are per-lane scalars and the stores are
// consecutive rows). Rows come in 32-row tiles numbered over all segments of
// the launch, so short segments (beta, alpha) share a row group. The units, a
// (token group, row group, 256-element block) triple each, are dealt out in
// equal contiguous ranges, one persistent work-group per CU; consecutive
// ranges go to one XCD, whose work-groups then read the same token group's
// activations from its L2. A tile covered by one work-group is stored
// directly, one shared by several is added by the last to arrive, in
// work-group order.
//
// Memory. The prep launch writes the activations in the order the lanes read
// them (kWideRec bytes per 32 tokens and block), so a stage of 64 inner
// elements is copied to LDS in whole KB by global_load_lds and read without
// bank conflicts; the weights' quants pass through LDS too (rows are 144 bytes
// apart in 16-byte pieces, permuted so that 16 lanes fall on distinct banks).
// Activations are requested one stage ahead, weights two. The copies are
// inline asm because the compiler would otherwise wait for all of them before
// every LDS read; they write no registers.
#include "common.h"
#include "kernels.h"
#include "xj_hip.h"

#include <algorithm>
#include <cstdint>

namespace xjk {
namespace {

typedef _Float16 h2 __attribute__((ext_vector_type(2)));
typedef _Float16 h4 __attribute__((ext_vector_type(4)));
typedef _Float16 h8 __attribute__((ext_vector_type(8)));
typedef float f4 __attribute__((ext_vector_type(4)));
typedef float f16v __attribute__((ext_vector_type(16)));
typedef unsigned int u4 __attribute__((ext_vector_type(4)));
typedef unsigned int u2 __attribute__((ext_vector_type(2)));

constexpr int kThreads = 512;
constexpr int kSkinnyT = 64;                      // tokens of the narrow kernel
constexpr int kRows = 256, kToks = 128;          // a work-group's tile
constexpr int kTokTiles = kToks / 32;
constexpr int kStageB = 8192;                     // a 32-token tile's activations of 64 inner elements
constexpr int kAux = 2048;                        // ... and of a block: group sums (1 KB), 2^e (128 B), padding

template <bool Q6>
struct Lds {
    static constexpr int WB = Q6 ? 96 : 64;       // quant bytes of a row's half block
    static constexpr int ACT = 0, ACT_N = kTokTiles * kStageB;
    static constexpr int W = ACT + 2 * ACT_N, W_N = kRows * WB;
    static constexpr int HD = W + 2 * W_N, HD_N = kRows * 16;      // Q4_K header, Q6_K scales
    static constexpr int D = HD + 2 * HD_N, D_N = Q6 ? kRows * 4 : 0;   // Q6_K: the word holding d
    static constexpr int AUX = D + 2 * D_N, AUX_N = kTokTiles * kAux;
    static constexpr int TSC = AUX + 2 * AUX_N;   // per-token RMSNorm scales of a stored tile
    static constexpr int SIZE = TSC + kToks * 4;
};

__device__ __forceinline__ f16v mfma(h8 a, h8 b, f16v c) { return __builtin_amdgcn_mfma_f32_32x32x16_f16(a, b, c, 0, 0, 0); }

__device__ __forceinline__ f4 mfma16(h8 a, h8 b, f4 c) { return __builtin_amdgcn_mfma_f32_16x16x32_f16(a, b, c, 0, 0, 0); }

// Lane l: 16 (4) bytes at p to LDS offset off + 16 l (4 l); off is uniform over the wavefront.
__device__ __forceinline__ void dma16(const uint8_t *p, uint32_t off) {
    asm volatile("s_mov_b32 m0, %1\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %0, off" ::"v"(p), "s"(off) : "memory", "m0");
}
__device__ __forceinline__ void dma4(const uint8_t *p, uint32_t off) {
    asm volatile("s_mov_b32 m0, %1\n\ts_nop 0\n\tglobal_load_lds_dword %0, off" ::"v"(p), "s"(off) : "memory", "m0");
}
template <int N>
__device__ __forceinline__ void wait_vm() {
    static_assert(N >= 0 && N < 16, "vmcnt range");
    asm volatile("s_waitcnt vmcnt(%0)" ::"n"(N) : "memory");
}
// Every wavefront's LDS reads are done (their values waited for) and its own
// copies awaited before; global loads in flight stay in flight.
__device__ __forceinline__ void stage_barrier() {
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "workgroup", "local");
    __builtin_amdgcn_s_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "workgroup", "local");
}

__device__ __forceinline__ h2 as_h2(uint32_t u) { return __builtin_bit_cast(h2, u); }
// f16 pairs 1024 + byte: an f16 whose high byte is 0x64 has the value 1024 + its low byte
__device__ __forceinline__ h2 biased01(uint32_t w) { return as_h2(__builtin_amdgcn_perm(0x64646464u, w, 0x04010400u)); }
__device__ __forceinline__ h2 biased23(uint32_t w) { return as_h2(__builtin_amdgcn_perm(0x64646464u, w, 0x04030402u)); }
__device__ __forceinline__ h8 cat8(h2 a, h2 b, h2 c, h2 d) {
    return __builtin_shufflevector(__builtin_shufflevector(a, b, 0, 1, 2, 3), __builtin_shufflevector(c, d, 0, 1, 2, 3), 0,
                                   1, 2, 3, 4, 5, 6, 7);
}
__device__ __forceinline__ h2 fma2(h2 a, h2 b, h2 c) { return __builtin_elementwise_fma(a, b, c); }

// 32-row tile index -> segment; row of the tile's line i, clamped into the segment
struct RowRef {
    int seg, row;
};
__device__ __forceinline__ RowRef row_ref(const WideArgs &a, int tile, int i) {
    tile = min(tile, a.rt0[a.nseg] - 1);
    int s = 0;
#pragma unroll
    for (int k = 1; k < kGemmMaxSeg; k++) s += k < a.nseg && tile >= a.rt0[k];
    return RowRef{s, min((tile - a.rt0[s]) * 32 + i, a.seg[s].N - 1)};
}

// This thread's weight copies of one row group (addresses of block 0).
template <bool Q6>
struct WSrc {
    const uint8_t *q[2];    // Q4_K quants / Q6_K low nibbles: two 16-byte slots
    const uint8_t *qh;      // Q6_K high bits: one slot
    const uint8_t *hd;      // header / scales (lanes 0..31)
    const uint8_t *d;       // Q6_K: d's address, block 0
};
template <bool Q6>
__device__ __forceinline__ void wsrc(const WideArgs &a, int rg, int wv, int lane, WSrc<Q6> &s) {
    const int nb = a.nb;
#pragma unroll
    for (int i = 0; i < 2; i++) {
        const int r = (i * 8 + wv) * 16 + lane / 4, piece = (lane & 3) ^ ((r >> 2) & 3);
        const RowRef x = row_ref(a, rg * 8 + r / 32, r & 31);
        const int64_t b = (int64_t)x.row * nb;
        s.q[i] = Q6 ? a.seg[x.seg].w + b * 128 + 16 * piece : a.seg[x.seg].w + b * 144 + 16 + 16 * piece;
    }
    const RowRef x = row_ref(a, rg * 8 + wv, lane & 31);
    const int64_t b = (int64_t)x.row * nb, NB = (int64_t)a.seg[x.seg].N * nb;
    const uint8_t *w = a.seg[x.seg].w;
    if constexpr (Q6) {
        s.hd = w + NB * 192 + b * 16;
        s.d = w + NB * 208 + b * 2;
        const RowRef y = row_ref(a, rg * 8 + wv, lane / 2);
        const int64_t by = (int64_t)y.row * nb, NBy = (int64_t)a.seg[y.seg].N * nb;
        s.qh = a.seg[y.seg].w + NBy * 128 + by * 64 + 16 * ((lane & 1) ^ ((lane >> 4) & 1));
    } else {
        s.hd = w + b * 144;
    }
}
template <bool Q6>
__device__ __forceinline__ void copy_w(const WSrc<Q6> &s, int blk, int half, uint32_t dst, int wv) {
#pragma unroll
    for (int i = 0; i < 2; i++)
        dma16(s.q[i] + (int64_t)blk * (Q6 ? 128 : 144) + 64 * half, dst + (i * 8 + wv) * 1024);
    if constexpr (Q6) dma16(s.qh + (int64_t)blk * 64 + 32 * half, dst + kRows * 64 + wv * 1024);
}

__device__ __forceinline__ void store_sys2(float *p, float x, float y) {
    const unsigned long long v = (unsigned long long)__float_as_uint(x) | ((unsigned long long)__float_as_uint(y) << 32);
    __hip_atomic_store((unsigned long long *)p, v, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_SYSTEM);
}
__device__ __forceinline__ unsigned long long load_sys2(const float *p) {
    return __hip_atomic_load((unsigned long long *)const_cast<float *>(p), __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_SYSTEM);
}

// Work-group whose range [w P / G, (w + 1) P / G) holds unit u.
__device__ __forceinline__ int wg_of(int64_t u, int64_t P, int G) { return (int)(((u + 1) * G - 1) / P); }

// Operands of a lane's row for kstep ks of a stage (inner elements 32 g +
// 16 hh + 8 (ks & 1) .. + 7 of the block, g the group).
// Q4_K: sc_g q from the 16 bytes of the group pair's chunk; header words 1..3
// hold the 6-bit scales (xj_quant.h:49-52).
__device__ __forceinline__ h8 q4_operand(u4 q, const uint32_t (&hw)[4], int g, int ks) {
    const uint32_t scw = g < 4 ? hw[1] & 0x3F3F3F3Fu : (hw[3] & 0x0F0F0F0Fu) | ((hw[1] >> 2) & 0x30303030u);
    const uint32_t sel = 0x04000400u | ((uint32_t)(g & 3) << 16) | (uint32_t)(g & 3);
    const h2 s2 = as_h2(__builtin_amdgcn_perm(0x64646464u, scw, sel)) - h2{1024, 1024};
    const h2 n2 = s2 * h2{-1024, -1024};
    const uint32_t w0 = q[2 * (ks & 1)], w1 = q[2 * (ks & 1) + 1];
    const uint32_t q0 = (ks >> 1 ? w0 >> 4 : w0) & 0x0F0F0F0Fu, q1 = (ks >> 1 ? w1 >> 4 : w1) & 0x0F0F0F0Fu;
    // (1024 + q) sc - 1024 sc = q sc, exact
    return cat8(fma2(biased01(q0), s2, n2), fma2(biased23(q0), s2, n2), fma2(biased01(q1), s2, n2), fma2(biased23(q1), s2, n2));
}
// Q6_K: sc (q - 32) = F + R. Group G = g & 3 of the half block: low nibbles of
// its bytes 32 (G & 1) .. (ql), high nibbles for G >= 2, two high bits at bit
// 2 G of qh; scale 2 g + hh is byte 2 (g & 1) + hh of word g / 2 (scw).
__device__ __forceinline__ void q6_operands(u4 ql, u4 qh, uint32_t scw, int g, int k, int hh, h8 &F, h8 &R) {
    const int G = g & 3, sh = G >> 1 ? 4 : 0, c = 2 * k;
    uint32_t q[2];
#pragma unroll
    for (int i = 0; i < 2; i++) {
        const uint32_t lo = (ql[c + i] >> sh) & 0x0F0F0F0Fu, hb = qh[c + i];
        q[i] = lo | ((G == 0 ? hb << 4 : G == 1 ? hb << 2 : G == 2 ? hb : hb >> 2) & 0x30303030u);
    }
    const _Float16 fs = (_Float16)(short)__builtin_amdgcn_sbfe((int)scw, 16 * (g & 1) + 8 * hh, 8);
    const h2 s2 = {fs, fs}, b = {-1056, -1056};
    const h2 x0 = biased01(q[0]) + b, x1 = biased23(q[0]) + b, x2 = biased01(q[1]) + b, x3 = biased23(q[1]) + b;
    const h2 f0 = x0 * s2, f1 = x1 * s2, f2 = x2 * s2, f3 = x3 * s2;
    F = cat8(f0, f1, f2, f3);
    R = cat8(fma2(x0, s2, -f0), fma2(x1, s2, -f1), fma2(x2, s2, -f2), fma2(x3, s2, -f3));
}

template <bool Q6>
__global__ __launch_bounds__(kThreads, 2) void gemm_wide_kernel(const WideArgs a) {
    using L = Lds<Q6>;
    extern __shared__ __align__(1024) uint8_t lds[];
    __shared__ int last_sh;
    const int tid = threadIdx.x, lane = tid & 63, wv = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int li = lane & 31, hh = lane >> 5, wm = wv & 3, wn = wv >> 2;
    const int nb = a.nb, G = a.G;
    // consecutive ranges on one XCD (work-groups are dealt to the 8 XCDs in turn)
    const int w = G % 8 == 0 ? (blockIdx.x & 7) * (G / 8) + (blockIdx.x >> 3) : blockIdx.x;
    const int64_t P = a.P;
    const int64_t u0 = w * P / G, u1 = (w + 1) * P / G;
    const uint32_t l0 = (uint32_t)(uintptr_t)(__attribute__((address_space(3))) uint8_t *)lds;
    const int first_tile = (int)(u0 / nb);
    int tile = first_tile, blk = (int)(u0 - (int64_t)tile * nb);
    int tg = tile / a.nrg, rg = tile - tg * a.nrg;
    WSrc<Q6> ws;
    wsrc<Q6>(a, rg, wv, lane, ws);
    // this wavefront's activation copies: token tile wv / 2, KBs 4 (wv & 1) .. + 3 of a stage
    auto rec = [&](int tg_, int blk_) {
        return a.wq + ((int64_t)(tg_ * kTokTiles + (wv >> 1)) * nb + blk_) * kWideRec + 16 * lane;
    };
    auto copy_act = [&](const uint8_t *r, int s, int buf) {
#pragma unroll
        for (int i = 0; i < 4; i++)
            dma16(r + s * kStageB + (4 * (wv & 1) + i) * 1024, l0 + L::ACT + buf * L::ACT_N + (wv >> 1) * kStageB + (4 * (wv & 1) + i) * 1024);
    };
    // headers, d words and the activations' sums and exponents of a block
    constexpr int kHdOps = Q6 ? 3 : 2, kWOps = Q6 ? 3 : 2;
    auto copy_hd = [&](const uint8_t *r, int blk_, int buf) {
        dma16(r + 4 * kStageB + 1024 * (wv & 1), l0 + L::AUX + buf * L::AUX_N + (wv >> 1) * kAux + 1024 * (wv & 1));
        if (lane < 32) {
            dma16(ws.hd + (int64_t)blk_ * (Q6 ? 16 : 144), l0 + L::HD + buf * L::HD_N + wv * 512);
            if constexpr (Q6)
                dma4((const uint8_t *)((uintptr_t)(ws.d + 2 * blk_) & ~(uintptr_t)3), l0 + L::D + buf * L::D_N + wv * 128);
        }
    };
    const uint8_t *r0 = rec(tg, blk);
    copy_hd(r0, blk, 0);
    copy_w<Q6>(ws, blk, 0, l0 + L::W, wv);
    copy_act(r0, 0, 0);
    f16v acc[2][2], s1[2][2];
#pragma unroll
    for (int t = 0; t < 2; t++)
#pragma unroll
        for (int r = 0; r < 2; r++) acc[t][r] = f16v(0.f);
    int bp = 0;   // buffer parity of this block's header and sums
    for (int64_t u = u0; u < u1; u++) {
        const bool more = u + 1 < u1;
        int tg2 = tg, rg2 = rg, blk2 = blk + 1;
        if (blk2 == nb) {
            blk2 = 0;
            if (++rg2 == a.nrg) rg2 = 0, tg2++;
        }
        uint32_t hw[2][4];   // Q4_K: this lane's rows' headers
        uint32_t dw[2];
#pragma unroll
        for (int s = 0; s < 4; s++) {
            // this stage's activations (and at even stages its weights) are in LDS
            if (s == 1) wait_vm<kWOps>();
            else if (s == 3 && more) wait_vm<kWOps + kHdOps>();
            else wait_vm<0>();
            stage_barrier();
            if (s < 3) copy_act(r0, s + 1, (s + 1) & 1);
            if (s == 0) copy_w<Q6>(ws, blk, 1, l0 + L::W + L::W_N, wv);
            if (s == 2 && more) {
                if (blk2 == 0) wsrc<Q6>(a, rg2, wv, lane, ws);
                r0 = rec(tg2, blk2);
                copy_hd(r0, blk2, bp ^ 1);
                copy_w<Q6>(ws, blk2, 0, l0 + L::W, wv);
            }
            if (s == 3 && more) copy_act(r0, 0, 0);
            uint32_t scw[2];   // Q6_K: the stage's four scales
#pragma unroll
            for (int rt = 0; rt < 2; rt++) {
                const int row = 64 * wm + 32 * rt + li;
                const uint8_t *hp = lds + L::HD + bp * L::HD_N + row * 16;
                if constexpr (Q6) {
                    scw[rt] = *(const uint32_t *)(hp + 4 * s);
                    if (s == 0) {   // d is the low or high half of its aligned word by its block index's parity
                        const RowRef x = row_ref(a, rg * 8 + row / 32, li);
                        const uint32_t v32 = *(const uint32_t *)(lds + L::D + bp * L::D_N + row * 4);
                        dw[rt] = (((int64_t)x.row * nb + blk) & 1) ? v32 >> 16 : v32 & 0xFFFFu;
                    }
                } else if (s == 0) {
                    const u4 v = *(const u4 *)hp;
#pragma unroll
                    for (int i = 0; i < 4; i++) hw[rt][i] = v[i];
                    dw[rt] = v[0];
                }
            }
            const uint8_t *wb = lds + L::W + (s >> 1) * L::W_N;
            const uint8_t *ab = lds + L::ACT + (s & 1) * L::ACT_N + 2 * wn * kStageB + 16 * lane;
            auto act = [&](int t, int ks, int plane) { return *(const h8 *)(ab + t * kStageB + (2 * ks + plane) * 1024); };
            const uint8_t *xb = lds + L::AUX + bp * L::AUX_N + 2 * wn * kAux;
            auto exps = [&](int t, f4 (&ex)[4]) {   // 2^e of the tokens 8 i + 4 hh .. + 3 of tile t
#pragma unroll
                for (int i = 0; i < 4; i++) ex[i] = *(const f4 *)(xb + t * kAux + 1024 + 4 * (8 * i + 4 * hh));
            };
            // the block's (Q6_K: the stage's) sums are added to the tile: lane = weight row li of its tile,
            // register i = token 8 (i / 4) + 4 hh + i % 4
            if constexpr (!Q6) {
                u4 qv[2];
#pragma unroll
                for (int rt = 0; rt < 2; rt++) {
                    const int row = 64 * wm + 32 * rt + li;
                    qv[rt] = *(const u4 *)(wb + row * 64 + 16 * ((2 * (s & 1) + hh) ^ ((row >> 2) & 3)));
                }
#pragma unroll
                for (int ks = 0; ks < 4; ks++) {
                    h8 ah[2], al[2], A[2];
#pragma unroll
                    for (int t = 0; t < 2; t++) ah[t] = act(t, ks, 0), al[t] = act(t, ks, 1);
#pragma unroll
                    for (int rt = 0; rt < 2; rt++) A[rt] = q4_operand(qv[rt], hw[rt], 2 * s + (ks >> 1), ks);
#pragma unroll
                    for (int rt = 0; rt < 2; rt++)
#pragma unroll
                        for (int t = 0; t < 2; t++) s1[t][rt] = mfma(ah[t], A[rt], s == 0 && ks == 0 ? f16v(0.f) : s1[t][rt]);
#pragma unroll
                    for (int rt = 0; rt < 2; rt++)
#pragma unroll
                        for (int t = 0; t < 2; t++) s1[t][rt] = mfma(al[t], A[rt], s1[t][rt]);
                }
                if (s == 3) {
                    h8 mB[2];
#pragma unroll
                    for (int rt = 0; rt < 2; rt++) {
                        const uint32_t m0 = hw[rt][2] & 0x3F3F3F3Fu,
                                       m1 = ((hw[rt][3] >> 4) & 0x0F0F0F0Fu) | ((hw[rt][2] >> 2) & 0x30303030u);
                        const h2 b = {-1024, -1024};
                        mB[rt] = cat8(biased01(m0) + b, biased23(m0) + b, biased01(m1) + b, biased23(m1) + b);
                    }
#pragma unroll
                    for (int t = 0; t < 2; t++) {
                        f4 ex[4];
                        exps(t, ex);
                        const h8 sx = *(const h8 *)(xb + t * kAux + 16 * lane);
#pragma unroll
                        for (int rt = 0; rt < 2; rt++) {
                            const float d = xjd::f16_to_f32(dw[rt] & 0xFFFFu);
                            const float dm = -32.f * xjd::f16_to_f32(dw[rt] >> 16);   // the sums are stored / 32
                            const f16v m = mfma(sx, mB[rt], f16v(0.f));
#pragma unroll
                            for (int i = 0; i < 16; i++)
                                acc[t][rt][i] = fmaf(ex[i >> 2][i & 3], fmaf(dm, m[i], d * s1[t][rt][i]), acc[t][rt][i]);
                        }
                    }
                }
            } else {
                // every operand of the stage, then per token tile the small terms R hi + F lo, then F hi; each
                // stage is added to the tile by itself: few roundings at full magnitude (relative error 0.9e-7
                // at K = 256 against 1.6e-7 with one sum per block in the Q4_K order, and 1.0e-7 in gemm.hip)
                h8 F[4][2], R[4][2];
#pragma unroll
                for (int rt = 0; rt < 2; rt++) {
                    const int row = 64 * wm + 32 * rt + li;
                    const u4 qh = *(const u4 *)(wb + kRows * 64 + row * 32 + 16 * (hh ^ ((row >> 3) & 1)));
#pragma unroll
                    for (int p = 0; p < 2; p++) {
                        const u4 ql = *(const u4 *)(wb + row * 64 + 16 * ((2 * p + hh) ^ ((row >> 2) & 3)));
#pragma unroll
                        for (int k = 0; k < 2; k++) q6_operands(ql, qh, scw[rt], 2 * s + p, k, hh, F[2 * p + k][rt], R[2 * p + k][rt]);
                    }
                }
#pragma unroll
                for (int t = 0; t < 2; t++) {
                    f16v z[2] = {f16v(0.f), f16v(0.f)};
#pragma unroll
                    for (int ks = 0; ks < 4; ks++) {
                        const h8 ah = act(t, ks, 0), al = act(t, ks, 1);
#pragma unroll
                        for (int rt = 0; rt < 2; rt++) z[rt] = mfma(ah, R[ks][rt], z[rt]);
#pragma unroll
                        for (int rt = 0; rt < 2; rt++) z[rt] = mfma(al, F[ks][rt], z[rt]);
                    }
#pragma unroll
                    for (int ks = 0; ks < 4; ks++) {
                        const h8 ah = act(t, ks, 0);
#pragma unroll
                        for (int rt = 0; rt < 2; rt++) z[rt] = mfma(ah, F[ks][rt], z[rt]);
                    }
                    f4 ex[4];
                    exps(t, ex);
#pragma unroll
                    for (int rt = 0; rt < 2; rt++) {
                        const float d = xjd::f16_to_f32(dw[rt] & 0xFFFFu);
#pragma unroll
                        for (int i = 0; i < 16; i++) acc[t][rt][i] = fmaf(ex[i >> 2][i & 3], d * z[rt][i], acc[t][rt][i]);
                    }
                    // (added here and now: the compiler would otherwise keep the sums of several stages)
                    asm volatile("" : "+v"(acc[t][0]), "+v"(acc[t][1]));
                }
            }
        }
        bp ^= 1;
        if (!more || blk2 == 0) {   // the last of this tile's blocks here (uniform)
            const int64_t first = (int64_t)tile * nb;
            const int wf = wg_of(first, P, G), wl = wg_of(first + nb - 1, P, G);
            bool store = wf == wl;
            if (!store) {
                // slot 0 of a work-group: the tile its range starts in, slot 1: the one it ends in
                float *slot = a.part + (int64_t)(2 * w + (tile != first_tile)) * (kRows * kToks) + wv * 4096 + 2 * lane;
#pragma unroll
                for (int t = 0; t < 2; t++)
#pragma unroll
                    for (int r = 0; r < 2; r++)
#pragma unroll
                        for (int i = 0; i < 8; i++)
                            store_sys2(slot + ((t * 2 + r) * 8 + i) * 128, acc[t][r][2 * i], acc[t][r][2 * i + 1]);
                store = xjd::arrive_last(a.cnt + tile, wl - wf + 1, &last_sh);
                if (store) {
#pragma unroll
                    for (int t = 0; t < 2; t++)
#pragma unroll
                        for (int r = 0; r < 2; r++) acc[t][r] = f16v(0.f);
                    for (int x = wf; x <= wl; x++) {
                        const int ft = (int)((x * P / G) / nb);
                        const float *src = a.part + (int64_t)(2 * x + (tile != ft)) * (kRows * kToks) + wv * 4096 + 2 * lane;
#pragma unroll
                        for (int t = 0; t < 2; t++)
#pragma unroll
                            for (int r = 0; r < 2; r++) {
                                unsigned long long v[8];
#pragma unroll
                                for (int i = 0; i < 8; i++) v[i] = load_sys2(src + ((t * 2 + r) * 8 + i) * 128);
#pragma unroll
                                for (int i = 0; i < 8; i++) {
                                    acc[t][r][2 * i] += __uint_as_float((uint32_t)v[i]);
                                    acc[t][r][2 * i + 1] += __uint_as_float((uint32_t)(v[i] >> 32));
                                }
                            }
                    }
                }
            }
            if (store) {
                float *tsc = (float *)(lds + L::TSC);
                if (a.ss) {   // an RMSNorm input's scale per token, from the blocks' sums of x^2
                    if (tid < kToks) {
                        const int t = min(tg * kToks + tid, a.T - 1);
                        double sum = 0;
                        for (int b = 0; b < nb; b++) sum += a.ss[(int64_t)b * a.ss_n + t];
                        tsc[tid] = 1.0f / sqrtf((float)(sum / a.K) + a.eps);
                    }
                    __syncthreads();
                }
#pragma unroll
                for (int r = 0; r < 2; r++) {
                    const int rt = rg * 8 + 2 * wm + r;
                    if (rt >= a.rt0[a.nseg]) continue;
                    int sgi = 0;
#pragma unroll
                    for (int k = 1; k < kGemmMaxSeg; k++) sgi += k < a.nseg && rt >= a.rt0[k];
                    const GemmSeg &sg = a.seg[sgi];
                    const int row = (rt - a.rt0[sgi]) * 32 + li, rc = min(row, sg.N - 1);
#pragma unroll
                    for (int t = 0; t < 2; t++) {
                        // register i: token t0 + 8 (i / 4) + i % 4; what is read past T or N is not stored
                        const int tl0 = 64 * wn + 32 * t + 4 * hh, t0 = tg * kToks + tl0;
                        float *yp = sg.y + (int64_t)t0 * sg.ys + rc;
                        f16v v = acc[t][r];
                        if (a.ss) {
#pragma unroll
                            for (int i = 0; i < 4; i++) {
                                const f4 sc = *(const f4 *)(tsc + tl0 + 8 * i);
#pragma unroll
                                for (int k = 0; k < 4; k++) v[4 * i + k] *= sc[k];
                            }
                        }
                        if (sg.add) {
                            float old[16];
#pragma unroll
                            for (int i = 0; i < 16; i++) {
                                const int o = 8 * (i >> 2) + (i & 3);
                                old[i] = sg.y[(int64_t)min(t0 + o, a.T - 1) * sg.ys + rc];
                            }
#pragma unroll
                            for (int i = 0; i < 16; i++) v[i] = old[i] + v[i];
                        }
#pragma unroll
                        for (int i = 0; i < 16; i++) {
                            const int o = 8 * (i >> 2) + (i & 3);
                            if (row < sg.N && t0 + o < a.T) yp[(int64_t)o * sg.ys] = v[i];
                        }
                    }
                }
            }
#pragma unroll
            for (int t = 0; t < 2; t++)
#pragma unroll
                for (int r = 0; r < 2; r++) acc[t][r] = f16v(0.f);
            if (rg2 != rg || tg2 != tg) tile++;
        }
        blk = blk2; rg = rg2; tg = tg2;
    }
}

// ------------------------------------------------------- 33..64 tokens --
// The same products for a chunk of up to 64 tokens: a work-group takes few rows
// (RT tiles of 16), all tokens and a range of the inner elements, which its
// eight wavefronts share in contiguous chunks of 64 elements, each with sums of
// its own for the whole tile on v_mfma_f32_16x16x32_f16 (tokens as rows of a
// tile, weight rows as its columns). Every weight is decoded once; weights and
// activations go straight to registers (the activation records' order serves
// this operand too: group g's elements 8 kq .. + 7 are kstep kq & 1 of half
// kq >> 1), no wavefront waits for another before the end, and only there the
// sums meet, through LDS. Few rows (a 2560-row matrix is 160 tiles) are split
// over the inner elements as well, the partial tiles added in order by the last
// work-group to arrive.
// It is bound by the latency of each chunk's activations at two wavefronts per
// SIMD and by the 655 KB (K = 2560) of them that every work-group reads from
// L2. 64 tokens: 18432 x 2560 Q4_K 37.4 -> 28.0 us, 2560 x 4096 Q4_K 24.0 ->
// 13.5, 2560 x 9216 Q6_K 37.3 -> 27.8, against 128-row groups whose weights
// were decoded twice and whose K ranges met through HBM. Its error against
// float64 is no larger (Q4_K 2.4..3.1e-7 against 3.9..4.9e-7, Q6_K 0.9..1.3e-7
// against 1.0..1.5e-7, inputs normal or heavy-tailed: shorter sums).
// Below 33 tokens gemm.hip's kernels are as fast or faster (2560 x 9216 Q6_K at
// 16: 15 against 20 us).
template <bool Q6, int RT>
struct SkW {
    u2 q[RT][Q6 ? 3 : 1];   // Q4_K: the chunk's 8 bytes; Q6_K: low nibbles of its two groups, high bits
    u4 hd[RT];              // Q4_K header, Q6_K scales
    uint32_t d[RT];         // Q6_K
};

template <bool Q6, int RT, int NT>
__global__ __launch_bounds__(512, 2) void gemm_skinny_kernel(const WideArgs a) {
    extern __shared__ __align__(16) float red[];   // four wavefronts' sums
    __shared__ int last_sh;
    __shared__ float tsc[16 * NT];
    const int tid = threadIdx.x, lane = tid & 63, wv = __builtin_amdgcn_readfirstlane(tid >> 6), li = lane & 15, kq = lane >> 4;
    const int nb = a.nb, rg = blockIdx.x / a.G, ks = blockIdx.x - rg * a.G;   // row group, split
    const int C = 4 * nb, s0 = ks * C / a.G, s1 = (ks + 1) * C / a.G;
    const int c0 = s0 + wv * (s1 - s0) / 8, c1 = s0 + (wv + 1) * (s1 - s0) / 8;   // this wavefront's chunks
    const uint8_t *wp[RT];    // Q4_K: the row's blocks; Q6_K: its ql plane
    int64_t b0[RT], NB[RT];
#pragma unroll
    for (int r = 0; r < RT; r++) {
        const int tile = min(rg * RT + r, a.rt0[a.nseg] - 1);
        int sg = 0;
#pragma unroll
        for (int k = 1; k < kGemmMaxSeg; k++) sg += k < a.nseg && tile >= a.rt0[k];
        const int row = min((tile - a.rt0[sg]) * 16 + li, a.seg[sg].N - 1);
        wp[r] = Q6 ? a.seg[sg].w : a.seg[sg].w + (int64_t)row * nb * 144;
        b0[r] = (int64_t)row * nb;   // (Q6_K only)
        NB[r] = (int64_t)a.seg[sg].N * nb;
    }
    auto load_w = [&](int c, SkW<Q6, RT> &w) {
        const int blk = c >> 2, p = c & 3;
#pragma unroll
        for (int r = 0; r < RT; r++) {
            if constexpr (!Q6) {
                const uint8_t *x = wp[r] + blk * 144;
                w.q[r][0] = *(const u2 *)(x + 16 + 32 * p + 8 * kq);
                w.hd[r] = *(const u4 *)x;
            } else {
                const int64_t b = b0[r] + blk;
                const uint8_t *ql = wp[r] + b * 128 + 64 * (p >> 1) + 8 * kq;
                w.q[r][0] = *(const u2 *)ql;
                w.q[r][1] = *(const u2 *)(ql + 32);
                w.q[r][2] = *(const u2 *)(wp[r] + NB[r] * 128 + b * 64 + 32 * (p >> 1) + 8 * kq);
                w.hd[r][0] = *(const uint32_t *)(wp[r] + NB[r] * 192 + b * 16 + 4 * p);
                w.d[r] = *(const uint16_t *)(wp[r] + NB[r] * 208 + b * 2);
            }
        }
    };
    // a chunk's activations of token tile t (16 tokens), two planes of its two groups
    struct Act {
        h8 h[2], l[2];
        f4 ex;   // 2^e of tokens 16 t + 4 kq .. + 3
    };
    auto load_x = [&](int c, int t, Act &x) {
        const int blk = c >> 2, p = c & 3;
        const uint8_t *rec = a.wq + ((int64_t)(t >> 1) * nb + blk) * kWideRec;
        const uint8_t *y = rec + p * kStageB + (kq & 1) * 2048 + ((kq >> 1) * 32 + 16 * (t & 1) + li) * 16;
#pragma unroll
        for (int g = 0; g < 2; g++) {
            x.h[g] = *(const h8 *)(y + g * 4096);
            x.l[g] = *(const h8 *)(y + g * 4096 + 1024);
        }
        x.ex = *(const f4 *)(rec + 4 * kStageB + 1024 + 4 * (16 * (t & 1) + 4 * kq));
    };
    f4 acc[RT][NT];
#pragma unroll
    for (int r = 0; r < RT; r++)
#pragma unroll
        for (int t = 0; t < NT; t++) acc[r][t] = f4{0.f, 0.f, 0.f, 0.f};
    constexpr bool kAhead = RT * NT < 20;   // registers for the next chunk's weights
    SkW<Q6, RT> w;
    if (kAhead && c0 < c1) load_w(c0, w);
    for (int c = c0; c < c1; c++) {
        const int blk = c >> 2, p = c & 3;
        if (!kAhead) load_w(c, w);
        Act x[2];   // token tiles in turn, the one after next requested when one is done
        load_x(c, 0, x[0]);
        if constexpr (NT > 1) load_x(c, 1, x[1]);
        // the weights' operands; the next chunk's weights are in flight from here
        h8 A[RT][2], R[Q6 ? RT : 1][2], mB[Q6 ? 1 : RT];
        float d[RT], dm[RT];
#pragma unroll
        for (int r = 0; r < RT; r++) {
            if constexpr (!Q6) {
                d[r] = xjd::f16_to_f32(w.hd[r][0] & 0xFFFFu);
                dm[r] = -32.f * xjd::f16_to_f32(w.hd[r][0] >> 16);   // the group sums are stored / 32
                const uint32_t lo = p < 2 ? w.hd[r][1] & 0x3F3F3F3Fu : (w.hd[r][3] & 0x0F0F0F0Fu) | ((w.hd[r][1] >> 2) & 0x30303030u);
                const uint32_t sc2 = lo >> (16 * (p & 1));   // scales of groups 2 p and 2 p + 1 (xj_quant.h:49-52)
#pragma unroll
                for (int g = 0; g < 2; g++) {
                    const h2 s2 = as_h2(__builtin_amdgcn_perm(0x64646464u, sc2, g ? 0x04010401u : 0x04000400u)) - h2{1024, 1024};
                    const h2 n2 = s2 * h2{-1024, -1024};
                    const uint32_t q0 = (g ? w.q[r][0][0] >> 4 : w.q[r][0][0]) & 0x0F0F0F0Fu,
                                   q1 = (g ? w.q[r][0][1] >> 4 : w.q[r][0][1]) & 0x0F0F0F0Fu;
                    A[r][g] = cat8(fma2(biased01(q0), s2, n2), fma2(biased23(q0), s2, n2), fma2(biased01(q1), s2, n2),
                                   fma2(biased23(q1), s2, n2));
                }
                if (p == 0) {   // (uniform) the block's minimum terms with its first chunk
                    const uint32_t m0 = w.hd[r][2] & 0x3F3F3F3Fu,
                                   m1 = ((w.hd[r][3] >> 4) & 0x0F0F0F0Fu) | ((w.hd[r][2] >> 2) & 0x30303030u);
                    const h2 b = {-1024, -1024};
                    mB[r] = cat8(biased01(m0) + b, biased23(m0) + b, biased01(m1) + b, biased23(m1) + b);
                }
            } else {
                d[r] = xjd::f16_to_f32(w.d[r]);
#pragma unroll
                for (int g = 0; g < 2; g++) {
                    const int G = 2 * (p & 1) + g;   // low nibbles for G < 2, high bits at bit 2 G
                    uint32_t q[2];
#pragma unroll
                    for (int i = 0; i < 2; i++) {
                        const uint32_t l4 = (p & 1 ? w.q[r][g][i] >> 4 : w.q[r][g][i]) & 0x0F0F0F0Fu;
                        q[i] = l4 | (((w.q[r][2][i] >> (2 * G)) & 0x03030303u) << 4);
                    }
                    // scale 2 (2 p + g) + kq / 2: byte 2 g + kq / 2 of the chunk's word
                    const _Float16 fs = (_Float16)(short)__builtin_amdgcn_sbfe((int)w.hd[r][0], 16 * g + 8 * (kq >> 1), 8);
                    const h2 s2 = {fs, fs}, b = {-1056, -1056};
                    const h2 x0 = biased01(q[0]) + b, x1 = biased23(q[0]) + b, x2 = biased01(q[1]) + b, x3 = biased23(q[1]) + b;
                    const h2 f0 = x0 * s2, f1 = x1 * s2, f2 = x2 * s2, f3 = x3 * s2;
                    A[r][g] = cat8(f0, f1, f2, f3);
                    R[r][g] = cat8(fma2(x0, s2, -f0), fma2(x1, s2, -f1), fma2(x2, s2, -f2), fma2(x3, s2, -f3));
                }
            }
        }
        if (kAhead && c + 1 < c1) load_w(c + 1, w);
#pragma unroll
        for (int t = 0; t < NT; t++) {
            const Act &y = x[t & 1];
            f4 z[RT];
#pragma unroll
            for (int r = 0; r < RT; r++) z[r] = f4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
            for (int g = 0; g < 2; g++) {   // the small terms first
                if constexpr (Q6)
#pragma unroll
                    for (int r = 0; r < RT; r++) z[r] = mfma16(y.h[g], R[r][g], z[r]);
#pragma unroll
                for (int r = 0; r < RT; r++) z[r] = mfma16(y.l[g], A[r][g], z[r]);
            }
#pragma unroll
            for (int g = 0; g < 2; g++)
#pragma unroll
                for (int r = 0; r < RT; r++) z[r] = mfma16(y.h[g], A[r][g], z[r]);
#pragma unroll
            for (int r = 0; r < RT; r++) acc[r][t] = acc[r][t] + y.ex * (z[r] * d[r]);
            if constexpr (!Q6) {
                if (p == 0) {   // eight groups' sums, hi in lanes kq = 0, lo in kq = 1
                    const h8 v = *(const h8 *)(a.wq + ((int64_t)(t >> 1) * nb + blk) * kWideRec + 4 * kStageB + 512 * (kq & 1) +
                                               (16 * (t & 1) + li) * 16);
                    const h8 sx = kq < 2 ? v : h8{0, 0, 0, 0, 0, 0, 0, 0};
#pragma unroll
                    for (int r = 0; r < RT; r++)
                        acc[r][t] = acc[r][t] + y.ex * (mfma16(sx, mB[r], f4{0.f, 0.f, 0.f, 0.f}) * dm[r]);
                }
            }
            if (t + 2 < NT) load_x(c, t + 2, x[t & 1]);
        }
    }
    // the wavefronts' sums: 4..7 to 0..3, then the four copies to every thread's elements
    f4 *rv = (f4 *)red;
    constexpr int NV = RT * NT;   // f4 per lane
    if (wv >= 4)
#pragma unroll
        for (int i = 0; i < NV; i++) rv[((wv - 4) * NV + i) * 64 + lane] = acc[i / NT][i % NT];
    __syncthreads();
    if (wv < 4)
#pragma unroll
        for (int i = 0; i < NV; i++) acc[i / NT][i % NT] = acc[i / NT][i % NT] + rv[(wv * NV + i) * 64 + lane];
    __syncthreads();
    if (wv < 4)
#pragma unroll
        for (int i = 0; i < NV; i++) rv[(wv * NV + i) * 64 + lane] = acc[i / NT][i % NT];
    if (a.ss) {   // an RMSNorm input's scale per token, from the blocks' sums of x^2
        if (tid < 16 * NT) {
            const int t = min(tid, a.T - 1);
            double sum = 0;
            for (int b = 0; b < nb; b++) sum += a.ss[(int64_t)b * a.ss_n + t];
            tsc[tid] = 1.0f / sqrtf((float)(sum / a.K) + a.eps);
        }
    }
    __syncthreads();
    constexpr int NE = (NV * 64 + 511) / 512;   // f4 elements per thread: (tile pair i, lane)
    f4 v[NE];
#pragma unroll
    for (int j = 0; j < NE; j++) {
        const int e = min(tid + 512 * j, NV * 64 - 1);
        v[j] = (rv[e] + rv[NV * 64 + e]) + (rv[2 * NV * 64 + e] + rv[3 * NV * 64 + e]);
    }
    if (a.G > 1) {
        float *slot = a.part + (int64_t)blockIdx.x * (NV * 256);
#pragma unroll
        for (int j = 0; j < NE; j++) {
            const int e = tid + 512 * j;
            if (e >= NV * 64) continue;
            store_sys2(slot + 4 * e, v[j][0], v[j][1]);
            store_sys2(slot + 4 * e + 2, v[j][2], v[j][3]);
        }
        if (!xjd::arrive_last(a.cnt + rg, a.G, &last_sh)) return;
#pragma unroll
        for (int j = 0; j < NE; j++) v[j] = f4{0.f, 0.f, 0.f, 0.f};
        for (int x = 0; x < a.G; x++) {
            const float *src = a.part + (int64_t)(rg * a.G + x) * (NV * 256);
            unsigned long long u[NE][2];
#pragma unroll
            for (int j = 0; j < NE; j++) {
                const int e = min(tid + 512 * j, NV * 64 - 1);
                u[j][0] = load_sys2(src + 4 * e);
                u[j][1] = load_sys2(src + 4 * e + 2);
            }
#pragma unroll
            for (int j = 0; j < NE; j++)
#pragma unroll
                for (int k = 0; k < 2; k++) {
                    v[j][2 * k] += __uint_as_float((uint32_t)u[j][k]);
                    v[j][2 * k + 1] += __uint_as_float((uint32_t)(u[j][k] >> 32));
                }
        }
    }
#pragma unroll
    for (int j = 0; j < NE; j++) {
        const int e = tid + 512 * j, i = e >> 6, el = e & 63, r = i / NT, t = i - r * NT;
        const int tile = rg * RT + r;
        if (e >= NV * 64 || tile >= a.rt0[a.nseg]) continue;
        int sgi = 0;
#pragma unroll
        for (int k = 1; k < kGemmMaxSeg; k++) sgi += k < a.nseg && tile >= a.rt0[k];
        const GemmSeg &sg = a.seg[sgi];
        const int row = (tile - a.rt0[sgi]) * 16 + (el & 15);
#pragma unroll
        for (int k = 0; k < 4; k++) {
            const int tok = 16 * t + 4 * (el >> 4) + k;
            if (row >= sg.N || tok >= a.T) continue;
            float *yp = sg.y + (int64_t)tok * sg.ys + row;
            const float y = a.ss ? v[j][k] * tsc[tok] : v[j][k];
            *yp = sg.add ? *yp + y : y;
        }
    }
}

// The activations of 32 tokens and one 256-element block, in the order the
// GEMM's lanes read them. A wavefront takes four tokens, a lane four
// consecutive elements k = 4 lane ..; the record is built in LDS and written
// in one piece. What it holds for tokens past T reaches their own sums only,
// which are never stored.
__global__ __launch_bounds__(512) void wide_prep_kernel(const WidePrep a) {
    __shared__ __align__(16) uint8_t rec[kWideRec];
    const int blk = blockIdx.x, tt = blockIdx.y, tid = threadIdx.x, lane = tid & 63, wv = tid >> 6;
    const int k = blk * 256 + 4 * lane;
    const int g = lane >> 3, idx = 4 * (lane & 7), half = idx >> 4, ks = 2 * (g & 1) + ((idx >> 3) & 1);
    f4 pw = {1.f, 1.f, 1.f, 1.f};
    if (a.pro == PRO_RMSU) pw = *(const f4 *)(a.pro_w + k);
    if (a.pro == PRO_GATED_RMS) pw = *(const f4 *)(a.pro_w + k % a.group);
    f4 xr[4], zr[4];
#pragma unroll
    for (int j = 0; j < 4; j++) {
        const int t = min(tt * 32 + wv * 4 + j, a.T - 1);
        xr[j] = *(const f4 *)(a.x + (int64_t)t * a.xs + k);
        if (a.x2) zr[j] = *(const f4 *)(a.x2 + (int64_t)t * a.x2s + k);
    }
#pragma unroll
    for (int j = 0; j < 4; j++) {
        const int tl = wv * 4 + j, t = tt * 32 + tl;
        if (t >= a.T) break;   // uniform over the wavefront
        f4 v = xr[j];
        if (a.pro == PRO_RMSU) {
            double ss = 0;
#pragma unroll
            for (int i = 0; i < 4; i++) ss += (double)v[i] * v[i];
            ss = xjd::wave_sum_d(ss);
            if (lane == 0) a.ss[(int64_t)blk * a.T + t] = ss;
            v = v * pw;
        } else if (a.pro == PRO_SWIGLU) {
#pragma unroll
            for (int i = 0; i < 4; i++) v[i] = xjd::silu(v[i]) * zr[j][i];
        } else if (a.pro == PRO_GATED_RMS) {
            double ss = 0;
#pragma unroll
            for (int i = 0; i < 4; i++) ss += (double)v[i] * v[i];
            for (int off = 1; off < a.group / 4; off <<= 1) ss += __shfl_xor(ss, off, 64);   // group 64 or 128
            const float sc = 1.0f / sqrtf((float)(ss / a.group) + a.eps);
#pragma unroll
            for (int i = 0; i < 4; i++) v[i] = v[i] * sc * pw[i] * xjd::silu(zr[j][i]);
        }
        const float m = xjd::wave_max(fmaxf(fmaxf(fabsf(v[0]), fabsf(v[1])), fmaxf(fabsf(v[2]), fabsf(v[3]))));
        int E = 0;
        (void)frexpf(m, &E);   // m < 2^E
        if (E < -100) E = -100;
        const int e = E - 14;
        h4 hi, lo;
        float r = 0.f;
#pragma unroll
        for (int i = 0; i < 4; i++) {
            const float s = ldexpf(v[i], -e);
            hi[i] = (_Float16)s;
            lo[i] = (_Float16)(s - (float)hi[i]);   // s - hi is exact in fp32
            r += (float)hi[i] + (float)lo[i];
        }
        for (int off = 1; off < 8; off <<= 1) r += __shfl_xor(r, off, 64);
        uint8_t *p = rec + (g >> 1) * kStageB + 2 * ks * 1024 + (half * 32 + tl) * 16 + (idx & 7) * 2;
        *(h4 *)p = hi;
        *(h4 *)(p + 1024) = lo;
        if ((lane & 7) == 0) {   // group sums / 32 (below the f16 limit): lanes 0..31 of the operand hi, 32..63 lo
            const float q = r * 0.03125f;
            const _Float16 qh = (_Float16)q;
            ((_Float16 *)(rec + 4 * kStageB + tl * 16))[g] = qh;
            ((_Float16 *)(rec + 4 * kStageB + 512 + tl * 16))[g] = (_Float16)(q - (float)qh);
        }
        if (lane == 0) ((float *)(rec + 4 * kStageB + 1024))[tl] = ldexpf(1.0f, e);
    }
    __syncthreads();
    uint8_t *dst = a.wq + ((int64_t)tt * a.nb + blk) * kWideRec;
    for (int i = tid; i < (4 * kStageB + 1024 + 128) / 16; i += 512) ((u4 *)dst)[i] = ((const u4 *)rec)[i];
}

int wide_cus() {
    static int n = 0;
    if (!n) {
        int dev = 0;
        if (hipGetDevice(&dev) != hipSuccess || hipDeviceGetAttribute(&n, hipDeviceAttributeMultiprocessorCount, dev) != hipSuccess || n < 1)
            n = 256;
    }
    return n;
}

template <bool Q6>
int launch_w(const WideArgs &a, hipStream_t st) {
    static const bool raised = hipFuncSetAttribute((const void *)gemm_wide_kernel<Q6>, hipFuncAttributeMaxDynamicSharedMemorySize,
                                                   Lds<Q6>::SIZE) == hipSuccess;
    if (!raised) return -1;
    hipLaunchKernelGGL((gemm_wide_kernel<Q6>), dim3(a.G), dim3(kThreads), Lds<Q6>::SIZE, st, a);
    return hipGetLastError() == hipSuccess ? 0 : -1;
}

template <bool Q6, int RT, int NT>
int launch_s3(const WideArgs &a, int grid, hipStream_t st) {
    constexpr int lds = 4 * RT * NT * 64 * 16;
    static const bool raised = hipFuncSetAttribute((const void *)gemm_skinny_kernel<Q6, RT, NT>,
                                                   hipFuncAttributeMaxDynamicSharedMemorySize, lds) == hipSuccess;
    if (!raised) return -1;
    hipLaunchKernelGGL((gemm_skinny_kernel<Q6, RT, NT>), dim3(grid), dim3(512), lds, st, a);
    return hipGetLastError() == hipSuccess ? 0 : -1;
}
template <bool Q6, int RT>
int launch_s2(const WideArgs &a, int grid, hipStream_t st) {
    return a.T <= 48 ? launch_s3<Q6, RT, 3>(a, grid, st) : launch_s3<Q6, RT, 4>(a, grid, st);
}

// Row tiles per work-group and splits of the inner elements: the least cost in
// units of a wavefront's chunk: the rounds of work-groups over the CUs times the
// chunks' row tiles (dearer with the token tiles) and a fixed part, and for a
// split the adding. Measured best at 37 and 64 tokens: 18432 x 2560 five tiles
// unsplit (28.0 us at 64; three tiles 36.1), 12352 x 2560 four (22.4; five
// 26.0), 2560 x 4096 two in three splits (13.5; one unsplit 17.7), 2560 x 9216
// Q6_K two in three (27.8; three in four 31.0).
struct SkPlan {
    int rt, ks;
    double cost;
};
SkPlan skinny_plan(bool q6, int tiles, int nb, int nt) {
    SkPlan best{1, 1, 0.0};
    double lo = 1e30;
    for (int rt = 1; rt <= (q6 ? 3 : 5); rt++)
        for (int ks = 1; ks <= 16 && ks <= nb; ks++) {
            const int wgs = (tiles + rt - 1) / rt * ks, rounds = (wgs + wide_cus() - 1) / wide_cus();
            if (ks > 1 && rounds > 1) break;
            const int cw = ((4 * nb + ks - 1) / ks + 7) / 8;
            const double c = rounds * ((rt * (0.5 + 0.5 * nt) + 1.5) * cw + 4.0) + (ks > 1 ? 6.0 + 0.5 * rt * ks : 0.0);
            if (c < lo) lo = c, best = SkPlan{rt, ks, c};
        }
    return best;
}

// Whether T > 64 tokens go as slices of 64 on the narrow kernel: the wide one's
// tiles are few for small matrices, each shared by many work-groups whose
// partial sums one of them adds. Estimates in us, fitted to both kernels (wide /
// slices): 2560 x 4096 Q4_K at 128 tokens 46 / 27, at 192 50 / 42, at 256 51 /
// 57; 2560 x 9216 Q6_K at 128 84 / 55, at 192 77 / 82; 7168 x 1024 Q4_K at 128
// 23 / 16, at 256 27 / 33; 18432 x 2560 Q4_K at 128 45 / 55.
bool in_slices(const WideArgs &a, int rows16) {
    const bool q6 = a.type == XJ_Q6_K;
    const double slice = 2.5 + (q6 ? 0.45 : 0.38) * skinny_plan(q6, rows16, a.nb, 4).cost;
    const int64_t tiles = (int64_t)((rows16 + 15) / 16) * ((a.T + kToks - 1) / kToks), P = tiles * a.nb;
    const int64_t units = (P + wide_cus() - 1) / wide_cus(), share = (a.nb + units - 1) / units;
    const double wide = 10.0 + (q6 ? 10.0 : 9.0) * units + 1.8 * share;
    return (a.T + kSkinnyT - 1) / kSkinnyT * slice < wide;
}

}  // namespace

size_t wide_wq_bytes(int K, int T) {
    return (size_t)((T + kToks - 1) / kToks) * kTokTiles * (K / 256) * kWideRec;
}
int64_t wide_part_floats(int T) {
    const int64_t skinny = (int64_t)wide_cus() * 5 * 4 * 256;
    return T <= kSkinnyT ? skinny : std::max(skinny, (int64_t)2 * wide_cus() * kRows * kToks);
}
int wide_counters(int64_t rows, int T) {
    const int64_t tiles = ((rows + 32 * kGemmMaxSeg + kRows - 1) / kRows + 1) * ((T + kToks - 1) / kToks);
    return (int)(T <= kSkinnyT ? wide_cus() : std::max<int64_t>(wide_cus(), tiles));
}

int wide_prep_launch(const WidePrep &in, hipStream_t st) {
    WidePrep a = in;
    if (!a.x || !a.wq || a.K < 256 || a.K % 256 || a.T < 1 || ((uintptr_t)a.x & 15) || (a.xs & 3) || ((uintptr_t)a.wq & 15)) return -1;
    const bool two = a.pro == PRO_SWIGLU || a.pro == PRO_GATED_RMS;
    if (!two) a.x2 = nullptr;
    if (two && (!a.x2 || ((uintptr_t)a.x2 & 15) || (a.x2s & 3))) return -1;
    if (a.pro == PRO_RMSU && (!a.ss || !a.pro_w || ((uintptr_t)a.pro_w & 15))) return -1;
    if (a.pro == PRO_GATED_RMS && ((a.group != 64 && a.group != 128) || !a.pro_w || ((uintptr_t)a.pro_w & 15))) return -1;
    if (a.pro != PRO_NONE && a.pro != PRO_RMSU && !two) return -1;
    a.nb = a.K / 256;
    hipLaunchKernelGGL(wide_prep_kernel, dim3(a.nb, (a.T + 31) / 32), dim3(512), 0, st, a);
    return hipGetLastError() == hipSuccess ? 0 : -1;
}

int gemm_wide_kind(const WideArgs &in) {
    WideArgs a = in;
    a.nb = a.K / 256;
    int rows16 = 0;
    for (int i = 0; i < a.nseg; i++) rows16 += (a.seg[i].N + 15) / 16;
    return a.T <= kSkinnyT ? 0 : in_slices(a, rows16) ? 1 : 2;
}

int gemm_wide_launch(const WideArgs &in, int64_t part_floats, int n_cnt, hipStream_t st) {
    WideArgs a = in;
    if (!a.ss_n) a.ss_n = a.T;
    if ((a.type != XJ_Q4_K && a.type != XJ_Q6_K) || a.K < 256 || a.K % 256 || a.T < 1 || a.nseg < 1 || a.nseg > kGemmMaxSeg ||
        !a.wq || !a.part || !a.cnt || ((uintptr_t)a.wq & 15))
        return -1;
    a.rt0[0] = 0;
    const int tr = a.T <= kSkinnyT ? 16 : 32;   // rows per tile
    for (int i = 0; i < a.nseg; i++) {
        if (!a.seg[i].w || !a.seg[i].y || a.seg[i].N < 1 || ((uintptr_t)a.seg[i].w & 15)) return -1;
        a.rt0[i + 1] = a.rt0[i] + (a.seg[i].N + tr - 1) / tr;
    }
    for (int i = a.nseg + 1; i <= kGemmMaxSeg; i++) a.rt0[i] = a.rt0[a.nseg];
    a.nb = a.K / 256;
    const int kind = gemm_wide_kind(a);
    if (kind == 1) {
        for (int t0 = 0; t0 < a.T; t0 += kSkinnyT) {
            WideArgs b = a;
            b.T = std::min(kSkinnyT, a.T - t0);
            b.wq += (int64_t)(t0 / 32) * a.nb * kWideRec;
            if (b.ss) b.ss += t0;
            for (int i = 0; i < a.nseg; i++) b.seg[i].y += (int64_t)t0 * a.seg[i].ys;
            if (gemm_wide_launch(b, part_floats, n_cnt, st)) return -1;
        }
        return 0;
    }
    if (kind == 0) {
        const bool q6 = a.type == XJ_Q6_K;
        const int nt = a.T <= 48 ? 3 : 4;
        const SkPlan p = skinny_plan(q6, a.rt0[a.nseg], a.nb, nt);
        const int groups = (a.rt0[a.nseg] + p.rt - 1) / p.rt;
        a.G = p.ks;
        if (p.ks > 1 && (groups > n_cnt || (int64_t)groups * p.ks * p.rt * nt * 256 > part_floats)) return -1;
        switch (p.rt) {
        case 1: return q6 ? launch_s2<true, 1>(a, groups * p.ks, st) : launch_s2<false, 1>(a, groups * p.ks, st);
        case 2: return q6 ? launch_s2<true, 2>(a, groups * p.ks, st) : launch_s2<false, 2>(a, groups * p.ks, st);
        case 3: return q6 ? launch_s2<true, 3>(a, groups * p.ks, st) : launch_s2<false, 3>(a, groups * p.ks, st);
        case 4: return launch_s2<false, 4>(a, groups * p.ks, st);
        default: return launch_s2<false, 5>(a, groups * p.ks, st);
        }
    }
    a.nrg = (a.rt0[a.nseg] + 7) / 8;
    const int tiles = a.nrg * ((a.T + kToks - 1) / kToks);
    a.P = (int64_t)tiles * a.nb;
    a.G = (int)std::min<int64_t>(a.P, wide_cus());
    if (tiles > n_cnt || (int64_t)2 * a.G * kRows * kToks > part_floats) return -1;
    return a.type == XJ_Q6_K ? launch_w<true>(a, st) : launch_w<false>(a, st);
}

}  // namespace xjk
