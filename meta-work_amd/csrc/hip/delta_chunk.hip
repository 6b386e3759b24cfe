// Chunk-wise gated delta rule (gfx950) - the prefill form of the recurrence
// S_t = a_t S_{t-1} + beta_t (v_t - a_t S_{t-1} k_t) k_t^T, o_t = S_t q_t * qscale
// (per head; state [value j][key i] as src/xiaoju-pipe/core/xj_cpu.c:203-213).
// The reference evaluates it token by token; this is the published chunk form
// (Yang, Kautz, Hatamizadeh, "Gated Delta Networks", ICLR 2025; Yang et al.,
// "Parallelizing Linear Transformers with the Delta Rule over Sequence Length",
// NeurIPS 2024), derived for this state orientation:
//   within a chunk of C tokens with start state M0 and lg_t = sum_{s<=t} log a_s,
//   delta = X (V - diag(e^lg) K M0^T),  X = (I + A)^-1 diag(beta),
//   A[s][r] = beta_s e^(lg_s - lg_r) k_s.k_r  (r < s)
//   O     = diag(e^lg) Q M0^T + P delta,  P[t][r] = e^(lg_t - lg_r) q_t.k_r (r <= t)
//   M_C   = e^lg_C M0 + delta^T diag(e^(lg_C - lg)) K
// Decay ratios are formed as exp of differences of cumulative logs, so 64
// steps of small decays never underflow a product.
//
// Every chunk-level dense product runs on the matrix cores in fp32
// (v_mfma_f32_16x16x4f32: fp32 products, fp32 sums). Phase 1 (all chunks and
// heads in parallel) forms K K^T and P, inverts I + A by blocks of 16 (each
// wavefront one diagonal block by forward substitution, then the blocks below
// it by products on the matrix cores, one diagonal after the other), then
// W = X diag(e^lg) K and U = X V; two work-groups per CU (v and q go straight
// to registers, k to LDS) hide each other's latencies, and its bytes bound it.
// Phase 2 walks the chunks in order, one work-group per (head, 16 value rows)
// since the value rows of the state are independent: delta = U - W M0^T and
// M_C on four wavefronts, O on four others beside them. It is bound by the 112
// MFMAs per SIMD and chunk (1.5 us) and the two exchanges through LDS; every
// operand that does not depend on the state is in registers two chunks ahead.
// 16 heads of 128, 2048 tokens: phase 1 59.5 -> 33 us (against a solve over all
// 64 rows on one wavefront, one work-group per CU), phase 2 302 -> 94 us
// (against loads where they are used; one chunk ahead 128 us, in operand order
// two ahead 106 us, the outputs on wavefronts of their own 94 us).
#include "common.h"
#include "kernels.h"

namespace xjk {

constexpr int kC = 64;
typedef float v4f __attribute__((ext_vector_type(4)));

// D (16x16) += A (16x4) B (4x16) on the matrix cores. Lane l supplies
// A[l%16][l/16] and B[l/16][l%16]; element r of lane l is D[4*(l/16) + r][l%16].
// Tiles below walk an inner dimension in blocks of 16: lane group l/16 takes
// inner indices 16b + 4*(l/16) + s, s = 0..3 (one MFMA per s).
__device__ __forceinline__ v4f mma(v4f c, float a, float b) {
    return __builtin_amdgcn_mfma_f32_16x16x4f32(a, b, c, 0, 0, 0);
}
__device__ __forceinline__ v4f ld4(const float *p) { return *(const v4f *)p; }

// Work-group barrier ordering LDS accesses only (loads in flight stay in flight).
__device__ __forceinline__ void lds_barrier() {
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "workgroup", "local");
    __builtin_amdgcn_s_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "workgroup", "local");
}

// Work area of one chunk and head (floats): every operand of phase 2 in the
// order its lanes load it, so that each load is one contiguous piece. (Read in
// place, the rows of q and k are H S floats apart, for 16 heads of 128 a
// multiple of 4 KB: 128 -> 106 us for phase 2.) w = wavefront, l = lane = 16 lq + lr, r, s = 0..3:
//   W, Q [w][b][l][s]     row 16 w + lr, column 16 b + 4 lq + s
//   P    [w][b][l][s]     likewise, columns of the chunk's tokens
//   K    [w][b][s][l][j]  token 16 b + 4 lq + s, column 16 NJ w + NJ lr + j
//   U    [J][w][l][r]     row 16 w + 4 lq + r, column 16 J + lr
template <int S>
struct WorkLayout {
    static constexpr int W = 0, Q = kC * S, K = 2 * kC * S, U = 3 * kC * S, P = 4 * kC * S, GAM = P + kC * kC, GEND = GAM + kC,
                         GC = GEND + kC;
    static constexpr int SIZE = GC + 4;
};

template <int S>
constexpr size_t prep_lds_bytes() { return (size_t)(kC * (S + 4) + 2 * kC * (kC + 4)) * 4; }

template <int S>
__global__ __launch_bounds__(256, 2) void dc_prep(int H, int T, const float *__restrict__ q, const float *__restrict__ k,
                                                  const float *__restrict__ v, const float *__restrict__ decay,
                                                  const float *__restrict__ beta, float *__restrict__ work) {
    using WL = WorkLayout<S>;
    constexpr int KS = S + 4, XS = kC + 4;   // LDS row strides (floats)
    constexpr int NJ = S / 64;               // 16-column blocks per wavefront
    extern __shared__ __align__(16) float sm[];
    float *Ks = sm;                // [kC][KS] the chunk's k rows (zero past T)
    float *Ab = Ks + kC * KS;      // [kC][XS] A, blocks on and below the diagonal
    float *Xb = Ab + kC * XS;      // [kC][XS] (I + A)^-1, the same blocks
    __shared__ float lg[kC], bb[kC];
    __shared__ __align__(16) float gam[kC], bet[kC], bgam[kC];
    const int n = blockIdx.x, h = blockIdx.y, tid = threadIdx.x;
    const int w = __builtin_amdgcn_readfirstlane(tid >> 6), l = tid & 63, lr = l & 15, lq = l >> 4;
    float *wk = work + ((int64_t)n * H + h) * WL::SIZE;
#pragma unroll
    for (int i = 0; i < kC * S / 1024; i++) {
        const int idx = tid + 256 * i, t = idx / (S / 4), c = 4 * (idx % (S / 4)), tok = n * kC + t;
        v4f kv = ld4(k + ((int64_t)min(tok, T - 1) * H + h) * S + c);
        if (tok >= T) kv = v4f{0.f, 0.f, 0.f, 0.f};
        *(v4f *)(Ks + t * KS + c) = kv;
    }
    // the value columns of this wavefront's blocks, used last: inner index (token) 16 b + 4 lq + s
    float vr[NJ][4][4];
#pragma unroll
    for (int j = 0; j < NJ; j++)
#pragma unroll
        for (int b = 0; b < 4; b++)
#pragma unroll
            for (int s = 0; s < 4; s++) {
                const int tok = n * kC + 16 * b + 4 * lq + s;
                const float x = v[((int64_t)min(tok, T - 1) * H + h) * S + 16 * (w + 4 * j) + lr];
                vr[j][b][s] = tok < T ? x : 0.f;
            }
    __syncthreads();
    // k for phase 2
#pragma unroll
    for (int b = 0; b < 4; b++)
#pragma unroll
        for (int s = 0; s < 4; s++)
#pragma unroll
            for (int j = 0; j < NJ; j++)
                wk[WL::K + (((w * 4 + b) * 4 + s) * 64 + l) * NJ + j] = Ks[(16 * b + 4 * lq + s) * KS + 16 * NJ * w + NJ * lr + j];
    if (tid < kC) {
        const int tok = n * kC + tid;
        lg[tid] = tok < T ? logf(decay[(int64_t)tok * H + h]) : 0.f;
        bb[tid] = tok < T ? beta[(int64_t)tok * H + h] : 0.f;
    }
    __syncthreads();
    if (w == 0) {   // running sums of the 64 logs, in double
        double a = lg[l];
#pragma unroll
        for (int off = 1; off < 64; off <<= 1) {
            const double o = __shfl_up(a, off, 64);
            if (l >= off) a += o;
        }
        const float c = (float)a;
        lg[l] = c;
        const float g = expf(c), be = bb[l];
        gam[l] = g;
        bet[l] = be;
        bgam[l] = be * g;
    }
    __syncthreads();
    // the 10 tiles on and below the diagonal of K K^T (A[s][r] = beta_s e^(lg_s - lg_r) k_s.k_r, r < s) and of
    // Q K^T (P[t][r] = e^(lg_t - lg_r) q_t.k_r, r <= t), five per wavefront
#pragma unroll
    for (int x = 0; x < 5; x++) {
        const int tile = w + 4 * x, u = tile < 10 ? tile : tile - 10;
        const int I = u < 1 ? 0 : u < 3 ? 1 : u < 6 ? 2 : 3, J = u - I * (I + 1) / 2;
        const bool isP = tile >= 10;   // uniform over the wavefront
        v4f c0 = {0.f, 0.f, 0.f, 0.f}, c1 = c0;
        const float *qa = q + ((int64_t)min(n * kC + 16 * I + lr, T - 1) * H + h) * S + 4 * lq;
        const float *ka = Ks + (16 * I + lr) * KS + 4 * lq, *kb = Ks + (16 * J + lr) * KS + 4 * lq;
        v4f av[S / 16];
#pragma unroll
        for (int b = 0; b < S / 16; b++) av[b] = isP ? ld4(qa + 16 * b) : ld4(ka + 16 * b);
        if (isP && J == 0)
#pragma unroll
            for (int b = 0; b < S / 16; b++) *(v4f *)(wk + WL::Q + ((I * (S / 16) + b) * 64 + l) * 4) = av[b];
#pragma unroll
        for (int b = 0; b < S / 16; b++) {
            const v4f bv = ld4(kb + 16 * b);
#pragma unroll
            for (int s = 0; s < 4; s += 2) {
                c0 = mma(c0, av[b][s], bv[s]);
                c1 = mma(c1, av[b][s + 1], bv[s + 1]);
            }
        }
#pragma unroll
        for (int r = 0; r < 4; r++) {
            const int s_ = 16 * I + 4 * lq + r, r_ = 16 * J + lr;
            const float e = expf(lg[s_] - lg[r_]) * (c0[r] + c1[r]);
            if (isP) wk[WL::P + ((I * 4 + J) * 64 + 16 * (lr >> 2) + 4 * lq + r) * 4 + (lr & 3)] = r_ <= s_ && n * kC + s_ < T ? e : 0.f;
            else Ab[s_ * XS + r_] = r_ < s_ ? bb[s_] * e : 0.f;
        }
    }
    __syncthreads();
    // diagonal block w of (I + A)^-1: lane column lr (the four lane groups alike), by forward substitution
    {
        const float *Ad = Ab + 16 * w * XS + 16 * w;
        v4f ar[16][4];
#pragma unroll
        for (int s = 1; s < 16; s++)
#pragma unroll
            for (int j = 0; 4 * j < s; j++) ar[s][j] = ld4(Ad + s * XS + 4 * j);
        float xc[16];
#pragma unroll
        for (int s = 0; s < 16; s++) {
            float p[4] = {s == lr ? 1.f : 0.f, 0.f, 0.f, 0.f};
#pragma unroll
            for (int m = 0; m < s; m++) p[m & 3] = fmaf(-ar[s][m / 4][m & 3], xc[m], p[m & 3]);
            xc[s] = (p[0] + p[1]) + (p[2] + p[3]);
        }
        if (lq == 0)
#pragma unroll
            for (int s = 0; s < 16; s++) Xb[(16 * w + s) * XS + 16 * w + lr] = xc[s];
    }
    __syncthreads();
    // the blocks below, by diagonals: X_ij = -X_ii sum over j <= m < i of A_im X_mj (wavefront i); the inner
    // sum's result registers are the next product's operand
#pragma unroll
    for (int d = 1; d < 4; d++) {
        if (w >= d) {
            const int j = w - d;
            v4f g = {0.f, 0.f, 0.f, 0.f}, x = g;
            for (int m = j; m < w; m++) {
                const v4f a4 = ld4(Ab + (16 * w + lr) * XS + 16 * m + 4 * lq);
#pragma unroll
                for (int s = 0; s < 4; s++) g = mma(g, a4[s], Xb[(16 * m + 4 * lq + s) * XS + 16 * j + lr]);
            }
            const v4f t4 = ld4(Xb + (16 * w + lr) * XS + 16 * w + 4 * lq);
#pragma unroll
            for (int s = 0; s < 4; s++) x = mma(x, t4[s], g[s]);
#pragma unroll
            for (int r = 0; r < 4; r++) Xb[(16 * w + 4 * lq + r) * XS + 16 * j + lr] = -x[r];
        }
        __syncthreads();
    }
    // W = X diag(beta e^lg) K and U = X diag(beta) V: wavefront w takes key/value column blocks w, w + 4;
    // X is lower triangular, so row block I needs inner blocks <= I
#pragma unroll
    for (int j = 0; j < NJ; j++) {
        const int J = w + 4 * j;
        v4f aw[4], au[4];
#pragma unroll
        for (int I = 0; I < 4; I++) aw[I] = au[I] = v4f{0.f, 0.f, 0.f, 0.f};
#pragma unroll
        for (int b = 0; b < 4; b++) {
            const int c = 16 * b + 4 * lq;
            const v4f gw = ld4(bgam + c), gb = ld4(bet + c);
            float kw[4], vw[4];
#pragma unroll
            for (int s = 0; s < 4; s++) {
                kw[s] = gw[s] * Ks[(c + s) * KS + 16 * J + lr];
                vw[s] = gb[s] * vr[j][b][s];
            }
#pragma unroll
            for (int I = b; I < 4; I++) {
                const v4f xa = ld4(Xb + (16 * I + lr) * XS + c);
#pragma unroll
                for (int s = 0; s < 4; s++) {
                    aw[I] = mma(aw[I], xa[s], kw[s]);
                    au[I] = mma(au[I], xa[s], vw[s]);
                }
            }
        }
#pragma unroll
        for (int I = 0; I < 4; I++)
#pragma unroll
            for (int r = 0; r < 4; r++)
                wk[WL::W + ((I * (S / 16) + J) * 64 + 16 * (lr >> 2) + 4 * lq + r) * 4 + (lr & 3)] = aw[I][r];
#pragma unroll
        for (int I = 0; I < 4; I++) *(v4f *)(wk + WL::U + ((J * 4 + I) * 64 + l) * 4) = au[I];
    }
    if (tid < kC) {
        wk[WL::GAM + tid] = gam[tid];
        wk[WL::GEND + tid] = expf(lg[kC - 1] - lg[tid]);
    }
    if (tid == 0) wk[WL::GC] = gam[kC - 1];
}

template <int S>
__global__ __launch_bounds__(512, 2) void dc_scan(int H, int T, const float *__restrict__ work, float qscale,
                                                  float *__restrict__ state, float *__restrict__ out) {
    using WL = WorkLayout<S>;
    constexpr int JB = 16, KS = S + 4, DS = JB + 4, NB = S / 16, NJ = S / 64;
    __shared__ __align__(16) float Mb[JB * KS];     // state rows j0..j0+15 (value) x key
    __shared__ float dl[kC * DS], dg[kC * DS];      // delta[s][j], and times e^(lg_C - lg_s)
    const int h = blockIdx.x, j0 = blockIdx.y * JB, tid = threadIdx.x;
    // wavefronts 0..3: delta and the state; 4..7, one on each SIMD beside them: the outputs
    const int wv = __builtin_amdgcn_readfirstlane(tid >> 6), w = wv & 3, l = tid & 63, lr = l & 15, lq = l >> 4;
    const int nch = (T + kC - 1) / kC;
    auto wk_of = [&](int n) { return work + ((int64_t)min(n, nch - 1) * H + h) * WL::SIZE; };
    if (wv < 4) {
        // this wavefront's state tiles: rows 4 lq + r, key columns col + j (NJ consecutive ones per lane)
        const int col = 16 * NJ * w + NJ * lr;
        float *st = state + ((int64_t)h * S + j0 + 4 * lq) * S + col;
        v4f m[NJ];
#pragma unroll
        for (int r = 0; r < 4; r++)
#pragma unroll
            for (int j = 0; j < NJ; j++) Mb[(4 * lq + r) * KS + col + j] = m[j][r] = st[r * S + j];
        // operands of two chunks in turn, each set requested again as soon as it is used (always, the last
        // chunk's at the end: behind a branch, every wait would wait for all)
        struct Set {
            v4f wa[NB], u4, ge;
            float kr[4][4][NJ], gC;
        };
        auto load_a = [&](int n, Set &x) {
            const float *wk = wk_of(n);
#pragma unroll
            for (int b = 0; b < NB; b++) x.wa[b] = ld4(wk + WL::W + ((w * NB + b) * 64 + l) * 4);
            x.u4 = ld4(wk + WL::U + ((blockIdx.y * 4 + w) * 64 + l) * 4);
            x.ge = ld4(wk + WL::GEND + 16 * w + 4 * lq);
        };
        auto load_b = [&](int n, Set &x) {
            const float *wk = wk_of(n);
#pragma unroll
            for (int b = 0; b < 4; b++)
#pragma unroll
                for (int s = 0; s < 4; s++) {
                    const float *kp = wk + WL::K + (((w * 4 + b) * 4 + s) * 64 + l) * NJ;
                    if constexpr (NJ == 2) {
                        const float2 v = *(const float2 *)kp;
                        x.kr[b][s][0] = v.x;
                        x.kr[b][s][NJ - 1] = v.y;
                    } else {
                        x.kr[b][s][0] = *kp;
                    }
                }
            x.gC = wk[WL::GC];
        };
        auto step = [&](int n, Set &x) {
            // delta = U - W M0^T over the wavefront's 16 tokens
            v4f a0 = {0.f, 0.f, 0.f, 0.f}, a1 = a0;
#pragma unroll
            for (int b = 0; b < NB; b++) {
                const v4f mb = ld4(Mb + lr * KS + 16 * b + 4 * lq);
#pragma unroll
                for (int s = 0; s < 4; s += 2) {
                    a0 = mma(a0, x.wa[b][s], mb[s]);
                    a1 = mma(a1, x.wa[b][s + 1], mb[s + 1]);
                }
            }
#pragma unroll
            for (int r = 0; r < 4; r++) {
                const float d = x.u4[r] - (a0[r] + a1[r]);
                dl[(16 * w + 4 * lq + r) * DS + lr] = d;
                dg[(16 * w + 4 * lq + r) * DS + lr] = d * x.ge[r];
            }
            __builtin_amdgcn_sched_barrier(0);
            load_a(n + 2, x);
            lds_barrier();   // delta complete; every wavefront has read M0
            // M_C = e^lg_C M0 + (delta o e^(lg_C - lg))^T K (tokens past T: U = W = 0, so delta is zero)
            v4f m2[NJ];
#pragma unroll
            for (int j = 0; j < NJ; j++) {
                m[j] *= x.gC;
                m2[j] = v4f{0.f, 0.f, 0.f, 0.f};
            }
#pragma unroll
            for (int b = 0; b < 4; b++)
#pragma unroll
                for (int s = 0; s < 4; s++) {
                    const float dv = dg[(16 * b + 4 * lq + s) * DS + lr];
#pragma unroll
                    for (int j = 0; j < NJ; j++) m2[j] = mma(m2[j], dv, x.kr[b][s][j]);
                }
#pragma unroll
            for (int j = 0; j < NJ; j++) m[j] += m2[j];
#pragma unroll
            for (int r = 0; r < 4; r++)
#pragma unroll
                for (int j = 0; j < NJ; j++) Mb[(4 * lq + r) * KS + col + j] = m[j][r];
            __builtin_amdgcn_sched_barrier(0);
            load_b(n + 2, x);
            lds_barrier();   // M_C complete; delta free for the next chunk
        };
        Set x0, x1;
        load_a(0, x0);
        load_b(0, x0);
        load_a(1, x1);
        load_b(1, x1);
        lds_barrier();
        for (int n = 0; n < nch; n += 2) {
            step(n, x0);
            if (n + 1 < nch) step(n + 1, x1);
        }
#pragma unroll
        for (int j = 0; j < NJ; j++)
#pragma unroll
            for (int r = 0; r < 4; r++) st[r * S + j] = m[j][r];
    } else {
        struct Set {
            v4f qa[NB], pa[4], ga;
        };
        auto load_q = [&](int n, Set &x) {
            const float *wk = wk_of(n);
#pragma unroll
            for (int b = 0; b < NB; b++) x.qa[b] = ld4(wk + WL::Q + ((w * NB + b) * 64 + l) * 4);
        };
        auto load_p = [&](int n, Set &x) {
            const float *wk = wk_of(n);
#pragma unroll
            for (int b = 0; b < 4; b++)   // P is zero above the diagonal
                x.pa[b] = ld4(wk + WL::P + ((w * 4 + (b <= w ? b : 0)) * 64 + l) * 4);
            x.ga = ld4(wk + WL::GAM + 16 * w + 4 * lq);
        };
        auto step = [&](int n, Set &x) {
            // O = diag(e^lg) Q M0^T + P delta over the wavefront's 16 tokens
            v4f a0 = {0.f, 0.f, 0.f, 0.f}, a1 = a0, ap = a0;
#pragma unroll
            for (int b = 0; b < NB; b++) {
                const v4f mb = ld4(Mb + lr * KS + 16 * b + 4 * lq);
#pragma unroll
                for (int s = 0; s < 4; s += 2) {
                    a0 = mma(a0, x.qa[b][s], mb[s]);
                    a1 = mma(a1, x.qa[b][s + 1], mb[s + 1]);
                }
            }
            __builtin_amdgcn_sched_barrier(0);
            load_q(n + 2, x);
            lds_barrier();
#pragma unroll
            for (int b = 0; b < 4; b++) {
                if (b > w) break;   // uniform
#pragma unroll
                for (int s = 0; s < 4; s++) ap = mma(ap, x.pa[b][s], dl[(16 * b + 4 * lq + s) * DS + lr]);
            }
#pragma unroll
            for (int r = 0; r < 4; r++) {
                const int tok = n * kC + 16 * w + 4 * lq + r;
                if (tok < T) out[((int64_t)tok * H + h) * S + j0 + lr] = (x.ga[r] * (a0[r] + a1[r]) + ap[r]) * qscale;
            }
            __builtin_amdgcn_sched_barrier(0);
            load_p(n + 2, x);
            lds_barrier();
        };
        Set x0, x1;
        load_q(0, x0);
        load_p(0, x0);
        load_q(1, x1);
        load_p(1, x1);
        lds_barrier();
        for (int n = 0; n < nch; n += 2) {
            step(n, x0);
            if (n + 1 < nch) step(n + 1, x1);
        }
    }
}

size_t delta_chunked_work_bytes(int H, int S, int T, int chunk) {
    if (chunk != kC || T < 1 || H < 1) return 0;
    const int64_t nch = (T + kC - 1) / kC;
    if (S == 128) return (size_t)nch * H * WorkLayout<128>::SIZE * 4;
    if (S == 64) return (size_t)nch * H * WorkLayout<64>::SIZE * 4;
    return 0;
}

template <int S>
static int dc_launch(int H, int T, const float *q, const float *k, const float *v, const float *decay,
                     const float *beta, float qscale, float *state, float *out, float *work, hipStream_t st) {
    static const bool raised = hipFuncSetAttribute((const void *)dc_prep<S>, hipFuncAttributeMaxDynamicSharedMemorySize,
                                                   (int)prep_lds_bytes<S>()) == hipSuccess;
    if (!raised) return -1;
    const int nch = (T + kC - 1) / kC;
    hipLaunchKernelGGL(dc_prep<S>, dim3(nch, H), dim3(256), prep_lds_bytes<S>(), st, H, T, q, k, v, decay, beta, work);
    hipLaunchKernelGGL(dc_scan<S>, dim3(H, S / 16), dim3(512), 0, st, H, T, work, qscale, state, out);
    return hipGetLastError() == hipSuccess ? 0 : -1;
}

int delta_chunked_launch(int H, int S, int T, int chunk, const float *q, const float *k, const float *v,
                         const float *decay, const float *beta, float qscale, float *state, float *out, float *work,
                         hipStream_t st) {
    if (chunk != kC || T < 1 || H < 1) return -1;
    // the row loads are 16-byte vectors
    for (const void *p : {(const void *)q, (const void *)k, (const void *)v, (const void *)state, (const void *)work})
        if ((uintptr_t)p & 15) return -1;
    if (S == 128) return dc_launch<128>(H, T, q, k, v, decay, beta, qscale, state, out, work, st);
    if (S == 64) return dc_launch<64>(H, T, q, k, v, decay, beta, qscale, state, out, work, st);
    return -1;
}

}  // namespace xjk
