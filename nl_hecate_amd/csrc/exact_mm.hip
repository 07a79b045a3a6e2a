// Backward of the exact Titans / Delta rule from checkpoints every C <= 64 tokens, in chunk-parallel matrix form on
// the fp32 matrix cores (v_mfma_f32_16x16x4_f32), head sizes 64 and 32.
//
// Semantics are those of core/kernels/titans_backward.cu:66-341 run segment by segment from the checkpoints of
// core/kernels/titans_forward.cu (the schedule of core/src/gpu_backward.rs:1770-1962) with error_clip and the
// M-norm projection off: every error is taken against the CURRENT memory, u_t = M_(t-1) k_t - v_t.
//
// The rule is linear in (M, S).  Inside a chunk that starts at the checkpoint (M0, S0), with the coefficients of
// the frozen-M0 form (mm_coef.h: a, beta, h, c, bb; W[t][j] = -theta_j c[t][j], wM = W[L-1], wS_j = -theta_j
// bb[j][L-1]) and am, bm = a, beta shifted by one token (am_0 = 1, bm_0 = 0), the errors of a chunk obey a unit
// lower triangular system
//   (I - Lam) U = R,   Lam[t][j] = W[t-1][j] (k_j . k_t)  (j < t),   R = am.(K M0^T) + bm.(K S0^T) - V
// and everything else is the frozen rule with its errors replaced by U plus the terms through T = (I - Lam)^-1:
//   dU = (W.P)^T dY + wM.(K dMo^T) + wS.(K dSo^T)     dR = T^T dU      (P = Q K^T; dMo, dSo: adjoints at chunk end)
//   dV = -dR     dQ = a.(dY M0) + beta.(dY S0) + (W.tril(dY U^T)) K
//   dK = (W.tril(dY U^T))^T Q + wM.(U dMo) + wS.(U dSo) + am.(dR M0) + bm.(dR S0) + (dG + dG^T) K,
//        dG[t][j] = W[t-1][j] strict_tril(dR U^T)[t][j]
//   adjoints at chunk start:  dM' = a_L dMo + (a.dY)^T Q + (am.dR)^T K,   dS' = beta_L dMo + h_L dSo + (beta.dY)^T Q + (bm.dR)^T K
// The last line is affine in (dMo, dSo) with matrices that depend on the chunk only, so the reverse scan over the
// chunks of a chain multiplies by four 64x64 matrices per step and the rest is chunk-parallel:
//   1. ex_local_kernel   per chunk: T (blocked inverse: 16x16 diagonal blocks by substitution, then
//                        (I + N)(I + N^2) D with N = D Lam_off, N^4 = 0), U, dU_loc = (W.P)^T dY, the four matrices
//                        Phi = (w.K)^T T (m.K) and the two additive terms of the scan
//   2. ex_scan_kernel    per (chain, 16-row block): the adjoints at every chunk boundary
//   3. ex_grads_kernel   per chunk: dQ, dK, dV, dtheta and the hand-off of the gate pass
//   4. cw_gates_sweep_kernel (chunkwise_gates.hip): dalpha, deta.  The inner products <M_s, J_t> it sweeps obey the
//      rule's own recurrence with J_t = dy_t q_t^T + dR_(t+1) k_(t+1)^T, i.e. per-token terms
//      xs[s][t] = -theta_s [ (dy_t.u_s)(q_t.k_s) + (dR_(t+1).u_s)(k_(t+1).k_s) ].
// The algebra is written out and checked against the reference's token loops in float64 in tests/np_rules.py
// (titans_exact_chunk_backward).
//
// FROZEN: the frozen-M0 chunkwise rule (core/kernels/titans_chunkwise_backward.cu) in the same kernels: its errors are
// taken against the chunk-start memory, i.e. T = I, am = 1, bm = 0, and the terms through Lam are absent.  Serves head
// size 32, which the chunkwise matrix kernels of chunkwise_mm.hip do not have.
//
// P64: which sums are float64 (mm_tiles.h).  The walks that this form stands in for add a row's product up in a tree and
// are 0.6 to 1.2e-7 off the exact gradients (gates spread over (0, 1); 2 to 4e-7 where the states live for 150 tokens); with
// fp32 sums throughout the form is at 1.5 to 2.6e-7.  So wherever a walk was replaced (wide_sums, and the forward's chunk
// maps), the coefficients' recurrences, the gate sweeps and every product whose rounding reaches a result are float64 sums
// rounded once: 0.6 to 1.0e-7, each output at or below its walk over spread gates, gates at a model's start and long-lived
// states.  Left in fp32 are the products that do not show: the inverse, K K^T, K M^T, the maps
// of the adjoint scan and the products with the adjoint at the chunk's end.  512 tokens of 32 chains, head size 64: first
// kernel 38 -> 46 us, gradients 38 -> 49, scan 16 -> 23, gates 10 -> 15; head size 32, 777 tokens of 16: 21 -> 25, 24 -> 32,
// 5 -> 8, 7 -> 9.  Head size 64 with checkpoints every 32 tokens and more keeps fp32 sums: there the form is the path that
// there was, and its two kernels are bound by their products.
//
// Under a finite m_norm_max / error clip the pass also leaves the ChainTracks of chunkwise_chain.h behind (|u_t|^2 per
// token, sums of squares of the checkpoints); the caller tests on them whether a coupling could have fired.
#include <hip/hip_runtime.h>
#include <stdint.h>

#include <type_traits>

#include "chunkwise_chain.h"
#include "chunkwise_grads.h"
#include "chunkwise_guard.h"
#include "exact_mm.h"
#include "mm_coef.h"
#include "mm_tiles.h"
#include "rule_common.h"
#include "runtime.h"

namespace nlh {
namespace {

using namespace mmt;

// Waves w and w + 4 share a SIMD.  Products with the lower triangular T (or its transpose) cost a 16-row block
// ib + 1 (or 4 - ib) quarter products, so the row blocks are dealt out as (0, 3) and (1, 2) per SIMD.
#define NLH_STRIP_ORIGIN_OF(w) \
    const int ib = w < 4 ? w >> 1 : 3 - ((w - 4) >> 1), m0 = 16 * ib, n0 = 32 * (w & 1), nh = w & 1; \
    (void)nh
#define NLH_STRIP_ORIGIN() \
    const int w = threadIdx.x >> 6; \
    NLH_STRIP_ORIGIN_OF(w)

// Sums of the products: fp32 or float64 (mm_tiles.h).
template <bool P64> using real = std::conditional_t<P64, double, float>;
template <bool P64, class FA, class FB>
__device__ __forceinline__ void product(Strip &acc, FA a, FB b, int l) {
    if constexpr (P64) mma_f64(acc, a, b, l); else mma(acc, a, b, l);
}
template <bool P64, class FA, class FB>
__device__ __forceinline__ void product_range(Strip &acc, FA a, FB b, int p0, int p1, int l) {
    if constexpr (P64) mma_range_f64(acc, a, b, p0, p1, l); else mma_range(acc, a, b, p0, p1, l);
}

// per chunk, for the scan: Phi_MM, Phi_SM, Phi_MS, Phi_SS (source state, destination state), C_M, C_S
constexpr size_t kExLocMats = 6;
constexpr size_t kDD = (size_t)HD * HD;   // a token x token or token x head-size matrix of a chunk in memory

// Staging of a row-major [nrows <= ROWS][D] tile as fetch / commit of mm_tiles.h, for either head size.
template <int D, int ROWS>
struct TileD {
    static constexpr int N = ROWS * D / 4, PER = (N + kThr - 1) / kThr;
    float4 x[PER];
};
template <int D, int ROWS>
__device__ __forceinline__ void fetch(TileD<D, ROWS> &r, const float *src, int nrows, int tid) {
    using T = TileD<D, ROWS>;
#pragma unroll
    for (int it = 0; it < T::PER; it++) {
        const int e = it * kThr + tid, rr = e / (D / 4), cc = 4 * (e % (D / 4));
        r.x[it] = rr < nrows ? *reinterpret_cast<const float4 *>(src + rr * D + cc) : make_float4(0, 0, 0, 0);
    }
}
template <int D, int ROWS>
__device__ __forceinline__ void commit(float *dst, const TileD<D, ROWS> &r, int tid) {
    using T = TileD<D, ROWS>;
#pragma unroll
    for (int it = 0; it < T::PER; it++) {
        const int e = it * kThr + tid, rr = e / (D / 4), cc = 4 * (e % (D / 4));
        if (T::N % kThr == 0 || e < T::N) {
            float *p = dst + rr * LDM + cc;
            p[0] = r.x[it].x; p[1] = r.x[it].y; p[2] = r.x[it].z; p[3] = r.x[it].w;
        }
    }
}
template <int D, int ROWS>
__device__ __forceinline__ float tile_dot(const TileD<D, ROWS> &a, const TileD<D, ROWS> &b) {
    float x = 0.f;
#pragma unroll
    for (int it = 0; it < TileD<D, ROWS>::PER; it++)
        x += a.x[it].x * b.x[it].x + a.x[it].y * b.x[it].y + a.x[it].z * b.x[it].z + a.x[it].w * b.x[it].w;
    return x;
}

// The scan matrices leave in the order in which the scan's waves take them as the second operand of their product:
// lane 16 g + n % 16 of the wave for the 16 columns n / 16 takes the contraction indices (D / 4) g + 0 .. D / 4 - 1 of
// its column as 16-byte pieces of four, and pieces are stored [column tile][piece][lane], so that a load instruction
// of the scan reads 1 KB of consecutive memory.  A lane of a 16 x 16 accumulator tile (rows 16 ib + 4 (l / 16) + i,
// columns 16 ct + l % 16) holds exactly one piece.
template <int D>
__device__ __forceinline__ void store_operand_tile(float *mat, const f32x4 &t, int ib, int ct, int l) {
    const int k0 = 16 * ib + 4 * (l >> 4), g = k0 / (D / 4), piece = (k0 % (D / 4)) / 4;
    *reinterpret_cast<f32x4 *>(mat + ((size_t)(ct * (D / 16) + piece) * 64 + 16 * g + (l & 15)) * 4) = t;
}
// The additive terms leave in the accumulator order of the wave that adds them: [row block][column tile][lane].
template <int D>
__device__ __forceinline__ void store_acc_tile(float *mat, const f32x4 &t, int ib, int ct, int l) {
    *reinterpret_cast<f32x4 *>(mat + ((size_t)(ib * (D / 16) + ct) * 64 + l) * 4) = t;
}

struct ChunkVecs { float wM[CW], wS[CW], am[CW], bm[CW]; };
template <bool FROZEN>
__device__ __forceinline__ void chunk_vectors(ChunkVecs &cv, const Coef &cf, int L) {
    const int j = threadIdx.x;
    if (j < CW) {
        cv.wM[j] = -cf.th[j] * cf.cl[j];
        cv.wS[j] = -cf.th[j] * cf.bl[j];
        cv.am[j] = FROZEN ? 1.f : j == 0 ? 1.f : (j < L ? cf.a[j - 1] : 0.f);
        cv.bm[j] = (FROZEN || j == 0 || j >= L) ? 0.f : cf.beta[j - 1];
    }
}

// ── pass 1: chunk-local matrices ────────────────────────────────────────────
template <int D, bool FROZEN, bool TRACK, bool P64>
__global__ __launch_bounds__(kThr) void ex_local_kernel(
    const float *__restrict__ k, const float *__restrict__ v, const float *__restrict__ q, const float *__restrict__ d_y,
    const float *__restrict__ alpha, const float *__restrict__ theta, const float *__restrict__ eta,
    const float *__restrict__ m_ckpt, const float *__restrict__ s_ckpt, float *__restrict__ loc,
    float *__restrict__ Tg, float *__restrict__ Ug, float *__restrict__ dUg, int s, int C, int nc, int nck, int cstep, int has_s,
    int ntask, ChainTracks tr) {
    constexpr size_t DD = (size_t)D * D;
    extern __shared__ float smem[];
    float *Ks = smem, *Vs = Ks + MAT, *Qs = Vs + MAT, *Ds = Qs + MAT, *Ms = Ds + MAT, *Ss = Ms + MAT, *Cc = Ss + MAT,
          *B8 = Cc + MAT, *B9 = B8 + MAT;
    __shared__ Coef cf;
    __shared__ ChunkVecs cv;
    // Persistent over a contiguous range of chunks.  A workgroup fills the compute unit's LDS, so nothing else would
    // hide its loads: the next chunk's tiles are requested at the start of this chunk's last phase (the longest one,
    // ten products back to back) and land in LDS at the top of the next round.
    TileD<D, 64> tk, tv, tq, td;
    TileD<D, D> tm, ts;
    Gates gt;
    auto fetch_task = [&](int task, int tid) {
        const int chain = task / nc, ci = task % nc, t0 = ci * C, L = min(C, s - t0);
        const size_t tok = (size_t)chain * s + t0, st = ((size_t)chain * nck + (size_t)ci * cstep) * DD;
        gt = fetch_gates(alpha + tok, theta + tok, eta + tok, L, has_s != 0);
        fetch(tk, k + tok * D, L, tid);
        fetch(tv, v + tok * D, L, tid);
        fetch(tq, q + tok * D, L, tid);
        fetch(td, d_y + tok * D, L, tid);
        fetch(tm, m_ckpt + st, D, tid);
        if (has_s) fetch(ts, s_ckpt + st, D, tid);
    };
    const int per = (ntask + (int)gridDim.x - 1) / (int)gridDim.x, task_lo = blockIdx.x * per, task_hi = min(ntask, task_lo + per);
    if (task_lo < task_hi) fetch_task(task_lo, threadIdx.x);
    for (int itask = task_lo; itask < task_hi; itask++) {
    // thread and wave index through opaque copies, once per chunk (see mm_tiles.h)
    int tid = threadIdx.x;
    asm volatile("" : "+v"(tid));
    const int l = tid & 63;
    int w = __builtin_amdgcn_readfirstlane(tid >> 6);
    asm volatile("" : "+s"(w));
    NLH_STRIP_ORIGIN_OF(w);
    auto MMA = [&](Strip &acc, auto fa, auto fb) { product<P64>(acc, fa, fb, l); };
    auto MMAR = [&](Strip &acc, auto fa, auto fb, int p0, int p1) { product_range<P64>(acc, fa, fb, p0, p1, l); };
    auto MMAT = [&](f32x4 &acc, auto fa, auto fb, int k0) { mma_tile16(acc, fa, fb, k0, l); };
    // over the head size
    auto MMD = [&](Strip &acc, auto fa, auto fb) { if constexpr (D == 64) MMA(acc, fa, fb); else MMAR(acc, fa, fb, 0, D / 32); };
    auto MMD32 = [&](Strip &acc, auto fa, auto fb) { if constexpr (D == 64) mma(acc, fa, fb, l); else mma_range(acc, fa, fb, 0, D / 32, l); };
    const bool dcol = D == 64 || nh == 0;   // this wave's strip lies inside a token x head-size product
    auto FORC = [&](Strip &acc, auto f) { for_c(acc, f, l); };
    const int chain = itask / nc, ci = itask % nc, t0 = ci * C, L = min(C, s - t0);
    const size_t task = (size_t)itask;
    (void)t0;
    {
        load_gates(cf, gt);
        coefficients<real<P64>>(cf, gt, L, Cc);
        commit(Ks, tk, tid);
        commit(Vs, tv, tid);
        commit(Qs, tq, tid);
        commit(Ds, td, tid);
        commit(Ms, tm, tid);
        if (has_s) commit(Ss, ts, tid);
        if (TRACK) {
            float msq = wave_allreduce(tile_dot(tm, tm)), ssq = has_s ? wave_allreduce(tile_dot(ts, ts)) : 0.f;
            if (l == 0) *reinterpret_cast<float2 *>(tr.nrm + (task * 8 + w) * 2) = make_float2(msq, ssq);
        }
    }
    __syncthreads();
    chunk_vectors<FROZEN>(cv, cf, L);
    {
        Strip g = zero_strip(), km = zero_strip(), ks = zero_strip(), p = zero_strip();
        auto aK = [&](int m, int kk) { return Ks[(m0 + m) * LDM + kk]; };
        if (!FROZEN) MMD32(g, aK, [&](int kk, int n) { return Ks[(n0 + n) * LDM + kk]; });
        if (dcol) MMD32(km, aK, [&](int kk, int n) { return Ms[(n0 + n) * LDM + kk]; });
        if (!FROZEN && dcol && has_s) MMD32(ks, aK, [&](int kk, int n) { return Ss[(n0 + n) * LDM + kk]; });
        MMD(p, [&](int m, int kk) { return Qs[(m0 + m) * LDM + kk]; }, [&](int kk, int n) { return Ks[(n0 + n) * LDM + kk]; });
        __syncthreads();   // the vectors are there
#pragma unroll
        for (int tl = 0; tl < 2; tl++)
#pragma unroll
            for (int i = 0; i < 4; i++) {
                const int row = m0 + row_of(i, l), col = n0 + 16 * tl + (l & 15);
                if (dcol) {   // R in place over V (own strip)
                    float *d = Vs + row * LDM + col;
                    *d = FROZEN ? km.t[tl][i] - *d : cv.am[row] * km.t[tl][i] + cv.bm[row] * ks.t[tl][i] - *d;
                }
                const float nth = -cf.th[col];
                if (!FROZEN) B8[row * LDM + col] = (col < row) ? nth * Cc[(row - 1) * LDM + col] * g.t[tl][i] : 0.f;   // Lam
                B9[row * LDM + col] = nth * Cc[row * LDM + col] * p.t[tl][i];                            // W.P
            }
    }
    __syncthreads();
    Strip dul = zero_strip();
    if (dcol) MMA(dul, [&](int m, int kk) { return B9[kk * LDM + m0 + m]; }, [&](int kk, int n) { return Ds[kk * LDM + n0 + n]; });
    float *goT = Tg + task * kDD, *goU = dUg + task * kDD;
    auto track = [&](Strip &u) {   // squared error norm of the strip's 16 tokens over its 32 memory rows
        FORC(u, [&](int, int, float &x) { x *= x; });
        strip_row_sums(u);
        if (row_writer(l)) {
            float *eo = tr.e2 + (((size_t)chain * 2 + nh) * nc + ci) * CW + m0;
#pragma unroll
            for (int i = 0; i < 4; i++) eo[row_of(i, l)] = u.t[0][i];
        }
    };
    if constexpr (FROZEN) {   // U = R, Z1 = K
        __syncthreads();      // W.P is read
        if (dcol) {
            Strip u;
            float *go = Ug + task * kDD;
            FORC(dul, [&](int r, int c, float &x) { B9[(m0 + r) * LDM + n0 + c] = x; goU[(m0 + r) * HD + n0 + c] = x; });
            FORC(u, [&](int r, int c, float &x) { x = Vs[(m0 + r) * LDM + n0 + c]; go[(m0 + r) * HD + n0 + c] = x; });
            if (TRACK) track(u);
        }
    } else {
#define INV_L B8
#define INV_D Ms
#define INV_N Ss
#define INV_X Cc
#define INV_BESIDE_N \
    if (dcol)        \
        FORC(dul, [&](int r, int c, float &x) { B9[(m0 + r) * LDM + n0 + c] = x; goU[(m0 + r) * HD + n0 + c] = x; });
#define INV_OUT(row, col, x) goT[(row) * HD + (col)] = x;
#include "exact_inverse.h"
    if (dcol) {   // U = T R -> out;  Z1 = T (am.K) -> B8,  Z2 = T (bm.K) -> Ms
        Strip u = zero_strip(), z1 = zero_strip(), z2 = zero_strip();
        auto aT = [&](int m, int kk) { return Ss[(m0 + m) * LDM + kk]; };
        // T is lower triangular: row block ib contracts over the first ib + 1 blocks of 16 (taken in pairs)
        const int pe = (ib >> 1) + 1;
        MMAR(u, aT, [&](int kk, int n) { return Vs[kk * LDM + n0 + n]; }, 0, pe);
        mma_range(z1, aT, [&](int kk, int n) { return cv.am[kk] * Ks[kk * LDM + n0 + n]; }, 0, pe, l);
        if (has_s) mma_range(z2, aT, [&](int kk, int n) { return cv.bm[kk] * Ks[kk * LDM + n0 + n]; }, 0, pe, l);
        float *go = Ug + task * kDD;
        FORC(u, [&](int r, int c, float &x) { go[(m0 + r) * HD + n0 + c] = x; });
        FORC(z1, [&](int r, int c, float &x) { B8[(m0 + r) * LDM + n0 + c] = x; });
        if (has_s) FORC(z2, [&](int r, int c, float &x) { Ms[(m0 + r) * LDM + n0 + c] = x; });
        if (TRACK) track(u);
    }
    }
    if (TRACK && !dcol && row_writer(l)) {   // head size 32 has no second half
        float *eo = tr.e2 + (((size_t)chain * 2 + nh) * nc + ci) * CW + m0;
#pragma unroll
        for (int i = 0; i < 4; i++) eo[row_of(i, l)] = 0.f;
    }
    __syncthreads();
    if (itask + 1 < task_hi) fetch_task(itask + 1, tid);
    float *out = loc + task * kExLocMats * DD;
    // One product at a time (no unrolling over the outputs): the next chunk's tiles are in registers during this phase.
    // At head size 32 a wave's strip is half a matrix's rows, so the outputs are dealt to the waves in pairs of strips.
    const int sib = D == 64 ? ib : w & 1, sn0 = D == 64 ? n0 : 0, sm0 = 16 * sib;
    const int o0 = D == 64 ? 0 : w >> 1, ostep = D == 64 ? 1 : 4;
    const float aL = cf.a[L - 1], bL = cf.beta[L - 1], hL = cf.h[L - 1];
    const bool on_diag = sm0 == sn0 || sm0 == sn0 + 16;
#pragma unroll 1
    for (int o = o0; o < (has_s ? 4 : 1); o += ostep) {   // Phi_MM, Phi_SM, Phi_MS, Phi_SS = (w.K)^T Z
        const float *wv = (o & 1) ? cv.wS : cv.wM, *Z = FROZEN ? Ks : (o & 2) ? Ms : B8;
        Strip x = zero_strip();
        if (!(FROZEN && (o & 2)))
            mma(x, [&](int m, int kk) { return wv[kk] * Ks[kk * LDM + sm0 + m]; }, [&](int kk, int n) { return Z[kk * LDM + sn0 + n]; }, l);
        if (on_diag) {   // the chunk's own decay
            const float dg = o == 0 ? aL : o == 2 ? bL : o == 3 ? hL : 0.f;
            FORC(x, [&](int r, int c, float &y) { if (sm0 + r == sn0 + c) y += dg; });
        }
#pragma unroll
        for (int tl = 0; tl < 2; tl++) store_operand_tile<D>(out + (size_t)o * DD, x.t[tl], sib, sn0 / 16 + tl, l);
    }
#pragma unroll 1
    for (int o = o0; o < (has_s ? 2 : 1); o += ostep) {   // C_M = (a.dY)^T Q + dU_loc^T Z1,  C_S = (beta.dY)^T Q + dU_loc^T Z2
        const float *vec = o ? cf.beta : cf.a, *Z = FROZEN ? Ks : o ? Ms : B8;
        Strip x = zero_strip();
        MMA(x, [&](int m, int kk) { return (real<P64>)vec[kk] * Ds[kk * LDM + sm0 + m]; }, [&](int kk, int n) { return Qs[kk * LDM + sn0 + n]; });
        if (!(FROZEN && o))
            MMA(x, [&](int m, int kk) { return B9[kk * LDM + sm0 + m]; }, [&](int kk, int n) { return Z[kk * LDM + sn0 + n]; });
#pragma unroll
        for (int tl = 0; tl < 2; tl++) store_acc_tile<D>(out + (size_t)(4 + o) * DD, x.t[tl], sib, sn0 / 16 + tl, l);
    }
    __syncthreads();   // LDS is rewritten by the next chunk
    }
}
constexpr size_t kExLocalLds = 9 * MAT * sizeof(float);

// ── pass 2: scan over the chunks of a chain, one workgroup per 16-row block ──
//   X1' = X1 Phi_MM + X2 Phi_SM + C_M,   X2' = X1 Phi_MS + X2 Phi_SS + C_S   (the chunk's decay is on the diagonals)
// REV: adjoints, last chunk first, from zero; states [chain][nc + 1][D*D]: slot c = adjoint of the state at the start of
// chunk c (slot nc = 0, slot 0 = the gradient of the initial state, also written to first [chain][D*D]).
// Forward: the states themselves from the initial ones; chunk c's start state goes to slot c * sstep of the chain's
// states, for as many chunks as there are steps (sstep 0: only the last one stays).
// One wave per (destination, 16 columns): both sources' contributions, 2 D / 16 products of 16 x 16 x 16, so a step needs
// no exchange of partial sums and, with X in two LDS buffers, one barrier.  The second operand comes straight from memory
// in the lane order of the product (store_operand_tile), the additive term in accumulator order: every load is 1 KB of
// consecutive memory, requested two steps ahead of its use.  All waves run the same number of loads and stores per step:
// the memory counter of this hardware counts both in order, and only a fixed number in flight can be waited past.
// Bound by the step's own chain: LDS read, 2 D / 4 matrix instructions on each of two waves per SIMD, LDS write, barrier.
// 64 chains x 32 chunks, head size 64: 84 -> 78 us (four source / destination waves that swapped tiles through LDS,
// two barriers a step and loads one step ahead before).
template <int D, bool HAS_S, bool REV, bool P64>
__global__ __launch_bounds__((HAS_S ? 2 : 1) * D * 4) void ex_scan_kernel(
    const float *__restrict__ loc, const float *__restrict__ m_initial, const float *__restrict__ s_initial, long long m_stride,
    float *__restrict__ mst, float *__restrict__ sst, long long state_stride, int sstep, float *__restrict__ first_m,
    float *__restrict__ first_s, int nc, int steps) {
    constexpr int NS = HAS_S ? 2 : 1, NT = D / 16, NB = D / 16, LDX = D + 4, DD = D * D;
    __shared__ __align__(16) float X[2][NS][16 * LDX];
    // the row blocks of a chain sit 8 workgroups apart: consecutive workgroups go to consecutive XCDs, so they share one
    // XCD's L2 for the chunk matrices they all read
    const int bx = blockIdx.x, span = 8 * NT;
    const bool whole = (bx / span + 1) * span <= (int)gridDim.x;   // a full group of workgroups
    const int chain = whole ? (bx & 7) + 8 * (bx / span) : bx / NT, rb = whole ? (bx >> 3) % NT : bx % NT;
    const int l = threadIdx.x & 63, w = threadIdx.x >> 6, dst = w / NT, ct = w % NT;
    const int col = 16 * ct + (l & 15), rw = 4 * (l >> 4);   // this wave's tile: rows 16 rb + rw + i
    const size_t at = (size_t)(16 * rb + rw) * D + col;      // its first element in a D x D matrix
    float *st = (dst ? sst : mst) + (size_t)chain * state_stride + at;
    f32x4 x = {0.f, 0.f, 0.f, 0.f};
    if (!REV) {
        const float *in = dst ? s_initial : m_initial;
        if (in) {   // no initial momentum: zero
            in += (size_t)chain * m_stride + at;
#pragma unroll
            for (int i = 0; i < 4; i++) x[i] = in[i * D];
        }
    }
#pragma unroll
    for (int i = 0; i < 4; i++) {
        X[0][dst][(rw + i) * LDX + col] = x[i];
        st[(REV ? (size_t)nc * DD : 0) + i * D] = x[i];
    }
    struct Step { f32x4 b[NS][NB], c; };
    const f32x4 *lc = reinterpret_cast<const f32x4 *>(loc) + (size_t)chain * nc * kExLocMats * (DD / 4) + l;
    auto request = [&](Step &r, int i) {   // step i of the scan (past the end: the last one again, unused)
        const int ci = REV ? max(nc - 1 - i, 0) : min(i, nc - 1);
        const f32x4 *p = lc + (size_t)ci * kExLocMats * (DD / 4);
#pragma unroll
        for (int sr = 0; sr < NS; sr++)
#pragma unroll
            for (int j = 0; j < NB; j++) r.b[sr][j] = p[(HAS_S ? dst * 2 + sr : 0) * (DD / 4) + (ct * NB + j) * 64];
        r.c = p[(4 + dst) * (DD / 4) + (rb * NT + ct) * 64];
    };
    auto step = [&](Step &r, int i) {
        const float *Xr = X[i & 1][0] + (P64 ? f64_row(l) : l & 15) * LDX + (D / 4) * (l >> 4);
        f32x4 a[NS][NB];
#pragma unroll
        for (int sr = 0; sr < NS; sr++)
#pragma unroll
            for (int j = 0; j < NB; j++) a[sr][j] = *reinterpret_cast<const f32x4 *>(Xr + sr * 16 * LDX + 4 * j);
        using Acc = std::conditional_t<P64, f64x4, f32x4>;
        Acc acc[2] = {Acc{r.c[0], r.c[1], r.c[2], r.c[3]}, Acc{0, 0, 0, 0}};
#pragma unroll
        for (int j = 0; j < NB; j++)
#pragma unroll
            for (int sr = 0; sr < NS; sr++)
#pragma unroll
                for (int e = 0; e < 4; e++) {
                    Acc &to = acc[HAS_S ? sr : e & 1];
                    if constexpr (P64) to = __builtin_amdgcn_mfma_f64_16x16x4f64((double)a[sr][j][e], (double)r.b[sr][j][e], to, 0, 0, 0);
                    else to = __builtin_amdgcn_mfma_f32_16x16x4f32(a[sr][j][e], r.b[sr][j][e], to, 0, 0, 0);
                }
        request(r, i + 2);
        float *Xw = X[(i + 1) & 1][dst] + rw * LDX + col;
        const size_t slot = REV ? (size_t)(nc - 1 - i) * DD : (size_t)(i + 1) * sstep * DD;
#pragma unroll
        for (int e = 0; e < 4; e++) {
            x[e] = (float)(acc[0][e] + acc[1][e]);
            Xw[e * LDX] = x[e];
            st[slot + e * D] = x[e];
        }
        __syncthreads();
    };
    Step r0, r1;
    request(r0, 0);
    request(r1, 1);
    __syncthreads();
    int i = 0;
    for (; i + 2 <= steps; i += 2) {
        step(r0, i);
        step(r1, i + 1);
    }
    if (i < steps) step(r0, i);
    if (REV) {
        float *gf = (dst ? first_s : first_m) + (size_t)chain * DD + at;
#pragma unroll
        for (int e = 0; e < 4; e++) gf[e * D] = x[e];
    }
}

// ── pass 3: gradients of one chunk ──────────────────────────────────────────
//   pvec [chain][token][4] = <M0, J_t>, <S0, J_t>, -theta_t u_t^T dMo k_t, -theta_t u_t^T dSo k_t
//   xs [chain][chunk][s][t] as above     scal [chunk][4] = <M0, dMo>, <S0, dMo>, <S0, dSo>
template <int D, bool FROZEN, bool P64>
__global__ __launch_bounds__(kThr) void ex_grads_kernel(
    const float *__restrict__ k, const float *__restrict__ q, const float *__restrict__ d_y, const float *__restrict__ alpha,
    const float *__restrict__ theta, const float *__restrict__ eta, const float *__restrict__ m_ckpt,
    const float *__restrict__ s_ckpt, const float *__restrict__ Tg, const float *__restrict__ Ug,
    const float *__restrict__ dUg, const float *__restrict__ em, const float *__restrict__ es_, float *__restrict__ d_k,
    float *__restrict__ d_v, float *__restrict__ d_q, float *__restrict__ d_theta, float *__restrict__ pvec,
    float *__restrict__ xs, float *__restrict__ scal, int s, int C, int nc, int nck, int cstep, int has_s, int ntask) {
    constexpr size_t DD = (size_t)D * D;
    extern __shared__ float smem[];
    float *Ks = smem, *Qs = Ks + MAT, *Ds = Qs + MAT, *Ts = Ds + MAT, *Us = Ts + MAT, *A1 = Us + MAT, *A2 = A1 + MAT,
          *Cc = A2 + MAT, *B9 = Cc + MAT;
    __shared__ Coef cf;
    __shared__ ChunkVecs cv;
    __shared__ float part[7][2][CW];   // row sums per column half: p0, ps, g1, g2, dam, dbm, u.dR
    __shared__ float part_th[4][CW];   // column sums of dW.c per 16-row block
    __shared__ float dots[3][8];
    // Persistent over a contiguous range of chunks, as ex_local_kernel: the next chunk's nine tiles are requested at the
    // start of this chunk's last phase.
    TileD<D, 64> tk, tq, td;
    TileD<64, 64> tt, tu;
    TileD<D, D> tdm, tds, tm, ts;
    Gates gt;
    // K, Q, dY of the next chunk are requested during this chunk's last phase (more does not fit next to its
    // accumulators); the other six tiles at the top of the chunk, behind two products that need K and Q only
    auto fetch_a = [&](int task, int tid) {
        const int chain = task / nc, ci = task % nc, t0 = ci * C, L = min(C, s - t0);
        const size_t tok = (size_t)chain * s + t0;
        gt = fetch_gates(alpha + tok, theta + tok, eta + tok, L, has_s != 0);
        fetch(tk, k + tok * D, L, tid);
        fetch(tq, q + tok * D, L, tid);
        fetch(td, d_y + tok * D, L, tid);
    };
    auto fetch_b = [&](int task, int tid) {
        const int chain = task / nc, ci = task % nc;
        const size_t end = ((size_t)chain * (nc + 1) + ci + 1) * DD, st = ((size_t)chain * nck + (size_t)ci * cstep) * DD;
        if (!FROZEN) fetch(tt, Tg + (size_t)task * kDD, 64, tid);
        fetch(tu, Ug + (size_t)task * kDD, 64, tid);   // at head size 32 the right half is stale memory, never used
        fetch(tdm, em + end, D, tid);
        if (has_s) fetch(tds, es_ + end, D, tid);
        fetch(tm, m_ckpt + st, D, tid);
        if (has_s) fetch(ts, s_ckpt + st, D, tid);
    };
    const int per = (ntask + (int)gridDim.x - 1) / (int)gridDim.x, task_lo = blockIdx.x * per, task_hi = min(ntask, task_lo + per);
    if (task_lo < task_hi) fetch_a(task_lo, threadIdx.x);
    for (int itask = task_lo; itask < task_hi; itask++) {
    int tid = threadIdx.x;
    asm volatile("" : "+v"(tid));
    const int l = tid & 63;
    int w = __builtin_amdgcn_readfirstlane(tid >> 6);
    asm volatile("" : "+s"(w));
    NLH_STRIP_ORIGIN_OF(w);
    // Float64 sums at head size 64: the scheduler, left alone, reads the operands of several products ahead and spills 119 registers
    // a lane, one with the barrier (256 chunks 64 -> 49 us).  At head size 32, where it spills two, the barrier leaves none and no
    // time either (208 chunks 33.5 / 33.7 us between events); the other forms spill none.
    auto MMA = [&](Strip &acc, auto fa, auto fb) {
        product<P64>(acc, fa, fb, l);
        if (P64 && D == 64) __builtin_amdgcn_sched_barrier(0);
    };
    auto MMAR = [&](Strip &acc, auto fa, auto fb, int p0, int p1) { product_range<P64>(acc, fa, fb, p0, p1, l); };
    auto FORC = [&](Strip &acc, auto f) { for_c(acc, f, l); };
    auto MMD = [&](Strip &acc, auto fa, auto fb) { if constexpr (D == 64) MMA(acc, fa, fb); else MMAR(acc, fa, fb, 0, D / 32); };
    auto MMD32 = [&](Strip &acc, auto fa, auto fb) { if constexpr (D == 64) mma(acc, fa, fb, l); else mma_range(acc, fa, fb, 0, D / 32, l); };
    const bool dcol = D == 64 || nh == 0;   // this wave's strip lies inside a token x head-size product
    const int chain = itask / nc, ci = itask % nc, t0 = ci * C, L = min(C, s - t0);
    const size_t tok = (size_t)chain * s + t0, task = (size_t)itask;
    fetch_b(itask, tid);
    load_gates(cf, gt);
    coefficients<real<P64>>(cf, gt, L, Cc);
    commit(Ks, tk, tid);
    commit(Qs, tq, tid);
    commit(Ds, td, tid);
    __syncthreads();
    chunk_vectors<FROZEN>(cv, cf, L);
    auto aK = [&](int m, int kk) { return Ks[(m0 + m) * LDM + kk]; };
    Strip p = zero_strip(), g = zero_strip();   // Q K^T and K K^T while the other tiles are in flight
    MMD(p, [&](int m, int kk) { return Qs[(m0 + m) * LDM + kk]; }, [&](int kk, int n) { return Ks[(n0 + n) * LDM + kk]; });
    if (!FROZEN) MMD32(g, aK, [&](int kk, int n) { return Ks[(n0 + n) * LDM + kk]; });
    {
        if (!FROZEN) commit(Ts, tt, tid);
        commit(Us, tu, tid);
        commit(A1, tdm, tid);
        if (has_s) commit(A2, tds, tid);
        const float x0 = wave_allreduce(tile_dot(tm, tdm));
        const float x1 = has_s ? wave_allreduce(tile_dot(ts, tdm)) : 0.f;
        const float x2 = has_s ? wave_allreduce(tile_dot(ts, tds)) : 0.f;
        if (l == 0) { dots[0][w] = x0; dots[1][w] = x1; dots[2][w] = x2; }
    }
    __syncthreads();
    if (tid < 3) {
        const float *pp = dots[tid];
        scal[task * 4 + tid] = ((pp[0] + pp[1]) + (pp[2] + pp[3])) + ((pp[4] + pp[5]) + (pp[6] + pp[7]));
    }
    auto publish = [&](int which, Strip &x) {   // row sums of x -> part[which][column half][row]
        strip_row_sums(x);
        if (row_writer(l)) {
#pragma unroll
            for (int i = 0; i < 4; i++) part[which][nh][m0 + row_of(i, l)] = x.t[0][i];
        }
    };
    auto aU = [&](int m, int kk) { return Us[(m0 + m) * LDM + kk]; };
    Strip udm = zero_strip(), uds = zero_strip();
    if (dcol) {
        Strip kdm = zero_strip(), kds = zero_strip();
        MMD32(kdm, aK, [&](int kk, int n) { return A1[(n0 + n) * LDM + kk]; });
        MMD32(udm, aU, [&](int kk, int n) { return A1[kk * LDM + n0 + n]; });
        if (has_s) {
            MMD32(kds, aK, [&](int kk, int n) { return A2[(n0 + n) * LDM + kk]; });
            MMD32(uds, aU, [&](int kk, int n) { return A2[kk * LDM + n0 + n]; });
        }
        const float *gi = dUg + task * kDD;
        Strip ud;
#pragma unroll
        for (int tl = 0; tl < 2; tl++)
#pragma unroll
            for (int i = 0; i < 4; i++) {
                const int row = m0 + row_of(i, l), col = n0 + 16 * tl + (l & 15);
                const float du = gi[row * HD + col] + cv.wM[row] * kdm.t[tl][i] + cv.wS[row] * kds.t[tl][i];
                B9[row * LDM + col] = du;   // dU
                if constexpr (FROZEN) {     // dR = dU
                    Ts[row * LDM + col] = du;
                    if (row < L) d_v[(tok + row) * D + col] = -du;
                    ud.t[tl][i] = du * Us[row * LDM + col];
                }
            }
        if constexpr (FROZEN) publish(6, ud);
    }
    __syncthreads();   // dU complete; dMo, dSo no longer needed
    if constexpr (!FROZEN) {
        Strip dr = zero_strip();
        // T^T is upper triangular: row block ib contracts over the blocks ib .. 3 of 16 (taken in pairs)
        if (dcol) {
            MMAR(dr, [&](int m, int kk) { return Ts[kk * LDM + m0 + m]; }, [&](int kk, int n) { return B9[kk * LDM + n0 + n]; },
                 ib >> 1, 2);
            FORC(dr, [&](int r, int c, float &x) {
                if (m0 + r < L) d_v[(tok + m0 + r) * D + n0 + c] = -x;
            });
            Strip ud = dr;
            FORC(ud, [&](int r, int c, float &x) { x *= Us[(m0 + r) * LDM + n0 + c]; });
            publish(6, ud);
        }
        __syncthreads();   // T no longer needed
        if (dcol) FORC(dr, [&](int r, int c, float &x) { Ts[(m0 + r) * LDM + n0 + c] = x; });   // dR
        __syncthreads();
    }
    const float *dRs = Ts;
    Strip dwa;
    {
        Strip dlam = zero_strip(), dyu = zero_strip();
        auto bU = [&](int kk, int n) { return Us[(n0 + n) * LDM + kk]; };
        if (!FROZEN) MMD(dlam, [&](int m, int kk) { return dRs[(m0 + m) * LDM + kk]; }, bU);
        MMD(dyu, [&](int m, int kk) { return Ds[(m0 + m) * LDM + kk]; }, bU);
#pragma unroll
        for (int tl = 0; tl < 2; tl++)
#pragma unroll
            for (int i = 0; i < 4; i++) {
                const int row = m0 + row_of(i, l), col = n0 + 16 * tl + (l & 15);
                const float nth = -cf.th[col];
                const float c0 = Cc[row * LDM + col], c1 = row > 0 ? Cc[(row - 1) * LDM + col] : 0.f;
                const float lam = (col < row && row < L) ? dlam.t[tl][i] : 0.f;
                const float yu = (col <= row && row < L) ? dyu.t[tl][i] : 0.f;
                B9[row * LDM + col] = nth * c0 * yu;            // dP = W . tril(dY U^T)
                if constexpr (!FROZEN) {
                    A2[row * LDM + col] = lam * g.t[tl][i];     // dLam . G, read one row down below
                    const float dg = nth * c1 * lam;            // dG, stored symmetrised
                    if (col < row) { A1[row * LDM + col] = dg; A1[col * LDM + row] = dg; }
                    if (col == row) A1[row * LDM + col] = 0.f;
                }
                dwa.t[tl][i] = yu * p.t[tl][i];
            }
    }
    __syncthreads();
    {
        float *xo = xs + task * CW * CW;
        float cs[2] = {0.f, 0.f};
#pragma unroll
        for (int tl = 0; tl < 2; tl++)
#pragma unroll
            for (int i = 0; i < 4; i++) {
                const int row = m0 + row_of(i, l), col = n0 + 16 * tl + (l & 15);
                const float dw = dwa.t[tl][i] + (!FROZEN && row + 1 < CW ? A2[(row + 1) * LDM + col] : 0.f);
                xo[col * CW + row] = -cf.th[col] * dw;          // [s][t]
                cs[tl] = fmaf(dw, Cc[row * LDM + col], cs[tl]);
            }
#pragma unroll
        for (int tl = 0; tl < 2; tl++) {
            float x = xor_add<16>(cs[tl]);
            x = xor_add<32>(x);
            if (l < 16) part_th[ib][n0 + 16 * tl + l] = x;
        }
    }
    __syncthreads();   // c and U no longer needed
    commit(Us, tm, tid);
    if (has_s) commit(Cc, ts, tid);
    __syncthreads();
    if (itask + 1 < task_hi) fetch_a(itask + 1, tid);
    const float *M0s = Us, *S0s = Cc, *dPs = B9, *dGs = A1;
    if (dcol) {
        Strip dym = zero_strip(), dys = zero_strip(), dq = zero_strip(), r0 = zero_strip(), r1 = zero_strip();
        auto aD = [&](int m, int kk) { return Ds[(m0 + m) * LDM + kk]; };
        MMD(dym, aD, [&](int kk, int n) { return M0s[kk * LDM + n0 + n]; });
        if (has_s) MMD(dys, aD, [&](int kk, int n) { return S0s[kk * LDM + n0 + n]; });
        MMA(dq, [&](int m, int kk) { return dPs[(m0 + m) * LDM + kk]; }, [&](int kk, int n) { return Ks[kk * LDM + n0 + n]; });
#pragma unroll
        for (int tl = 0; tl < 2; tl++)
#pragma unroll
            for (int i = 0; i < 4; i++) {
                const int row = m0 + row_of(i, l), col = n0 + 16 * tl + (l & 15);
                const float qv = Qs[row * LDM + col];
                r0.t[tl][i] = dym.t[tl][i] * qv;
                r1.t[tl][i] = dys.t[tl][i] * qv;
                if (row < L)
                    d_q[(tok + row) * D + col] = cf.a[row] * dym.t[tl][i] + cf.beta[row] * dys.t[tl][i] + dq.t[tl][i];
            }
        publish(0, r0);
        publish(1, r1);
    }
    if (dcol) {   // d_k in two halves: fewer accumulators alive at once
        Strip dk = zero_strip();
        {
            Strip r2 = zero_strip(), r3 = zero_strip();
            MMA(dk, [&](int m, int kk) { return dPs[kk * LDM + m0 + m]; }, [&](int kk, int n) { return Qs[kk * LDM + n0 + n]; });
            if (!FROZEN) MMA(dk, [&](int m, int kk) { return dGs[(m0 + m) * LDM + kk]; }, [&](int kk, int n) { return Ks[kk * LDM + n0 + n]; });
#pragma unroll
            for (int tl = 0; tl < 2; tl++)
#pragma unroll
                for (int i = 0; i < 4; i++) {
                    const int row = m0 + row_of(i, l), col = n0 + 16 * tl + (l & 15);
                    const float kv = Ks[row * LDM + col];
                    r2.t[tl][i] = udm.t[tl][i] * kv;
                    r3.t[tl][i] = uds.t[tl][i] * kv;
                    dk.t[tl][i] += cv.wM[row] * udm.t[tl][i] + cv.wS[row] * uds.t[tl][i];
                }
            publish(2, r2);
            publish(3, r3);
        }
        {
            Strip drm = zero_strip(), drs = zero_strip(), r4 = zero_strip(), r5 = zero_strip();
            auto aR = [&](int m, int kk) { return dRs[(m0 + m) * LDM + kk]; };
            MMD(drm, aR, [&](int kk, int n) { return M0s[kk * LDM + n0 + n]; });
            if (!FROZEN && has_s) MMD(drs, aR, [&](int kk, int n) { return S0s[kk * LDM + n0 + n]; });
#pragma unroll
            for (int tl = 0; tl < 2; tl++)
#pragma unroll
                for (int i = 0; i < 4; i++) {
                    const int row = m0 + row_of(i, l), col = n0 + 16 * tl + (l & 15);
                    const float kv = Ks[row * LDM + col];
                    r4.t[tl][i] = drm.t[tl][i] * kv;
                    r5.t[tl][i] = drs.t[tl][i] * kv;
                    if (row < L)
                        d_k[(tok + row) * D + col] = dk.t[tl][i] + cv.am[row] * drm.t[tl][i] + cv.bm[row] * drs.t[tl][i];
                }
            if constexpr (!FROZEN) {
                publish(4, r4);
                publish(5, r5);
            }
        }
    }
    __syncthreads();
    if (tid < L) {
        const int t = tid;
        auto sum = [&](int which, int row) { return D == 64 ? part[which][0][row] + part[which][1][row] : part[which][0][row]; };
        const float g1 = sum(2, t), g2 = sum(3, t);
        const float dam = !FROZEN && t + 1 < CW ? sum(4, t + 1) : 0.f, dbm = !FROZEN && t + 1 < CW ? sum(5, t + 1) : 0.f;
        // theta_t enters the rule as theta_t u_t, so that d_theta_t = u_t . dR_t / theta_t: one dot where the sum over the
        // tokens behind t adds up to 64 rounded products; that sum is left for a theta that dR vanishes with
        const float th = cf.th[t];
        d_theta[tok + t] = th > 1e-18f ? sum(6, t) / th
            : -(((part_th[0][t] + part_th[1][t]) + (part_th[2][t] + part_th[3][t])) + cf.cl[t] * g1 + cf.bl[t] * g2);
        float *pv = pvec + (tok + t) * 4;
        pv[0] = sum(0, t) + dam;
        pv[1] = sum(1, t) + dbm;
        pv[2] = -cf.th[t] * g1;
        pv[3] = -cf.th[t] * g2;
    }
    __syncthreads();   // LDS is rewritten by the next chunk
    }
}
constexpr size_t kExGradsLds = 9 * MAT * sizeof(float);

// ── the forward of the rule, pass 1: the chunk maps of the state scan ────────
//   M' = a_L M + beta_L S + U^T (wM.K),  S' = h_L S + U^T (wS.K)  with  U = Z1 M^T + Z2 S^T - T V,  Z1 = T (am.K), Z2 = T (bm.K)
// so the end state is affine in the start state with the matrices Z^T (w.K): the same scan as the backward's, first chunk
// first.  Nothing else leaves this pass; the tokens of a chunk are then walked from its start state by the sequential
// kernel (rule_fwd_kernel with FwdArgs::sub_chunks), all chunks at once.
template <int D, bool FROZEN>
__global__ __launch_bounds__(kThr) void ex_fwd_local_kernel(
    const float *__restrict__ k, const float *__restrict__ v, const float *__restrict__ alpha, const float *__restrict__ theta,
    const float *__restrict__ eta, float *__restrict__ loc, int s, int stride, int C, int nc, int maps, int has_s) {
    constexpr size_t DD = (size_t)D * D;
    extern __shared__ float smem[];
    float *Ks = smem, *Vs = Ks + MAT, *B8 = Vs + MAT, *Dg = B8 + MAT, *Nn = Dg + MAT, *Cc = Nn + MAT;
    __shared__ Coef cf;
    __shared__ ChunkVecs cv;
    const int tid = threadIdx.x, l = tid & 63, w = __builtin_amdgcn_readfirstlane(tid >> 6);
    NLH_STRIP_ORIGIN_OF(w);
    const bool dcol = D == 64 || nh == 0;
    auto MMAT = [&](f32x4 &acc, auto fa, auto fb, int k0) { mma_tile16(acc, fa, fb, k0, l); };
    const int chain = blockIdx.x / maps, ci = blockIdx.x % maps, t0 = ci * C, L = min(C, s - t0);
    const size_t tok = (size_t)chain * stride + t0;
    {
        TileD<D, 64> tk, tv;
        fetch(tk, k + tok * D, L, tid);
        fetch(tv, v + tok * D, L, tid);
        const Gates gt = fetch_gates(alpha + tok, theta + tok, eta + tok, L, has_s != 0);
        load_gates(cf, gt);
        coefficients<double>(cf, gt, L, Cc);
        commit(Ks, tk, tid);
        commit(Vs, tv, tid);
    }
    __syncthreads();
    chunk_vectors<FROZEN>(cv, cf, L);
    if constexpr (!FROZEN) {
    {
        Strip g = zero_strip();
        auto a = [&](int m, int kk) { return Ks[(m0 + m) * LDM + kk]; };
        auto b = [&](int kk, int n) { return Ks[(n0 + n) * LDM + kk]; };
        if constexpr (D == 64) mma(g, a, b, l); else mma_range(g, a, b, 0, D / 32, l);
        for_c(g, [&](int r, int c, float &x) {
            const int row = m0 + r, col = n0 + c;
            B8[row * LDM + col] = (col < row) ? -cf.th[col] * Cc[(row - 1) * LDM + col] * x : 0.f;   // Lam
        }, l);
    }
    __syncthreads();
#define INV_L B8
#define INV_D Dg
#define INV_N Nn
#define INV_X Cc
#define INV_BESIDE_N
#define INV_OUT(row, col, x)
#include "exact_inverse.h"
    if (dcol) {   // Z1 -> B8, Z2 -> Dg, T V -> Cc
        Strip tv = zero_strip(), z1 = zero_strip(), z2 = zero_strip();
        auto aT = [&](int m, int kk) { return Nn[(m0 + m) * LDM + kk]; };
        const int pe = (ib >> 1) + 1;
        mma_range_f64(tv, aT, [&](int kk, int n) { return Vs[kk * LDM + n0 + n]; }, 0, pe, l);
        mma_range_f64(z1, aT, [&](int kk, int n) { return cv.am[kk] * Ks[kk * LDM + n0 + n]; }, 0, pe, l);
        if (has_s) mma_range_f64(z2, aT, [&](int kk, int n) { return cv.bm[kk] * Ks[kk * LDM + n0 + n]; }, 0, pe, l);
        for_c(tv, [&](int r, int c, float &x) { Cc[(m0 + r) * LDM + n0 + c] = x; }, l);
        for_c(z1, [&](int r, int c, float &x) { B8[(m0 + r) * LDM + n0 + c] = x; }, l);
        if (has_s) for_c(z2, [&](int r, int c, float &x) { Dg[(m0 + r) * LDM + n0 + c] = x; }, l);
    }
    __syncthreads();
    } else __syncthreads();   // the vectors are there
    float *out = loc + ((size_t)chain * nc + ci) * kExLocMats * DD;
    const int sib = D == 64 ? ib : w & 1, sn0 = D == 64 ? n0 : 0, sm0 = 16 * sib;
    const int o0 = D == 64 ? 0 : w >> 1, ostep = D == 64 ? 1 : 4;
    const float aL = cf.a[L - 1], bL = cf.beta[L - 1], hL = cf.h[L - 1];
#pragma unroll 1
    for (int o = o0; o < 6; o += ostep) {   // matrix 2 * destination + source, then C_M, C_S
        if (!has_s && (o == 1 || o == 2 || o == 3 || o == 5)) continue;
        const float *wv = (o == 2 || o == 3 || o == 5) ? cv.wS : cv.wM;
        const float *Z = FROZEN ? (o >= 4 ? Vs : Ks) : o >= 4 ? Cc : (o & 1) ? Dg : B8;   // FROZEN: Z1 = K, Z2 = 0, T V = V
        Strip x = zero_strip();
        auto zt = [&](int m, int kk) { return Z[kk * LDM + sm0 + m]; };
        auto wk = [&](int kk, int n) { return (double)wv[kk] * Ks[kk * LDM + sn0 + n]; };
        if (!(FROZEN && (o == 1 || o == 3))) mma_f64(x, zt, wk, l);
        const float dg = o == 0 ? aL : o == 1 ? bL : o == 3 ? hL : 0.f;
        for_c(x, [&](int r, int c, float &y) { y = o >= 4 ? -y : sm0 + r == sn0 + c ? y + dg : y; }, l);
        float *mat = out + (size_t)o * DD;
#pragma unroll
        for (int tl = 0; tl < 2; tl++) {
            if (o < 4) store_operand_tile<D>(mat, x.t[tl], sib, sn0 / 16 + tl, l);
            else store_acc_tile<D>(mat, x.t[tl], sib, sn0 / 16 + tl, l);
        }
    }
}
constexpr size_t kExFwdLds = 6 * MAT * sizeof(float);

template <class K>
void set_lds(K kernel, size_t bytes) {
    check_hip(hipFuncSetAttribute(reinterpret_cast<const void *>(kernel), hipFuncAttributeMaxDynamicSharedMemorySize,
                                  (int)bytes), "dynamic LDS size");
}

}  // namespace

bool exact_mm_applies(int d, int C) { return (d == 64 || d == 32) && C >= 1 && C <= CW; }

// A chunk of the matrix form spans as many whole checkpoint intervals as fit into 64 tokens: a chunk costs the same
// whatever its length, and only the states at chunk starts are read.
static int chunk_of(int C) { return C * (CW / C); }

// Float64 sums (above) for what the walks served: head size 32, full trajectories, and intervals below 32, which pay since
// a chunk spans several of them.
static bool wide_sums(int d, int C) { return d == 32 || C < 32; }

// Cost models from measurements on one MI355X (us).  A chunk costs the two chunk-parallel kernels of the backward about
// 65 us of a compute unit whatever its length (95 with float64 sums, 46 + 49; the pass takes 92 more a round of chunks over
// 2 to 16 rounds, intervals of 8; 54 at head size 32), a scan step 2.0 (2.9, 0.65); the
// fused sequential kernel walks a chain's tokens at 0.6 each on a quarter of a compute unit's worth of workgroups (four per
// chain, one at head size 32), the kernel that reads a whole trajectory at 1.1.  Under a clip or a bound the test on the
// errors adds two launches to the matrix form where the fused kernel's only adds one on its maxima.  Matrix form / walk on
// both sides of the line, intervals of 8: 128 chains of 64 tokens 110 / 97, 160 115 / 137; 64 of 128 105 / 89, of 200 120 / 132;
// 192 of 96 202 / 194, 256 216 / 254.
bool exact_backward_mm_pays(int seq_len, int batch, int d, int C, bool tested, bool frozen) {
    const int nc = ceil_div(seq_len, frozen ? C : chunk_of(C)), cus = compute_units();
    const bool wide = wide_sums(d, C);
    const double chunk = d == 32 ? 54.0 : wide ? 95.0 : 65.0, step = d == 32 ? 0.65 : wide ? 2.9 : 2.0;
    const double t_mm = (double)ceil_div(batch * nc, cus) * chunk + nc * step + (tested ? 20.0 : 10.0);
    const double t_seq = (double)seq_len * (C == 1 ? 1.1 : 0.6) * ceil_div(batch * (d == 64 ? 4 : 1), cus);
    return t_mm < t_seq;
}

// The sequential forward takes 0.15 a token as long as its workgroups (four per chain, one at head size 32) fit the chip,
// and writes the states it keeps at 4.2 TB/s (32 chains of 512 tokens with their trajectory, 537 MB: 128 us).  The chunk
// maps cost 35 of a compute unit per chunk (20 at head size 32), a scan step 2.6 (0.65), and, unless only the final states
// are wanted, the walk of the chunks' tokens again 0.15 a token for whatever does not run at the same time, and the same
// writes.
bool exact_forward_mm_pays(int seq_len, int batch, int d, bool final_only, int run, long long kept_bytes) {
    const int nc = ceil_div(seq_len, run), cus = compute_units(), parts = d == 64 ? 4 : 1;
    if (nc < 2) return false;
    auto walk = [&](double tokens, long long groups) {
        const double t = 0.15 * tokens * ceil_div(groups, cus), w = (double)kept_bytes / 4.2e6;
        return t > w ? t : w;
    };
    double t_mm = (double)ceil_div(batch * (final_only ? nc : nc - 1), cus) * (d == 64 ? 35.0 : 20.0) + nc * (d == 64 ? 2.6 : 0.65) + 8.0;
    if (!final_only) t_mm += walk(run, (long long)batch * nc * parts);
    return t_mm < walk(seq_len, (long long)batch * parts);
}

template <int D, bool FROZEN>
static bool forward_states_t(bool has_s, const float *k, const float *v, const float *alpha, const float *theta, const float *eta,
                             const float *m_initial, const float *s_initial, long long m_stride, float *m_states, float *s_states,
                             long long state_stride, int sstep, int seq_len, int input_stride, int batch, int C) {
    const ErrorScope es;
    constexpr size_t DD = (size_t)D * D;
    // to the starts of all chunks, or (sstep 0) through the last one to the end; in stretches whose maps fit the scratch,
    // each from the states that the one before it left
    const int nc = ceil_div(seq_len, C), maps = sstep ? nc - 1 : nc;
    const size_t per_chunk = (size_t)batch * kExLocMats * DD * sizeof(float);
    const long long fit = (long long)(kOptionalScratch / per_chunk);
    const int stretch = fit < maps ? (int)fit : maps;
    if (stretch < 1) return false;
    float *loc = scratch_if_free(40, stretch * per_chunk);
    if (!loc) return false;
    static bool attr_set = false;
    if (!attr_set) {
        set_lds(ex_fwd_local_kernel<D, FROZEN>, kExFwdLds);
        attr_set = true;
    }
    for (int c0 = 0; c0 < maps && !es.failed(); c0 += stretch) {
        const int n = c0 + stretch < maps ? stretch : maps - c0;
        const size_t t0 = (size_t)c0 * C;
        {
            KernelTimer kt("ex_fwd_local_kernel");
            hipLaunchKernelGGL((ex_fwd_local_kernel<D, FROZEN>), dim3((unsigned)batch * n), dim3(kThr), kExFwdLds, stream(), k + t0 * D,
                               v + t0 * D, alpha + t0, theta + t0, (has_s ? eta : alpha) + t0, loc, seq_len - (int)t0, input_stride, C, n, n,
                               (int)has_s);
            check_launch("ex_fwd_local_kernel");
        }
        KernelTimer kt("ex_scan_kernel");
        const dim3 grid((unsigned)batch * (D / 16));
        float *ms = m_states + (size_t)c0 * sstep * DD, *ss = has_s ? s_states + (size_t)c0 * sstep * DD : nullptr;
        const float *mi = c0 ? ms : m_initial, *si = c0 ? ss : s_initial;
        const long long stride = c0 ? state_stride : m_stride;
        if (has_s)
            hipLaunchKernelGGL((ex_scan_kernel<D, true, false, true>), grid, dim3(8 * D), 0, stream(), loc, mi, si, stride, ms, ss,
                               state_stride, sstep, nullptr, nullptr, n, n);
        else
            hipLaunchKernelGGL((ex_scan_kernel<D, false, false, true>), grid, dim3(4 * D), 0, stream(), loc, mi, nullptr, stride, ms, nullptr,
                               state_stride, sstep, nullptr, nullptr, n, n);
        check_launch("ex_scan_kernel");
    }
    return true;
}

bool exact_forward_states(bool has_s, bool frozen, int d, int run, const float *k, const float *v, const float *alpha, const float *theta,
                          const float *eta, const float *m_initial, const float *s_initial, long long m_stride, float *m_states,
                          float *s_states, long long state_stride, int sstep, int seq_len, int input_stride, int batch) {
    auto fn = frozen ? forward_states_t<32, true> : d == 64 ? forward_states_t<64, false> : forward_states_t<32, false>;
    return fn(has_s, k, v, alpha, theta, eta, m_initial, s_initial, m_stride, m_states, s_states, state_stride, sstep, seq_len,
              input_stride, batch, run);
}

template <int D, bool FROZEN, bool P64>
static bool backward_mm_t(const char *fn, bool has_s, const float *k, const float *v, const float *q, const float *alpha,
                          const float *theta, const float *eta, const float *m_ckpt, const float *s_ckpt, const float *d_y,
                          float *d_k, float *d_v, float *d_q, float *d_alpha, float *d_theta, float *d_eta, float *d_m_initial,
                          float *d_s_initial, int seq_len, int batch, int interval, float error_clip, float m_norm_guard) {
    const ErrorScope es;
    constexpr size_t DD = (size_t)D * D;
    const int C = FROZEN ? interval : chunk_of(interval), cstep = C / interval;   // a frozen chunk is what the caller says
    const int nc = ceil_div(seq_len, C), nck = interval == 1 ? seq_len + 1 : n_ckpt_count(seq_len, interval);
    const size_t nchunks = (size_t)batch * nc;
    const bool guard = error_clip > 0.f || m_norm_guard > 0.f;
    ChainTracks tracks{nullptr, nullptr};
    if (guard) tracks = chain_tracks(seq_len, batch, C);
    float *loc = scratch(32, nchunks * kExLocMats * DD * sizeof(float));
    float *Tg = scratch(33, nchunks * kDD * sizeof(float));
    float *Ug = scratch(34, nchunks * kDD * sizeof(float));
    float *dUg = scratch(35, nchunks * kDD * sizeof(float));
    float *em = scratch(5, (size_t)batch * (nc + 1) * DD * sizeof(float));
    float *esn = has_s ? scratch(6, (size_t)batch * (nc + 1) * DD * sizeof(float)) : nullptr;
    float *xs = scratch(7, nchunks * CW * CW * sizeof(float));
    float *pvec = scratch(8, (size_t)batch * seq_len * 4 * sizeof(float));
    float *scal = scratch(9, nchunks * 4 * sizeof(float));
    const int per = 8, rows = ceil_div(batch, per), nsum = has_s ? 2 : 1;
    float *tmp = scratch(10, (size_t)nsum * rows * DD * sizeof(float));
    float *first = scratch(36, (size_t)2 * batch * DD * sizeof(float));
    if (es.failed()) return true;
    float *first_m = first, *first_s = first + (size_t)batch * DD;
    static bool attr_set = false;
    if (!attr_set) {
        set_lds(ex_local_kernel<D, FROZEN, false, P64>, kExLocalLds);
        set_lds(ex_local_kernel<D, FROZEN, true, P64>, kExLocalLds);
        set_lds(ex_grads_kernel<D, FROZEN, P64>, kExGradsLds);
        attr_set = true;
    }
    if (es.failed()) return true;
    const int cus = compute_units(), pgrid = nchunks < (size_t)cus ? (int)nchunks : cus;   // one workgroup per compute unit (LDS)
    const float *et = has_s ? eta : alpha;
    {
        KernelTimer kt("ex_local_kernel");
        auto kernel = guard ? ex_local_kernel<D, FROZEN, true, P64> : ex_local_kernel<D, FROZEN, false, P64>;
        hipLaunchKernelGGL(kernel, dim3((unsigned)pgrid), dim3(kThr), kExLocalLds, stream(), k, v, q, d_y, alpha, theta, et,
                           m_ckpt, s_ckpt, loc, Tg, Ug, dUg, seq_len, C, nc, nck, cstep, (int)has_s, (int)nchunks, tracks);
        check_launch("ex_local_kernel");
    }
    {
        KernelTimer kt("ex_scan_kernel");
        const dim3 grid((unsigned)batch * (D / 16));
        const long long stride = (long long)(nc + 1) * DD;
        if (has_s)
            hipLaunchKernelGGL((ex_scan_kernel<D, true, true, P64>), grid, dim3(8 * D), 0, stream(), loc, nullptr, nullptr, 0LL, em, esn,
                               stride, 1, first_m, first_s, nc, nc);
        else
            hipLaunchKernelGGL((ex_scan_kernel<D, false, true, P64>), grid, dim3(4 * D), 0, stream(), loc, nullptr, nullptr, 0LL, em, nullptr,
                               stride, 1, first_m, nullptr, nc, nc);
        check_launch("ex_scan_kernel");
    }
    {
        KernelTimer kt("ex_grads_kernel");
        hipLaunchKernelGGL((ex_grads_kernel<D, FROZEN, P64>), dim3((unsigned)pgrid), dim3(kThr), kExGradsLds, stream(), k, q, d_y, alpha, theta,
                           et, m_ckpt, s_ckpt, Tg, Ug, dUg, em, esn, d_k, d_v, d_q, d_theta, pvec, xs, scal, seq_len, C, nc, nck, cstep,
                           (int)has_s, (int)nchunks);
        check_launch("ex_grads_kernel");
    }
    chunkwise_gate_gradients(alpha, eta, pvec, xs, scal, d_alpha, d_eta, seq_len, batch, C, has_s, first_m, first_s, DD, per,
                             nsum, tmp, (int)DD, P64);
    if (es.failed()) return true;
    if (guard && couplings_may_fire_tracked(k, alpha, theta, eta, tracks, has_s, seq_len, batch, C, error_clip, m_norm_guard, D))
        return false;
    accumulate_over_batch2(tmp, d_m_initial, has_s ? tmp + (size_t)rows * DD : nullptr, d_s_initial, rows, (int)DD);
    return true;
}

bool exact_backward_mm(const char *fn, bool has_s, bool frozen, int d, const float *k, const float *v, const float *q, const float *alpha,
                       const float *theta, const float *eta, const float *m_ckpt, const float *s_ckpt, const float *d_y,
                       float *d_k, float *d_v, float *d_q, float *d_alpha, float *d_theta, float *d_eta, float *d_m_initial,
                       float *d_s_initial, int seq_len, int batch, int C, float error_clip, float m_norm_guard) {
    if (seq_len <= 0 || batch <= 0 || !exact_mm_applies(d, C)) {
        fail("%s: the matrix form needs seq_len=%d and batch=%d positive, head size %d of 64 or 32 and a checkpoint interval %d in [1, %d].",
             fn, seq_len, batch, d, C, CW);
        return true;
    }
    auto run = frozen ? backward_mm_t<32, true, true>
               : d == 32 ? backward_mm_t<32, false, true>
               : wide_sums(d, C) ? backward_mm_t<64, false, true> : backward_mm_t<64, false, false>;
    return run(fn, has_s, k, v, q, alpha, theta, eta, m_ckpt, s_ckpt, d_y, d_k, d_v, d_q, d_alpha, d_theta, d_eta, d_m_initial,
               d_s_initial, seq_len, batch, C, error_clip, m_norm_guard);
}

}  // namespace nlh
