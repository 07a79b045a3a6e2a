// HOPE self-referential memory, forward for chunks of up to 64 tokens, as three launches or as the same work in one.
//
// With the snapshot F_c of the chunk's start every memory moves by one outer product a token,
//     M_c <- (1-a_t) M_c + th_t w_c,t k_t^T,    w_c,t = v_t - F_c k_t   (self-generated values: F_c (v_t - k_t)),
// and only k_t = M_k x_t, v_t = M_v x_t and the gates (means over the rows of M_alpha x_t, M_eta x_t) feed back into
// the recurrence.  So the part that is bound to one workgroup per chain carries M_k, M_v and the row means of M_alpha,
// M_eta, M_v; what hangs off it (the other four memories, q_t = M_q x_t and y_t = M_mem q_t) is left to kernels that
// use the whole chip:
//   selfref_chain_kernel  one workgroup per chain:               k, v, gates, snapshots of M_k, M_v
//   selfref_scan_kernel   one workgroup per (chain, memory):     M_q, M_eta, M_alpha, M_mem chunk by chunk
//   selfref_read_kernel   one workgroup per (chain, chunk):      q and y from the snapshots
//   selfref_forward_kernel   all of it, the others a chunk behind the chains: where these leave compute units idle
#include <hip/hip_runtime.h>

#include <utility>

#include "../../include/nl_hecate_ffi.h"
#include "handover.h"
#include "lane_ops.h"
#include "quad_rows.h"
#include "runtime.h"
#include "selfref_chunk.h"

namespace nlh {
namespace {

template <int Q>
__device__ __forceinline__ float quad_lane(float x) { return dpp_mov<Q * 0x55>(x); }
// The gates of x without a branch, from e = 1 + exp(-x) and e = 1 + exp(x).
__device__ __forceinline__ float sigmoid_of(float x, float e) {
    const float y = __builtin_amdgcn_rcpf(e);
    return x >= 15.f ? 1.f : x <= -15.f ? 0.f : y;
}
__device__ __forceinline__ float softplus_of(float x, float e) {
    constexpr float ln2 = 0x1.62e43p-1f, ln2_rest = -0x1.05c61p-29f;  // ln 2 in two parts
    const float l = __builtin_amdgcn_logf(e), p = l * ln2;
    const float y = p + fmaf(l, ln2_rest, fmaf(l, ln2, -p));
    return x >= 15.f ? x : x <= -15.f ? 0.f : y;
}

__device__ __forceinline__ double lane_value64(double x, int lane) {
    const long long u = __builtin_bit_cast(long long, x);
    const unsigned lo = __builtin_amdgcn_readlane((int)u, lane), hi = __builtin_amdgcn_readlane((int)(u >> 32), lane);
    return __builtin_bit_cast(double, (long long)(((unsigned long long)hi << 32) | lo));
}

// What lanes of a wave hand to each other through LDS: the hardware keeps a wave's LDS accesses in order, this the compiler.
__device__ __forceinline__ void wave_lds_fence() { asm volatile("" ::: "memory"); }

// f(0), f(1), ... with the argument as a type, until one returns false
template <class Fn, int... I>
__device__ __forceinline__ void while_true(Fn &f, std::integer_sequence<int, I...>) {
    (void)(f(std::integral_constant<int, I>{}) && ...);
}

// ── the recurrence ───────────────────────────────────────────────────────────────────────────────────────────────
// Tiles of 16 tokens.  At a tile's start P0_c = M_c X^T for the whole tile comes off the matrix cores; inside the tile
// token t adds its outer product to the later columns only, P_c[t'] = (1-a_t) P_c[t'] + th_t w_c,t (k_t . x_t') from
// zero, and the value of column t' is A_t' P0_c[t'] + P_c[t'] with A the retentions so far, so a token needs k_t in all
// waves (one LDS exchange), the products F_k k_t, F_v k_t and the dots of k_t with the tile's x and with the row means;
// at the tile's end M_c takes the sum of the 16 outer products on the matrix cores.
//
// Rounding feeds back (k into the gates, the gates into every later state), and a saturated gate is the rounding of its
// mean, whose terms are large and of one sign.  So what the tile starts with and what its tokens add are kept apart, each
// sum is formed by itself and joined once, the retentions are a float64 product, and the means' P0 is summed and kept in
// float64.  With one running fp32 value per column y was 1.25 times as far from float64 as with token by token products,
// the gates 1.4 to 2 times; so it is 0.65 and 0.4 times, for 0.08 ms.
//
// Two lane layouts, one a permutation of the other's lanes: the matrix cores' (ml, kg) = (lane % 16, lane / 16) and the
// quads' (r, cq) = (lane / 4, lane % 4).  Lane (ml, kg) holds row ml of the wave's 16 rows, columns 16 kt + 4 kg + v,
// which is at once operand and result of the two products (the contraction index runs over (v, kt) in any order);
// lane (r, cq) holds row r, columns 16 kt + 4 cq + v of F, so that a product with a vector is 16 fused
// multiply-adds and two DPP adds.  Tokens of a tile go to the matrix cores in the order sigma(4 a + b) = 4 b + a:
// lane cq then owns the columns t' = 4 j + cq of P, and column group j is finished with token 4 j + 3.
// The row means (alpha, eta, v) and the gates are one more wave's: a token's gates are wanted only at the end of its step, so
// the wave hands them over with the token's exchange and works a token ahead in the others' shadow.  It keeps the means and
// the next token's x as four rows of 16 lanes (four multiply-adds and four DPP adds give the means' products and k . x of the
// next token at once), its own columns' values a lane each, and goes first on the SIMD that it shares.
//
// Bound by the issue rate of one wave per SIMD: 820 clocks a token (120 vector and LDS instructions of the first four waves,
// the exchange), 4000 for a tile's start and end.  64 chains of 2048 tokens, head size 64, chunks of 64: 0.92 ms, 1.26 with the
// means in every wave; with the two kernels below 1.14 ms one after the other and 0.98 beside each other; one kernel that formed all products of a token with all six
// memories in sequence (it serves longer chunks, selfref.hip) takes 2.29 ms.  Chunks of 1, 4, 8, 16 tokens at 64 chains of
// 512: 6.64, 2.04, 1.27, 0.88 ms there, 3.84, 1.15, 0.70, 0.47 ms with the means in every wave.

// done: with others waiting for this chain's chunks (selfref_forward_kernel), how many of them there are.
template <int D, bool SG, bool WAITED>
__device__ __forceinline__ void chain_of(const SelfrefForward &a, size_t b, unsigned *done) {
    float *const mems = a.mems, *const k_cache = a.k, *const v_cache = a.v, *const alpha_cache = a.alpha, *const theta_cache = a.theta,
                 *const amean_cache = a.amean, *const emean_cache = a.emean, *const frozen = a.frozen;
    const float *const emb = a.emb;
    const int s = a.s, C = a.C, nc = a.nc;
    constexpr int KT = D / 16, NW = D / 16, DD = D * D, LD = D + 16, V4 = D / 4;
    __shared__ __align__(16) float xt[2][kTB * LD];
    __shared__ __align__(16) float Kt[2][kTB * LD], Vt[2][kTB * LD];  // the tile's k, v: exchange and operand
    // k - v, exchange only; two as well: a tile of one token has a single barrier, behind which a slow wave still reads its
    // row while a fast one writes the next tile's first
    __shared__ __align__(16) float Ut[2][SG ? kTB * LD : 4];
    // k_t . x_t' of the tile's later tokens: a wave's own, two of them because the gates' wave reads the first wave's a step later
    __shared__ __align__(16) float Sx[2][NW][kTB];
    __shared__ __align__(16) float mean[4][D];         // row means of M_alpha, M_eta, M_v, as the tile starts; a row of zeros
    __shared__ __align__(16) float mean_c[3][D];       // the same as the chunk starts
    __shared__ __align__(16) float gate[2][kTB][4];    // a token's 1 - alpha, the retentions of the tile up to it, theta twice

    const int tid = threadIdx.x, wave = tid >> 6, lane = tid & 63, wr = 16 * wave;
    const int ml = lane & 15, kg = lane >> 4, r = lane >> 2, cq = lane & 3;
    const int to_quad = 4 * (r + 16 * cq), to_mm = 4 * (4 * ml + kg);  // source lanes of the two permutations, in bytes
    const size_t tok0 = b * (size_t)s;
    float *mb = mems + b * 6 * DD;

    for (int e = tid; e < 4 * D; e += 4 * D + 64) {
        const int which = e / D;
        float a = 0.f;
        if (which < 3) {
            const float *src = mb + (which == 0 ? 4 : which == 1 ? 3 : 1) * DD + e % D;
#pragma unroll 8
            for (int c = 0; c < D; c++) a += src[c * D];
        }
        mean[which][e % D] = a * (1.f / D);
    }
    // the rows of a partial tile behind its last token enter the end-of-tile product times zero
    for (int e = tid; e < kTB * LD; e += 4 * D + 64) Kt[0][e] = Kt[1][e] = 0.f;
    // first token behind the tile that starts at t
    auto tile_end = [&](int t) { return min(min(t + kTB, (t / C + 1) * C), s); };

    if (wave == NW) {  // the gates
        __builtin_amdgcn_s_setprio(3);   // every token waits for them, and another wave issues on the same SIMD
        // lane (row, col): row of the means, or token t + 1's x as a fourth; columns 4 col .. 4 col + 3 of it, or the tile's token col
        constexpr int LR = D / 4;   // lanes of a row that hold columns
        const int row = lane >> 4, col = lane & 15, c4 = 4 * (col & (LR - 1));
        const bool writer = row < 3 && (D == 64 || col < LR);
        const float scale = row == 0 ? -1.4426950408889634f : 1.4426950408889634f;   // exp(-x) of alpha's mean, exp(x) of eta's
        __syncthreads();
        f32x4 M = *reinterpret_cast<const f32x4 *>(&mean[row][c4]);
        int chunk_t = 0, whole = 0, told = 0;   // chunks in front of the tile before; as the others know
        for (int tb = 0, te, buf = 0; tb < s; tb = te, buf ^= 1) {
            te = tile_end(tb);
            const int nt = te - tb;
            const float *Kb = Kt[buf], *Ub = Ut[buf];
            if (writer) *reinterpret_cast<f32x4 *>(&mean[row][c4]) = M;
            if (tb == chunk_t) {
                if (writer) *reinterpret_cast<f32x4 *>(&mean_c[row][c4]) = M;
                chunk_t += C;
            }
            wave_lds_fence();
            // Means times the tile's x in float64: a block of the instruction is the means' four rows by four tokens, its
            // result row lane / 16, token lane % 16.
            double P0 = 0.;
#pragma unroll
            for (int kt = 0; kt < KT; kt++) {
                const f32x4 m4 = *reinterpret_cast<const f32x4 *>(&mean[lane & 3][16 * kt + 4 * row]);
                const f32x4 x4 = *reinterpret_cast<const f32x4 *>(&xt[buf][col * LD + 16 * kt + 4 * row]);
#pragma unroll
                for (int v = 0; v < 4; v++) P0 = __builtin_amdgcn_mfma_f64_4x4x4f64((double)m4[v], (double)x4[v], P0, 0, 0, 0);
            }
            // Value of column t' = col before token t': retentions times P0, as two floats, plus what the tile's tokens added.
            float P = 0.f, pw = 0.f, pkeep = 1.f, mine = 0.f;
            float high = (float)P0, low = (float)(P0 - (double)high), now = high;
            double kept = 1.;
            float W[kTB], th[kTB], keep[kTB];
#pragma unroll
            for (int t = 0; t < kTB; t++) { W[t] = th[t] = 0.f; keep[t] = 1.f; }
            const float *other = row == 3 ? &xt[buf][LD + c4] : &mean_c[row][c4];
            auto step = [&](auto T) __attribute__((always_inline)) -> bool {
                constexpr int t = decltype(T)::value;
                // lane (0, t): alpha's mean, lane (1, t): eta's; both gates in every lane
                const float e = 1.f + __builtin_amdgcn_exp2f(now * scale);
                const float sig = sigmoid_of(now, e), soft = softplus_of(now, e);
                const float mean_v = now;
                mine = col == t ? now : mine;
                const float keep_l = 1.f - sig;
                const double kept_l = kept * (1. - (double)sig);
                if (col == t && row < 2)
                    *reinterpret_cast<float2 *>(&gate[buf][t][2 * row]) = row == 0 ? make_float2(keep_l, (float)kept_l) : make_float2(soft, soft);
                const f32x4 m = *reinterpret_cast<const f32x4 *>(other);
                if (t + 2 < kTB) other += row == 3 ? LD : 0;
                lds_barrier();
                if (WAITED && t == 0) {
                    if (whole >= told + kTellChunks || (whole > told && whole >= nc - kTellChunks)) {
                        told = whole;
                        tell(done, told);
                    }
                    whole = tb / C;
                }
                // row 3: x of the next token against k, the other rows the means against u
                const f32x4 u = *reinterpret_cast<const f32x4 *>((SG && row < 3 ? Ub : Kb) + t * LD + c4);
                float ps = 0.f;
                if (t > 0 && t + 1 < kTB) ps = Sx[(t - 1) & 1][0][sigma(col)];
                __builtin_amdgcn_sched_barrier(0);
                keep[t] = lane_value(keep_l, t);
                th[t] = SG ? -lane_value(soft, 16 + t) : lane_value(soft, 16 + t);
                const float vm = SG ? 0.f : lane_value(mean_v, 32 + t);
                kept = lane_value64(kept_l, t);
                const double P1 = kept * P0;
                high = (float)P1;
                low = (float)(P1 - (double)high);
                if (t > 0 && t + 1 < kTB) P = fmaf(pw, ps, pkeep * P);
                const float rest = fmaf(keep[t], P, low);
                const float dot = group_allreduce<LR>((m[0] * u[0] + m[1] * u[1]) + (m[2] * u[2] + m[3] * u[3]));
                W[t] = SG ? dot : vm - dot;
                if constexpr (t + 1 < kTB) {
                    pw = th[t] * W[t];
                    pkeep = keep[t];
                    now = high + fmaf(pw, lane_value(dot, 48), rest);
                }
                return t + 1 < nt;
            };
            while_true(step, std::make_integer_sequence<int, kTB>{});
            // as the other memories: the tile's sum by itself, joined once
            f32x4 add = f32x4{0.f, 0.f, 0.f, 0.f};
            float behind = 1.f;
#pragma unroll
            for (int t = kTB - 1; t >= 0; t--) {
                const f32x4 k4 = *reinterpret_cast<const f32x4 *>(Kb + t * LD + c4);
                const float c = W[t] * (th[t] * behind);
                behind *= keep[t];
#pragma unroll
                for (int v = 0; v < 4; v++) add[v] = fmaf(c, k4[v], add[v]);
            }
#pragma unroll
            for (int v = 0; v < 4; v++) M[v] = fmaf((float)kept, M[v], add[v]);
            if (WAITED) stores_arrived();
            if (col < nt) {
                const size_t o = tok0 + tb + col;
                const float e = 1.f + __builtin_amdgcn_exp2f(mine * scale);
                if (row == 0) { alpha_cache[o] = sigmoid_of(mine, e); amean_cache[o] = mine; }
                if (row == 1) { theta_cache[o] = softplus_of(mine, e); emean_cache[o] = mine; }
            }
        }
        if (WAITED) {
            stores_arrived();
            lds_barrier();
            tell(done, nc);
        }
        return;
    }
    const int stt = tid / V4, sj = (tid % V4) * 4;  // staging slot: token, column
    auto load_x = [&](int t, int n) -> float4 {
        return stt < n ? *reinterpret_cast<const float4 *>(emb + (tok0 + t + stt) * D + sj) : make_float4(0, 0, 0, 0);
    };
    int te = tile_end(0);
    *reinterpret_cast<float4 *>(&xt[0][stt * LD + sj]) = load_x(0, te);
    float4 xnext = te < s ? load_x(te, tile_end(te) - te) : make_float4(0, 0, 0, 0);
    // M_k, M_v in the matrix cores' layout
    f32x4 M[2][KT];
#pragma unroll
    for (int c = 0; c < 2; c++) {
#pragma unroll
        for (int kt = 0; kt < KT; kt++)
            M[c][kt] = *reinterpret_cast<const f32x4 *>(mb + c * DD + (wr + ml) * D + 16 * kt + 4 * kg);
    }
    __syncthreads();

    float F[2][4 * KT];
    int chunk_t = 0, ci = 0;
    for (int tb = 0, buf = 0; tb < s; tb = te, buf ^= 1) {
        te = tile_end(tb);
        const int nt = te - tb;
        float *Kb = Kt[buf], *Vb = Vt[buf], *Ub = Ut[buf];
        if (tb == chunk_t) {  // snapshot
            float *fb = frozen + (b * nc + ci) * (size_t)6 * DD;
#pragma unroll
            for (int c = 0; c < 2; c++) {
#pragma unroll
                for (int kt = 0; kt < KT; kt++) {
                    *reinterpret_cast<f32x4 *>(fb + c * DD + (wr + ml) * D + 16 * kt + 4 * kg) = M[c][kt];
#pragma unroll
                    for (int v = 0; v < 4; v++) F[c][4 * kt + v] = lane_from(to_quad, M[c][kt][v]);
                }
            }
            ci++;
            chunk_t += C;
        }
        // the next tile's x: requested a tile ago, visible after this tile's first exchange
        if (te < s) {
            *reinterpret_cast<float4 *>(&xt[buf ^ 1][stt * LD + sj]) = xnext;
            const int t2 = tile_end(te);
            if (t2 < s) xnext = load_x(t2, tile_end(t2) - t2);
        }
        float P0[2][4], P[2][4], X[4 * KT];   // M_c X^T as the tile starts, and what its tokens add
        {
            f32x4 acc[2][KT];   // a sum per 16 columns, added up in a tree
#pragma unroll
            for (int kt = 0; kt < KT; kt++) {
                const f32x4 xa = *reinterpret_cast<const f32x4 *>(&xt[buf][sigma(ml) * LD + 16 * kt + 4 * kg]);
                const f32x4 xq = *reinterpret_cast<const f32x4 *>(&xt[buf][sigma(r) * LD + 16 * kt + 4 * cq]);
#pragma unroll
                for (int c = 0; c < 2; c++) acc[c][kt] = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
                for (int v = 0; v < 4; v++) {
                    X[4 * kt + v] = xq[v];
#pragma unroll
                    for (int c = 0; c < 2; c++) acc[c][kt] = mfma4(xa[v], M[c][kt][v], acc[c][kt]);
                }
            }
#pragma unroll
            for (int c = 0; c < 2; c++) {
                f32x4 t = acc[c][0];
                if constexpr (KT == 2) t += acc[c][1];
                if constexpr (KT == 4) t = (t + acc[c][1]) + (acc[c][2] + acc[c][3]);
#pragma unroll
                for (int v = 0; v < 4; v++) P0[c][v] = lane_from(to_quad, t[v]);
            }
#pragma unroll
            for (int v = 0; v < 4; v++) {
                P[0][v] = P[1][v] = 0.f;
            }
        }
        float W[2][4], cs[4], kept = 1.f;  // w_c of token 4 j + cq, th times the retention since, of the whole tile
#pragma unroll
        for (int j = 0; j < 4; j++) W[0][j] = W[1][j] = cs[j] = 0.f;
        float k = quad_lane<0>(P0[0][0]), v = quad_lane<0>(P0[1][0]);
        // what token t - 1 adds to the columns behind t is added while token t's exchange is under way
        float pw[2] = {0.f, 0.f}, pkeep = 1.f;
        float *const out = (SG ? (cq == 0 ? Kb : cq == 1 ? Vb : Ub) : (cq & 1) ? Vb : Kb) + wr + r;

        auto step = [&](auto T) __attribute__((always_inline)) -> bool {
            constexpr int t = decltype(T)::value, J = t / 4, Q = t % 4;
            // every lane of a quad writes, so that no lane is masked out
            float val = k;
            if (SG) {
                const float u = k - v;
                val = cq == 1 ? v : u;
                val = cq == 0 ? k : val;
            } else {
                val = (cq & 1) ? v : k;
            }
            out[t * LD] = val;
            lds_barrier();
            float kc[4 * KT], uc[4 * KT];
            f32x4 ps = f32x4{0.f, 0.f, 0.f, 0.f};
            if (t > 0 && t + 1 < kTB) ps = *reinterpret_cast<const f32x4 *>(&Sx[(t - 1) & 1][wave][4 * cq]);
            const f32x4 g = *reinterpret_cast<const f32x4 *>(gate[buf][t]);
#pragma unroll
            for (int kt = 0; kt < KT; kt++) {
                const f32x4 k4 = *reinterpret_cast<const f32x4 *>(Kb + t * LD + 16 * kt + 4 * cq);
                f32x4 u4 = k4;
                if (SG) u4 = *reinterpret_cast<const f32x4 *>(Ub + t * LD + 16 * kt + 4 * cq);
#pragma unroll
                for (int i = 0; i < 4; i++) { kc[4 * kt + i] = k4[i]; uc[4 * kt + i] = u4[i]; }
            }
            __builtin_amdgcn_sched_barrier(0);  // what follows runs while the reads are under way, not ahead of the barrier
            if constexpr (t > 0 && t + 1 < kTB) {
#pragma unroll
                for (int j = (t + 1) / 4; j < 4; j++) {
#pragma unroll
                    for (int c = 0; c < 2; c++) {
                        P[c][j] = fmaf(pw[c], ps[j], pkeep * P[c][j]);
                        asm volatile("" : "+v"(P[c][j]));  // here, not when the column is needed
                    }
                }
            }
            const float S = quad_allreduce(dotn<4 * KT>(X, kc));  // row r: k_t . x of token sigma(r)
            float w[2];  // w_c,t (self-generated values: its negative)
#pragma unroll
            for (int c = 0; c < 2; c++) {
                w[c] = quad_allreduce(dotn<4 * KT>(F[c], uc));
                if (!SG) w[c] = v - w[c];
            }
            const float th = SG ? -g[2] : g[2], keep = g[0];
#pragma unroll
            for (int j = 0; j <= J; j++) cs[j] *= keep;
            kept = g[1];
            cs[J] = cq == Q ? th : cs[J];
#pragma unroll
            for (int c = 0; c < 2; c++) W[c][J] = cq == Q ? w[c] : W[c][J];
            if constexpr (t + 1 < kTB) {
                constexpr int J1 = (t + 1) / 4, Q1 = (t + 1) % 4;
                const float s1 = lane_value(S, 4 * sigma(t + 1));
#pragma unroll
                for (int c = 0; c < 2; c++) pw[c] = th * w[c];
                pkeep = keep;
                k = fmaf(kept, quad_lane<Q1>(P0[0][J1]), fmaf(pw[0], s1, keep * quad_lane<Q1>(P[0][J1])));
                v = fmaf(kept, quad_lane<Q1>(P0[1][J1]), fmaf(pw[1], s1, keep * quad_lane<Q1>(P[1][J1])));
                if (t + 2 < kTB) Sx[t & 1][wave][r] = S;  // read behind the next exchange
            }
            return t + 1 < nt;
        };
        while_true(step, std::make_integer_sequence<int, kTB>{});

        // M_c <- keep M_c + sum_t cs_t w_c,t k_t^T; every wave has written its part of Kb, Vb.  The tile's sum is formed by
        // itself, so that M_c rounds once a tile and not once a token
        f32x4 add[2][KT];
#pragma unroll
        for (int c = 0; c < 2; c++) {
#pragma unroll
            for (int kt = 0; kt < KT; kt++) add[c][kt] = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
            for (int j = 0; j < 4; j++) W[c][j] = lane_from(to_mm, W[c][j] * cs[j]);
        }
#pragma unroll
        for (int j = 0; j < 4; j++) {
            if (4 * j < nt) {
#pragma unroll
                for (int kt = 0; kt < KT; kt++) {
                    const float a = Kb[(4 * j + kg) * LD + 16 * kt + ml];
#pragma unroll
                    for (int c = 0; c < 2; c++) add[c][kt] = mfma4(a, W[c][j], add[c][kt]);
                }
            }
        }
#pragma unroll
        for (int c = 0; c < 2; c++) {
#pragma unroll
            for (int kt = 0; kt < KT; kt++) {
#pragma unroll
                for (int v = 0; v < 4; v++) M[c][kt][v] = fmaf(kept, M[c][kt][v], add[c][kt][v]);
            }
        }
        // What this wave stored in earlier tiles has arrived long ago; behind the next tile's first barrier that holds for all.
        if (WAITED) stores_arrived();
        if (stt < nt) {
            const size_t o = (tok0 + tb + stt) * D + sj;
            *reinterpret_cast<float4 *>(k_cache + o) = *reinterpret_cast<const float4 *>(Kb + stt * LD + sj);
            *reinterpret_cast<float4 *>(v_cache + o) = *reinterpret_cast<const float4 *>(Vb + stt * LD + sj);
        }
    }
#pragma unroll
    for (int c = 0; c < 2; c++) {
#pragma unroll
        for (int kt = 0; kt < KT; kt++)
            *reinterpret_cast<f32x4 *>(mb + c * DD + (wr + ml) * D + 16 * kt + 4 * kg) = M[c][kt];
    }
    if (WAITED) {
        stores_arrived();
        lds_barrier();
    }
}
template <int D, bool SG>
__global__ __launch_bounds__(4 * D + 64) void selfref_chain_kernel(SelfrefForward a) {
    chain_of<D, SG, false>(a, blockIdx.x, nullptr);
}

// ── the other memories ───────────────────────────────────────────────────────────────────────────────────────────
// Chunk by chunk F <- A_L F + sum_s c_s (v_s - F k_s) k_s^T with c_s = th_s prod_{r>s} (1-a_r), both products on the
// fp32 matrix cores; a wave owns 16 rows, its lane (ml, kg) row ml, columns 16 kt + 4 kg + v, which serves as operand
// and as result.  The next chunk's k, v, gates are requested before the products of the current one.
// A workgroup takes N of the four memories, the first of them number `first`.  done, mine: the chain's chunks as they come, and
// the snapshots that this workgroup has written (selfref_forward_kernel); a chunk is then requested when it is there.
template <int D>
constexpr int scan_lds_floats(bool waits) { return (waits ? 1 : 2) * (2 * kLrC * (D + 4) + kLrC + 4); }
template <int D, bool SG, int N, bool WAITS>
__device__ __forceinline__ void scan_of(const SelfrefForward &a, size_t b, int first, float *lds, const unsigned *done, unsigned *mine) {
    constexpr int KT = D / 16, ST = kLrC / 16, DD = D * D, NT = 4 * D, LD = D + 4, V4 = D / 4;
    constexpr int LOADS = kLrC * V4 / NT;  // 4 at every D
    constexpr int SET = scan_lds_floats<D>(true);
    const float *const k_cache = a.k, *const v_cache = a.v, *const alpha_cache = a.alpha, *const theta_cache = a.theta;
    const int s = a.s, C = a.C, nc = a.nc;
    const int tid = threadIdx.x, wave = tid >> 6, lane = tid & 63, wr = 16 * wave, ml = lane & 15, kg = lane >> 4;
    const size_t tok0 = b * (size_t)s, at = (size_t)(wr + ml) * D + 4 * kg;
    float *mb = a.mems + (b * 6 + 2 + first) * DD + at;
    f32x4 F[N][KT];
#pragma unroll
    for (int m = 0; m < N; m++) {
#pragma unroll
        for (int kt = 0; kt < KT; kt++) F[m][kt] = *reinterpret_cast<const f32x4 *>(mb + m * DD + 16 * kt);
    }

    float4 nk[LOADS], nv[LOADS];
    float nal = 0.f, nth = 0.f;
    auto request = [&](int ci) {
        const int t0 = ci * C, L = min(C, s - t0);
#pragma unroll
        for (int i = 0; i < LOADS; i++) {
            const int e = tid + i * NT, li = e / V4, j = (e % V4) * 4;
            const size_t o = (tok0 + t0 + li) * D + j;
            nk[i] = li < L ? *reinterpret_cast<const float4 *>(k_cache + o) : make_float4(0, 0, 0, 0);
            nv[i] = li < L ? *reinterpret_cast<const float4 *>(v_cache + o) : make_float4(0, 0, 0, 0);
        }
        if (wave == 0) {
            nal = lane < L ? alpha_cache[tok0 + t0 + lane] : 0.f;
            nth = lane < L ? theta_cache[tok0 + t0 + lane] : 0.f;
        }
    };
    auto stage = [&](float *Ks) {   // k and v (self-generated values: k - v), the products, the chunk's retention
        float *Us = Ks + kLrC * LD, *cs = Us + kLrC * LD;
#pragma unroll
        for (int i = 0; i < LOADS; i++) {
            const int e = tid + i * NT, li = e / V4, j = (e % V4) * 4;
            *reinterpret_cast<float4 *>(&Ks[li * LD + j]) = nk[i];
            *reinterpret_cast<float4 *>(&Us[li * LD + j]) =
                SG ? make_float4(nk[i].x - nv[i].x, nk[i].y - nv[i].y, nk[i].z - nv[i].z, nk[i].w - nv[i].w) : nv[i];
        }
        if (wave == 0) {  // products of the retentions behind each token
            float x = 1.f - nal;
#pragma unroll
            for (int off = 1; off < 64; off *= 2) {
                const float y = __shfl_down(x, off, 64);
                if (lane + off < 64) x *= y;
            }
            const float behind = __shfl_down(x, 1, 64);
            cs[lane] = nth * (lane < 63 ? behind : 1.f);
            if (lane == 0) cs[kLrC] = x;
        }
    };
    auto snapshot = [&](int ci) {
        float *fb = a.frozen + ((b * nc + ci) * 6 + 2 + first) * (size_t)DD + at;
#pragma unroll
        for (int m = 0; m < N; m++) {
#pragma unroll
            for (int kt = 0; kt < KT; kt++) *reinterpret_cast<f32x4 *>(fb + m * DD + 16 * kt) = F[m][kt];
        }
    };
    if (!WAITS) {
        request(0);
        stage(lds);
        __syncthreads();
    }
    for (int ci = 0; ci < nc; ci++) {
        const int L = min(C, s - ci * C);
        float *const K = lds + (WAITS ? 0 : ci & 1) * SET, *const U = K + kLrC * LD, *const cs = U + kLrC * LD;
        snapshot(ci);
        if (WAITS) {
            stores_arrived();
            wait_told(done, 1, ci + 1);   // everybody's snapshot has arrived
            if (wave == 0) tell(mine, ci + 1);
            request(ci);
            stage(K);
            __syncthreads();
        } else if (ci + 1 < nc) {
            request(ci + 1);
        }
        const float keep = cs[kLrC];
        // Tiles behind the chunk's last token hold zeros.  Operands are read one step ahead: left to the compiler, every
        // read stands right before its use.  M memories at a time, so that their sums fit the registers.
        constexpr int M = N > 2 ? 2 : N;
#pragma unroll
        for (int m0 = 0; m0 < N; m0 += M) {
            f32x4 w[M][ST], S[M][KT], x[2][ST];
            auto read_w = [&](int kt, int p) __attribute__((always_inline)) {
#pragma unroll
                for (int st = 0; st < ST; st++)
                    x[p][st] = *reinterpret_cast<const f32x4 *>((SG ? U : K) + (16 * st + ml) * LD + 16 * kt + 4 * kg);
            };
            float kb[2][KT];
            auto read_n = [&](int i, int p) __attribute__((always_inline)) {
#pragma unroll
                for (int kt = 0; kt < KT; kt++) kb[p][kt] = K[(16 * (i >> 2) + 4 * kg + (i & 3)) * LD + 16 * kt + ml];
            };
            read_w(0, 0);
#pragma unroll
            for (int m = 0; m < M; m++) {
#pragma unroll
                for (int st = 0; st < ST; st++) w[m][st] = f32x4{0.f, 0.f, 0.f, 0.f};
            }
#pragma unroll
            for (int kt = 0; kt < KT; kt++) {
                if (kt + 1 < KT) read_w(kt + 1, (kt + 1) & 1);
                else read_n(0, 0);
                __builtin_amdgcn_sched_barrier(0);
#pragma unroll
                for (int v = 0; v < 4; v++) {
#pragma unroll
                    for (int m = 0; m < M; m++) {
#pragma unroll
                        for (int st = 0; st < ST; st++) w[m][st] = mfma4(x[kt & 1][st][v], F[m0 + m][kt][v], w[m][st]);
                    }
                }
                __builtin_amdgcn_sched_barrier(0);
            }
#pragma unroll
            for (int m = 0; m < M; m++) {
#pragma unroll
                for (int kt = 0; kt < KT; kt++) S[m][kt] = f32x4{0.f, 0.f, 0.f, 0.f};   // the chunk's sum by itself: F rounds once a chunk
            }
#pragma unroll
            for (int st = 0; st < ST; st++) {
#pragma unroll
                for (int v = 0; v < 4; v++) {
                    const int t = 16 * st + 4 * kg + v;
#pragma unroll
                    for (int m = 0; m < M; m++) w[m][st][v] = cs[t] * ((SG ? 0.f : U[t * LD + wr + ml]) - w[m][st][v]);
                }
            }
#pragma unroll
            for (int i = 0; i < 4 * ST; i++) {
                if (16 * (i >> 2) >= L) break;
                if (i + 1 < 4 * ST) read_n(i + 1, (i + 1) & 1);
                __builtin_amdgcn_sched_barrier(0);
#pragma unroll
                for (int m = 0; m < M; m++) {
#pragma unroll
                    for (int kt = 0; kt < KT; kt++) S[m][kt] = mfma4(kb[i & 1][kt], w[m][i >> 2][i & 3], S[m][kt]);
                }
                __builtin_amdgcn_sched_barrier(0);
            }
#pragma unroll
            for (int m = 0; m < M; m++) {
#pragma unroll
                for (int kt = 0; kt < KT; kt++) {
#pragma unroll
                    for (int v = 0; v < 4; v++) F[m0 + m][kt][v] = fmaf(keep, F[m0 + m][kt][v], S[m][kt][v]);
                }
            }
        }
        if (!WAITS && ci + 1 < nc) stage(lds + ((ci + 1) & 1) * SET);
        __syncthreads();
    }
#pragma unroll
    for (int m = 0; m < N; m++) {
#pragma unroll
        for (int kt = 0; kt < KT; kt++) *reinterpret_cast<f32x4 *>(mb + m * DD + 16 * kt) = F[m][kt];
    }
}
template <int D, bool SG>
__global__ __launch_bounds__(4 * D) void selfref_scan_kernel(SelfrefForward a) {
    __shared__ __align__(16) float lds[scan_lds_floats<D>(false)];
    // the four memories of a chain share an XCD's L2
    scan_of<D, SG, 1, false>(a, blockIdx.x % a.batch, blockIdx.x / a.batch, lds, nullptr, nullptr);
}

// ── reads ────────────────────────────────────────────────────────────────────────────────────────────────────────
// q_t = F_q (G_t x_t) + H_t x_t, y_t = F_mem (G_t q_t) + H_t q_t with the shared factors in their explicit form
// (selfref_chunk.h).  A wave takes 16 tokens through both reads by itself: the scores with the earlier keys, masked and
// scaled, are the operand of G and H at once; its rows change layout through its own 16 rows of LDS without a barrier.
// 116 us for 2048 chunks of 64 at head size 64, two workgroups per compute unit; 40 are matrix instructions, the rest the
// tables at a chunk's start and the four waves' unequal numbers of earlier tokens.
template <int D>
constexpr int read_lds_floats() { return chunk_lds_floats<D>(0) + D / 16 * kTB * kWL; }
template <int D, bool SG>
__device__ __forceinline__ void read_of(const SelfrefForward &a, size_t b, int ci, float *chunk_lds) {
    const float *const emb = a.emb, *const frozen = a.frozen;
    float *const q_cache = a.q, *const y = a.y;
    const int s = a.s, C = a.C, nc = a.nc;
    constexpr int KT = D / 16, NW = D / 16, DD = D * D, KL = D + 4;
    const ChunkLds<D> m(chunk_lds);
    int tid = threadIdx.x;   // an opaque copy: addresses made of it are not to live across the chunks of a workgroup
    asm volatile("" : "+v"(tid));
    const int wave = tid >> 6, lane = tid & 63, ml = lane & 15, kg = lane >> 4;
    float *row = m.tiles + wave * kTB * kWL;  // the wave's rows
    const size_t chunk = b * nc + ci, tok0 = b * (size_t)s;
    const int t0 = ci * C, L = min(C, s - t0);
    chunk_setup<D, SG>(m, a.k, a.v, a.alpha, a.theta, tok0, t0, L, tid);
    const float *UC = SG ? m.XC : m.KC;

    for (int tile = wave; tile * kTB < L; tile += NW) {
        const int li0 = tile * kTB, nt = min(kTB, L - li0);
        const size_t o0 = (tok0 + t0 + li0) * D;
        f32x4 op[KT], in[KT];  // the read's argument: as operand, and row 4 kg + v, column 16 jt + ml
#pragma unroll
        for (int kt = 0; kt < KT; kt++) {
            op[kt] = ml < nt ? *reinterpret_cast<const f32x4 *>(emb + o0 + (size_t)ml * D + 16 * kt + 4 * kg)
                            : f32x4{0.f, 0.f, 0.f, 0.f};
            *reinterpret_cast<f32x4 *>(row + ml * kWL + 16 * kt + 4 * kg) = op[kt];
        }
        __builtin_amdgcn_wave_barrier();
#pragma unroll
        for (int jt = 0; jt < KT; jt++) {
#pragma unroll
            for (int v = 0; v < 4; v++) in[jt][v] = row[(4 * kg + v) * kWL + 16 * jt + ml];
        }
#pragma unroll
        for (int pass = 0; pass < 2; pass++) {
            const float *Fp = frozen + (chunk * 6 + (pass ? 5 : 2)) * DD;
            __builtin_amdgcn_wave_barrier();
            for (int st = 0; st <= tile; st++) {
                f32x4 acc = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
                for (int kt = 0; kt < KT; kt++) {
                    const f32x4 kk = *reinterpret_cast<const f32x4 *>(m.KC + (16 * st + ml) * KL + 16 * kt + 4 * kg);
#pragma unroll
                    for (int v = 0; v < 4; v++) acc = mfma4(op[kt][v], kk[v], acc);
                }
#pragma unroll
                for (int v = 0; v < 4; v++) {
                    const int tt = 4 * kg + v, li = li0 + tt, s1 = 16 * st + ml;
                    row[tt * kWL + s1] = (tt < nt && s1 < li) ? m.CT[li * kLrC + s1] * acc[v] : 0.f;
                }
            }
            __builtin_amdgcn_wave_barrier();
            f32x4 g[KT], h[KT];
#pragma unroll
            for (int jt = 0; jt < KT; jt++) g[jt] = h[jt] = f32x4{0.f, 0.f, 0.f, 0.f};
            for (int st = 0; st <= tile; st++) {
                const f32x4 w = *reinterpret_cast<const f32x4 *>(row + ml * kWL + 16 * st + 4 * kg);
#pragma unroll
                for (int v = 0; v < 4; v++) {
#pragma unroll
                    for (int jt = 0; jt < KT; jt++) {
                        const int o = (16 * st + 4 * kg + v) * KL + 16 * jt + ml;
                        g[jt] = mfma4(w[v], UC[o], g[jt]);
                        if (!SG) h[jt] = mfma4(w[v], m.XC[o], h[jt]);
                    }
                }
            }
            __builtin_amdgcn_wave_barrier();
#pragma unroll
            for (int jt = 0; jt < KT; jt++) {
#pragma unroll
                for (int v = 0; v < 4; v++) {
                    const int tt = 4 * kg + v;
                    row[tt * kWL + 16 * jt + ml] = tt < nt ? fmaf(m.cA[li0 + tt], in[jt][v], -g[jt][v]) : 0.f;
                }
            }
            __builtin_amdgcn_wave_barrier();
#pragma unroll
            for (int kt = 0; kt < KT; kt++) op[kt] = *reinterpret_cast<const f32x4 *>(row + ml * kWL + 16 * kt + 4 * kg);
            f32x4 f[2][KT];  // the next 16 rows of the snapshot are requested before the products of the current ones
            auto request = [&](int jt, int w) __attribute__((always_inline)) {
#pragma unroll
                for (int kt = 0; kt < KT; kt++)
                    f[w][kt] = *reinterpret_cast<const f32x4 *>(Fp + (16 * jt + ml) * D + 16 * kt + 4 * kg);
            };
            request(0, 0);
#pragma unroll
            for (int jt = 0; jt < KT; jt++) {
                if (jt + 1 < KT) request(jt + 1, (jt + 1) & 1);
                __builtin_amdgcn_sched_barrier(0);
#pragma unroll
                for (int kt = 0; kt < KT; kt++) {
#pragma unroll
                    for (int v = 0; v < 4; v++) h[jt] = mfma4(op[kt][v], f[jt & 1][kt][v], h[jt]);
                }
                float *dst = pass ? y : q_cache;
#pragma unroll
                for (int v = 0; v < 4; v++) {
                    in[jt][v] = h[jt][v];
                    if (4 * kg + v < nt) dst[o0 + (size_t)(4 * kg + v) * D + 16 * jt + ml] = h[jt][v];
                }
            }
            if (pass == 0) {  // q becomes the second read's argument
                __builtin_amdgcn_wave_barrier();
#pragma unroll
                for (int jt = 0; jt < KT; jt++) {
#pragma unroll
                    for (int v = 0; v < 4; v++) row[(4 * kg + v) * kWL + 16 * jt + ml] = in[jt][v];
                }
                __builtin_amdgcn_wave_barrier();
#pragma unroll
                for (int kt = 0; kt < KT; kt++)
                    op[kt] = *reinterpret_cast<const f32x4 *>(row + ml * kWL + 16 * kt + 4 * kg);
            }
        }
        __builtin_amdgcn_wave_barrier();
    }
}

template <int D, bool SG>
__global__ __launch_bounds__(4 * D) void selfref_read_kernel(SelfrefForward a) {
    extern __shared__ __align__(16) float lds[];
    read_of<D, SG>(a, blockIdx.x / a.nc, blockIdx.x % a.nc, lds);
}

// ── all three at once ────────────────────────────────────────────────────────────────────────────────────────────
// The chains leave most of the compute units idle and are followed by nothing but what hangs off their finished chunks.  So one
// launch has workgroups for the chains, for the other memories of each chain, which follow it chunk by chunk, and for the reads, which
// take the chunks in the order in which they are finished.  A workgroup waits only for those that started before it: what it does
// follows from the number it draws when it starts, chains first, and a chain waits for nobody, so every wait ends whatever part of
// the grid is resident.  The LDS keeps a chain's compute unit to itself.
// 64 chains of 2048 tokens, head size 64, chunks of 64: 0.98 ms; the chains by themselves 0.92, telling of their chunks 0.01, their
// company 0.03, and what follows the last chunk 0.02 (the three launches: 0.91 + 0.11 + 0.12).
template <int D, bool SG, int N>
__global__ __launch_bounds__(4 * D + 64) void selfref_forward_kernel(SelfrefForward a, unsigned *counters) {
    extern __shared__ __align__(16) float lds[];
    const int role = draw(counters);
    constexpr int PARTS = 4 / N;   // workgroups for a chain's other memories; its counters: the chain's own, then theirs
    auto counters_of = [&](size_t b) { return counters + (2 + b * (1 + PARTS)) * kTellStride; };
    if (role < a.batch) {
        chain_of<D, SG, true>(a, role, counters_of(role));
        return;
    }
    if (threadIdx.x >= 4 * D) return;
    const int followers = a.batch * (1 + PARTS);
    if (role < followers) {
        const size_t b = role % a.batch;
        const int part = role / a.batch - 1;
        scan_of<D, SG, N, true>(a, b, part * N, lds, counters_of(b), counters_of(b) + (1 + part) * kTellStride);
        return;
    }
    for (int task = draw(counters + kTellStride); task < a.batch * a.nc; task = draw(counters + kTellStride)) {
        const int ci = task / a.batch;
        const size_t b = task % a.batch;
        wait_told(counters_of(b), 1 + PARTS, ci + 1);
        read_of<D, SG>(a, b, ci, lds);
        __syncthreads();   // the chunk's LDS is free
    }
}
template <int D, bool SG, int N>
bool launch_together(const SelfrefForward &a) {
    const int n = (2 + (1 + 4 / N) * a.batch) * kTellStride, followers = (1 + 4 / N) * a.batch;
    const Counters counters(42, n);
    if (!counters.at) return false;
    constexpr int most = scan_lds_floats<D>(true) > read_lds_floats<D>() ? scan_lds_floats<D>(true) : read_lds_floats<D>();
    constexpr size_t lds = (most > kAloneFloats ? most : kAloneFloats) * sizeof(float);
    const long long tasks = (long long)a.batch * a.nc, rest = compute_units() - followers;
    const int readers = (int)(tasks < rest ? tasks : rest);
    check_hip(hipFuncSetAttribute(reinterpret_cast<const void *>(selfref_forward_kernel<D, SG, N>),
                                  hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds), "dynamic LDS size");
    KernelTimer kt("selfref_forward_kernel");
    hipLaunchKernelGGL((selfref_forward_kernel<D, SG, N>), dim3(followers + readers), dim3(4 * D + 64), lds, counters.on, a,
                       counters.at);
    check_launch("selfref_forward_kernel");
    return true;
}

// Together where compute units stay idle beside the chains and those that follow them keep up with them: the other memories
// take 10 us a chunk of any length, a chain 7 us for 16 tokens.  64 chains of 512 tokens, head size 64, apart / together:
// chunks of 8 0.57 / 0.73 ms, of 16 0.38 / 0.41, of 32 0.327 / 0.308, of 64 0.299 / 0.279.  Behind a short sequence follow the reads of
// its chunks on what the chains and their company leave of the chip, so the sequence has to be long enough; up to 8 chains every chunk
// has a workgroup of its own.  Times as fast together, with self-generated values (without them at or above these), chains x tokens:
//   head size 64, chunks of 32 / 64: 9 x 400 1.07 / 1.04, 33 x 400 0.99 / 1.01, 64 x 400 1.02 / 1.00, 64 x 2048 1.19 / 1.12;
//     4 x 65 1.04 / 1.06, 8 x 65 0.99 / 1.02, 8 x 100 0.99 / 1.05
//   32: 33 x 500 0.99 / 1.05, 64 x 500 0.98 / 1.01, 33 x 600 1.04 / 1.05, 64 x 600 1.04 / 1.03, 64 x 2048 1.13 / 1.11;
//     4 x 65 0.97 / 1.04, 8 x 100 0.96 / 1.04, 8 x 200 1.01 / 1.04
//   16: 32 x 500 1.02 / 1.01, 64 x 500 0.95 / 0.98, 33 x 600 1.03 / 1.02, 64 x 600 1.03 / 1.01, 64 x 2048 1.11 / 1.06;
//     4 x 65 1.04 / 1.02, 8 x 65 1.03 / 1.01
// On another stream than the null stream the counters' event adds 5 us: 4 x 100 0.96 / 1.01 there, 24 x 400 1.01 / 1.00, 64 x 600
// 1.10 / 1.08 (head size 64).
template <int D>
bool together_pays(const SelfrefForward &a) {
    if (a.nc < 2 || a.C < 2 * kTB || 4 * a.batch > compute_units()) return false;
    if (a.s >= 600) return true;
    if (stream()) return false;
    if (a.batch > 8) return D == 64 && a.s >= 400;
    return a.C >= 3 * kTB || a.s >= 200 || a.batch <= (D == 64 ? 4 : D == 32 ? 0 : 8);
}

template <int D, bool SG>
void launch(const SelfrefForward &a) {
    // One workgroup for a chain's other memories, as many as there are leave the more of the chip to the reads, or two where that is
    // most of it anyway: head size 64, two / one: 16 chains of 2048 tokens 958 / 960 us, 32 of 500 in chunks of 32 289 / 297, 64 of
    // 2048 1009 / 983; four, 16 of 2048 970.  At smaller head sizes one keeps up: 32, 16 of 2048 654 / 649 us; 16, 578 / 571.
    const bool two = D == 64 && 8 * a.batch <= compute_units();
    if (together_pays<D>(a) && (two ? launch_together<D, SG, D == 64 ? 2 : 4>(a) : launch_together<D, SG, 4>(a))) return;
    const dim3 block(4 * D);
    {
        KernelTimer kt("selfref_chain_kernel");
        hipLaunchKernelGGL((selfref_chain_kernel<D, SG>), dim3(a.batch), dim3(4 * D + 64), 0, stream(), a);
    }
    check_launch("selfref_chain_kernel");
    hipLaunchKernelGGL((selfref_scan_kernel<D, SG>), dim3(4 * a.batch), block, 0, stream(), a);
    check_launch("selfref_scan_kernel");
    const size_t lds = read_lds_floats<D>() * sizeof(float);
    check_hip(hipFuncSetAttribute(reinterpret_cast<const void *>(selfref_read_kernel<D, SG>),
                                  hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds), "dynamic LDS size");
    hipLaunchKernelGGL((selfref_read_kernel<D, SG>), dim3(a.batch * a.nc), block, lds, stream(), a);
    check_launch("selfref_read_kernel");
}

}  // namespace

void selfref_forward_chain(const SelfrefForward &a) {
    if (a.d == 16) a.sg ? launch<16, true>(a) : launch<16, false>(a);
    else if (a.d == 32) a.sg ? launch<32, true>(a) : launch<32, false>(a);
    else a.sg ? launch<64, true>(a) : launch<64, false>(a);
}

}  // namespace nlh
