// HOPE self-referential memory with self-generated values: the backward for chunks of up to 64 tokens.
//
// Inside a chunk (G, dG as in selfref.hip; W_t = dG_{t+1} k_t, Z_t = dG_{t+1}^T u_t, u = k - v)
//     dk_t = -th_t (Z_t + W_t),  dv_t = th_t W_t,  dth_t = -u_t . W_t,
//     dg_t = F_k^T dk_t + F_v^T dv_t + F_q^T dq_t + de_t csE + da_t csA,   dG_t = (1-a_t) dG_{t+1} + dg_t x_t^T + dp_t q_t^T.
// The part of dG that dp q^T drives depends on nothing the sweep produces, so its W, Z, and with them a first part of
// dk, dv, dth and dg, come from selfref_bwd_prepare_kernel (one workgroup per chunk, the whole chip), as do the outer
// products of those parts that make up dF.  What is left for selfref_bwd_sweep_kernel (one workgroup per chain) is the
// part that dg x^T and the chunk boundary drive, carried as Y_s = F_k^T Z_s + (F_k - F_v)^T W_s:
//     Y_s <- (1-a_t) Y_s + (F_k^T x_t) (dg_t . u_s) + ((F_k - F_v)^T dg_t) (x_t . k_s)      for the earlier tokens s of a tile
//     dg_s = dg0_s - th_s Y_s + de_s csE + da_s csA
// so that a token takes one exchange (dg_t), one product with a matrix and the dots of dg_t with the tile's u_s.
//
// 64 chains of 2048 tokens, head size 64, chunks of 64: preparation 0.36 ms (one workgroup per compute unit for its LDS;
// 0.10 are matrix instructions), sweep 1.45 ms: 850 clocks a token (115 instructions of one wave per SIMD and the exchange),
// 7 k clocks a tile and 26 k a chunk boundary, most of those matrix instructions.  The sweep that formed w, z, dk, dv and the
// update of dG token by token took 3.16 ms behind 0.23 ms of preparation; without self-generated values it is still the one
// (selfref.hip), since there dh_t comes back as a second vector.
//
// The sweep has two waves for each 16 rows.  The first half does what the tokens wait for, and across a chunk boundary the
// gradients of F_q and F_mem; the second half those of F_k and F_v, at the boundary and from every tile's dk and dv, stores
// dg, and brings the next boundary's matrices into LDS while the first is among the tokens.  One wave a SIMD did all of it
// in 1.60 ms (9.5 k clocks a tile, 34 k a boundary, half of either with the matrix cores idle; 774 a token: the second wave
// costs the tokens some issue slots and the registers beyond 256).
#include <hip/hip_runtime.h>

#include <type_traits>

#include "../../include/nl_hecate_ffi.h"
#include "lane_ops.h"
#include "quad_rows.h"
#include "runtime.h"
#include "selfref_chunk.h"

namespace nlh {
namespace {

constexpr f32x4 kZero = {0.f, 0.f, 0.f, 0.f};

// Sum over the 16 lanes of a DPP row.
__device__ __forceinline__ float row_sum(float x) { return group_allreduce<16>(x); }

// ── what does not depend on the sweep ────────────────────────────────────────────────────────────────────────────
// LDS: the chunk's k and u, the table of retentions, the masked scores of q with the earlier k and of dp with the
// earlier u (negative), dp, and 16 rows of every wave's own for changes of layout.  The first five make room for
// q, then for dk0, dv0, dq, g, p as the operands of the outer products.
template <int D>
struct PrepareLds {
    static constexpr int KL = D + 4, NW = D / 16;
    static constexpr int wq = 0, wd = wq + kLrC * kWL, dp = wd + kLrC * kWL, rows = dp + kLrC * KL,
                         floats = rows + NW * kTB * kWL;
};

template <int D>
__global__ __launch_bounds__(4 * D) void selfref_bwd_prepare_kernel(
    const float *__restrict__ emb, const float *__restrict__ d_y, const float *__restrict__ k_cache,
    const float *__restrict__ v_cache, const float *__restrict__ q_cache, const float *__restrict__ alpha_cache,
    const float *__restrict__ theta_cache, const float *__restrict__ amean_cache,
    const float *__restrict__ emean_cache, const float *__restrict__ frozen, float *__restrict__ gl,
    float *__restrict__ tok, float *__restrict__ outer, float *__restrict__ csv, int s, int C, int nc) {
    constexpr int KT = D / 16, NW = D / 16, NT = 4 * D, DD = D * D, KL = D + 4, V4 = D / 4, TPW = 4 / NW;
    constexpr int TF = sweep_token_floats(D);
    using P = PrepareLds<D>;
    extern __shared__ __align__(16) float lds[];
    const ChunkLds<D> m(lds);
    float *Wq = m.tiles + P::wq, *Wd = m.tiles + P::wd, *DP = m.tiles + P::dp;
    const int tid = threadIdx.x, wave = tid >> 6, lane = tid & 63, ml = lane & 15, kg = lane >> 4, wr = 16 * wave;
    float *row = m.tiles + P::rows + wave * kTB * kWL;
    const int ci = blockIdx.x % nc;
    const size_t b = blockIdx.x / nc, chunk = blockIdx.x, tok0 = b * (size_t)s;
    const int t0 = ci * C, L = min(C, s - t0), ntile = (L + kTB - 1) / kTB;
    const float *fz = frozen + chunk * 6 * DD;

    for (int e = tid; e < 2 * D; e += NT) {  // column sums of F_eta, F_alpha
        const float *src = fz + (size_t)(3 + e / D) * DD + (e % D);
        float a = 0.f;
#pragma unroll
        for (int c = 0; c < D; c++) a += src[c * D];
        csv[chunk * 2 * D + e] = a;
    }
    for (int e = tid; e < L; e += NT) {  // the sweep's scalars of a token
        const size_t i = tok0 + t0 + e;
        const float al = alpha_cache[i], keep = 1.f - al, sa = sr_sigmoid(amean_cache[i]);
        float *o = tok + i * TF + 3 * D + 16;
        o[0] = al;
        o[1] = theta_cache[i];
        // sigmoid' of the mean over d keep (the sweep forms keep <G_t, dG_{t+1}>): a saturated gate has no gradient
        o[2] = keep > 0.f ? sa * (1.f - sa) * (1.f / D) / keep : 0.f;
        o[3] = sr_sigmoid(emean_cache[i]) * (1.f / D);  // softplus' of the mean over d
    }
    f32x4 in[3][TPW][KT];  // x, q, dy of the wave's tokens, requested ahead of the tables
#pragma unroll
    for (int i = 0; i < TPW; i++) {
        const int li = (wave + i * NW) * kTB + ml;
        const size_t o = (tok0 + t0 + min(li, L - 1)) * D + 4 * kg;
#pragma unroll
        for (int kt = 0; kt < KT; kt++) {
            in[0][i][kt] = li < L ? *reinterpret_cast<const f32x4 *>(emb + o + 16 * kt) : kZero;
            in[1][i][kt] = li < L ? *reinterpret_cast<const f32x4 *>(q_cache + o + 16 * kt) : kZero;
            in[2][i][kt] = li < L ? *reinterpret_cast<const f32x4 *>(d_y + o + 16 * kt) : kZero;
        }
    }
    // scores that no token of the chunk has, and rows behind its last token, enter products times zero
    for (int e = tid; e < 2 * kLrC * kWL + kLrC * KL; e += NT) Wq[e] = 0.f;
    chunk_setup<D, true, false>(m, k_cache, v_cache, alpha_cache, theta_cache, tok0, t0, L, tid);
    for (int e = L + tid; e < kLrC; e += NT) m.cth[e] = 0.f;
    __syncthreads();

    // a wave's rows: 16 tokens as operand rows (token ml, dims 16 kt + 4 kg + v) or as results (token 4 kg + v, dim
    // 16 jt + ml)
    auto put = [&](const f32x4(&x)[KT]) {
        __builtin_amdgcn_wave_barrier();
#pragma unroll
        for (int jt = 0; jt < KT; jt++) {
#pragma unroll
            for (int v = 0; v < 4; v++) row[(4 * kg + v) * kWL + 16 * jt + ml] = x[jt][v];
        }
        __builtin_amdgcn_wave_barrier();
    };
    auto as_operand = [&](f32x4(&a)[KT]) {
#pragma unroll
        for (int kt = 0; kt < KT; kt++) a[kt] = *reinterpret_cast<const f32x4 *>(row + ml * kWL + 16 * kt + 4 * kg);
    };

    f32x4 g[TPW][KT], p[TPW][KT], dq[TPW][KT];
#pragma unroll
    for (int i = 0; i < TPW; i++) {
        const int tile = wave + i * NW, li0 = tile * kTB, nt = min(kTB, L - li0), tile_i = i;
#pragma unroll
        for (int jt = 0; jt < KT; jt++) g[i][jt] = p[i][jt] = dq[i][jt] = kZero;
        if (tile >= ntile) continue;
        const size_t tk = tok0 + t0 + li0;
        // out = A x - sum_s th_s c_ts (x_t . L_s) R_s; the scores without th go to sc (negative with NEG)
        auto low_rank = [&](const f32x4(&a)[KT], const float *Lr, const float *R, float *sc, float sign, float *gam,
                            f32x4(&out)[KT]) {
            for (int st = 0; st <= tile; st++) {
                f32x4 acc = kZero;
#pragma unroll
                for (int kt = 0; kt < KT; kt++) {
                    const f32x4 l = *reinterpret_cast<const f32x4 *>(Lr + (16 * st + ml) * KL + 16 * kt + 4 * kg);
#pragma unroll
                    for (int v = 0; v < 4; v++) acc = mfma4(a[kt][v], l[v], acc);
                }
#pragma unroll
                for (int v = 0; v < 4; v++) {
                    const int tt = 4 * kg + v, li = li0 + tt, s1 = 16 * st + ml;
                    const bool on = tt < nt && s1 < li;
                    sc[tt * kWL + s1] = on ? sign * m.CT[li * kLrC + s1] * acc[v] : 0.f;
                    // x_t . k_s of the tile's own tokens, in the order sigma
                    if (gam && st == tile && tt < nt) gam[(size_t)tt * TF + sigma(ml)] = on ? acc[v] : 0.f;
                }
            }
            __builtin_amdgcn_wave_barrier();
            f32x4 acc[KT];
#pragma unroll
            for (int jt = 0; jt < KT; jt++) acc[jt] = kZero;
            for (int st = 0; st <= tile; st++) {
                const f32x4 w = *reinterpret_cast<const f32x4 *>(sc + ml * kWL + 16 * st + 4 * kg);
                const f32x4 th = *reinterpret_cast<const f32x4 *>(m.cth + 16 * st + 4 * kg);
#pragma unroll
                for (int v = 0; v < 4; v++) {
#pragma unroll
                    for (int jt = 0; jt < KT; jt++)
                        acc[jt] = mfma4(sign * w[v] * th[v], R[(16 * st + 4 * kg + v) * KL + 16 * jt + ml], acc[jt]);
                }
            }
#pragma unroll
            for (int jt = 0; jt < KT; jt++) {
#pragma unroll
                for (int v = 0; v < 4; v++) {
                    const int tt = 4 * kg + v;
                    out[jt][v] = tt < nt ? fmaf(m.cA[li0 + tt], out[jt][v], -acc[jt][v]) : 0.f;
                }
            }
            __builtin_amdgcn_wave_barrier();
        };
        auto as_result = [&](const f32x4(&a)[KT], f32x4(&x)[KT]) {
            __builtin_amdgcn_wave_barrier();
#pragma unroll
            for (int kt = 0; kt < KT; kt++) *reinterpret_cast<f32x4 *>(row + ml * kWL + 16 * kt + 4 * kg) = a[kt];
            __builtin_amdgcn_wave_barrier();
#pragma unroll
            for (int jt = 0; jt < KT; jt++) {
#pragma unroll
                for (int v = 0; v < 4; v++) x[jt][v] = row[(4 * kg + v) * kWL + 16 * jt + ml];
            }
            __builtin_amdgcn_wave_barrier();
        };
        f32x4 a[KT];
        float *out = tok + tk * TF;
        as_result(in[0][i], g[i]);  // g = G x
        low_rank(in[0][i], m.KC, m.XC, row, 1.f, out + 3 * D, g[i]);
        as_result(in[1][i], p[i]);  // p = G q
        low_rank(in[1][i], m.KC, m.XC, Wq + li0 * kWL, 1.f, nullptr, p[i]);
        f32x4 dp[KT];  // dp = F_mem^T dy, dq = G^T dp
        {
            float f[2][4 * KT];  // the next 16 columns are requested before the products of the current ones
            auto request = [&](int jt, int w) __attribute__((always_inline)) {
#pragma unroll
                for (int i = 0; i < 4 * KT; i++)
                    f[w][i] = fz[5 * DD + (16 * (i >> 2) + 4 * kg + (i & 3)) * D + 16 * jt + ml];
            };
            request(0, 0);
#pragma unroll
            for (int jt = 0; jt < KT; jt++) {
                dp[jt] = kZero;
                if (jt + 1 < KT) request(jt + 1, (jt + 1) & 1);
                __builtin_amdgcn_sched_barrier(0);
#pragma unroll
                for (int i = 0; i < 4 * KT; i++) dp[jt] = mfma4(in[2][tile_i][i >> 2][i & 3], f[jt & 1][i], dp[jt]);
            }
        }
        float pp[4] = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
        for (int jt = 0; jt < KT; jt++) {
#pragma unroll
            for (int v = 0; v < 4; v++) {
                DP[(li0 + 4 * kg + v) * KL + 16 * jt + ml] = dp[jt][v];
                pp[v] = fmaf(dp[jt][v], p[i][jt][v], pp[v]);
            }
        }
#pragma unroll
        for (int v = 0; v < 4; v++) {
            pp[v] = row_sum(pp[v]);
            if (ml == 0 && 4 * kg + v < nt) out[(size_t)(4 * kg + v) * TF + 3 * D + 21] = pp[v];
        }
        put(dp);
        as_operand(a);
#pragma unroll
        for (int jt = 0; jt < KT; jt++) dq[i][jt] = dp[jt];
        low_rank(a, m.XC, m.KC, Wd + li0 * kWL, -1.f, nullptr, dq[i]);
#pragma unroll
        for (int jt = 0; jt < KT; jt++) {
#pragma unroll
            for (int v = 0; v < 4; v++)
                if (4 * kg + v < nt) out[(size_t)(4 * kg + v) * TF + 16 * jt + ml] = g[i][jt][v];
        }
    }
    if (ci < nc - 1) {  // G_L = A_L I - sum_s c_Ls u_s k_s^T; wave w takes rows 16 w ..
        f32x4 acc[KT];
#pragma unroll
        for (int jt = 0; jt < KT; jt++) acc[jt] = kZero;
        const int kend = (L + 3) & ~3;
        for (int k0 = 0; k0 < kend; k0 += 4) {
            const float au = m.XC[(k0 + kg) * KL + wr + ml] * m.cL[k0 + kg];
#pragma unroll
            for (int jt = 0; jt < KT; jt++) acc[jt] = mfma4(au, m.KC[(k0 + kg) * KL + 16 * jt + ml], acc[jt]);
        }
        const float aL = m.cA[L];
#pragma unroll
        for (int jt = 0; jt < KT; jt++) {
#pragma unroll
            for (int v = 0; v < 4; v++) {
                const int r = wr + 4 * kg + v, c = 16 * jt + ml;
                gl[chunk * DD + r * D + c] = (r == c ? aL : 0.f) - acc[jt][v];
            }
        }
    }
    __syncthreads();
    float *Q = m.KC;
    for (int e = tid; e < L * V4; e += NT) {
        const int li = e / V4, j = (e % V4) * 4;
        *reinterpret_cast<float4 *>(Q + li * KL + j) =
            *reinterpret_cast<const float4 *>(q_cache + (tok0 + t0 + li) * D + j);
    }
    __syncthreads();
    f32x4 dk[TPW][KT], dv[TPW][KT];
#pragma unroll
    for (int i = 0; i < TPW; i++) {
        const int tile = wave + i * NW, li0 = tile * kTB, nt = min(kTB, L - li0), tile_i = i;
#pragma unroll
        for (int jt = 0; jt < KT; jt++) dk[i][jt] = dv[i][jt] = kZero;
        if (tile >= ntile) continue;
        const size_t tk = tok0 + t0 + li0;
        float *out = tok + tk * TF;
        // W_s = sum_t c_ts (q_t . k_s) dp_t, -Z_s = -sum_t c_ts (dp_t . u_s) q_t over the later tokens
        for (int st = tile; st < ntile; st++) {
#pragma unroll
            for (int v = 0; v < 4; v++) {
                const int t = 16 * st + 4 * kg + v;
                const float wq = Wq[t * kWL + li0 + ml], wd = Wd[t * kWL + li0 + ml];
#pragma unroll
                for (int jt = 0; jt < KT; jt++) {
                    dv[i][jt] = mfma4(wq, DP[t * KL + 16 * jt + ml], dv[i][jt]);
                    dk[i][jt] = mfma4(wd, Q[t * KL + 16 * jt + ml], dk[i][jt]);
                }
            }
        }
        float uw[4] = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
        for (int jt = 0; jt < KT; jt++) {
#pragma unroll
            for (int v = 0; v < 4; v++) {
                const int li = li0 + 4 * kg + v;
                uw[v] = fmaf(m.XC[li * KL + 16 * jt + ml], dv[i][jt][v], uw[v]);
                const float th = m.cth[li];
                dk[i][jt][v] = th * (dk[i][jt][v] - dv[i][jt][v]);
                dv[i][jt][v] *= th;
            }
        }
#pragma unroll
        for (int v = 0; v < 4; v++) {
            uw[v] = row_sum(uw[v]);
            if (ml == 0 && 4 * kg + v < nt) out[(size_t)(4 * kg + v) * TF + 3 * D + 20] = -uw[v];
        }
        // dg0 = F_k^T dk + F_v^T dv + F_q^T dq, and F_k^T x
        f32x4 dg[KT], fx[KT], ak[KT], av[KT], aq[KT];
        put(dk[i]);
        as_operand(ak);
        put(dv[i]);
        as_operand(av);
        put(dq[i]);
        as_operand(aq);
        float f[2][3][4 * KT];  // the next 16 columns of F_k, F_v, F_q ahead of the products of the current ones
        auto request = [&](int jt, int w) __attribute__((always_inline)) {
#pragma unroll
            for (int c = 0; c < 3; c++) {
#pragma unroll
                for (int i = 0; i < 4 * KT; i++)
                    f[w][c][i] = fz[c * DD + (16 * (i >> 2) + 4 * kg + (i & 3)) * D + 16 * jt + ml];
            }
        };
        request(0, 0);
#pragma unroll
        for (int jt = 0; jt < KT; jt++) {
            f32x4 dgk[2] = {kZero, kZero}, dgv[2] = {kZero, kZero}, dgq[2] = {kZero, kZero}, fxk[2] = {kZero, kZero};
            if (jt + 1 < KT) request(jt + 1, (jt + 1) & 1);
            __builtin_amdgcn_sched_barrier(0);
#pragma unroll
            for (int i = 0; i < 4 * KT; i++) {
                const int h = i >= 2 * KT;
                dgk[h] = mfma4(ak[i >> 2][i & 3], f[jt & 1][0][i], dgk[h]);
                fxk[h] = mfma4(in[0][tile_i][i >> 2][i & 3], f[jt & 1][0][i], fxk[h]);
                dgv[h] = mfma4(av[i >> 2][i & 3], f[jt & 1][1][i], dgv[h]);
                dgq[h] = mfma4(aq[i >> 2][i & 3], f[jt & 1][2][i], dgq[h]);
            }
            dg[jt] = ((dgk[0] + dgk[1]) + (dgv[0] + dgv[1])) + (dgq[0] + dgq[1]);
            fx[jt] = fxk[0] + fxk[1];
#pragma unroll
            for (int v = 0; v < 4; v++) {
                if (4 * kg + v < nt) {
                    float *o = out + (size_t)(4 * kg + v) * TF + 16 * jt + ml;
                    o[D] = dg[jt][v];
                    o[2 * D] = fx[jt][v];
                }
            }
        }
    }
    // outer products: dF_k, dF_v, dF_q with g, dF_mem with p; stored as the sweep's lanes hold them
    float dy[kLrC / 4];
#pragma unroll
    for (int i = 0; i < kLrC / 4; i++) {
        const int li = 16 * (i >> 2) + 4 * kg + (i & 3);
        dy[i] = li < L ? d_y[(tok0 + t0 + li) * D + wr + ml] : 0.f;
    }
    __syncthreads();
    float *Es = lds;  // dk, dv, dq, g, p: rows of stride KL, in front of the waves' own rows
#pragma unroll
    for (int i = 0; i < TPW; i++) {
        const int li0 = (wave + i * NW) * kTB;
#pragma unroll
        for (int jt = 0; jt < KT; jt++) {
#pragma unroll
            for (int v = 0; v < 4; v++) {
                float *e = Es + (li0 + 4 * kg + v) * KL + 16 * jt + ml;
                e[0] = dk[i][jt][v];
                e[kLrC * KL] = dv[i][jt][v];
                e[2 * kLrC * KL] = dq[i][jt][v];
                e[3 * kLrC * KL] = g[i][jt][v];
                e[4 * kLrC * KL] = p[i][jt][v];
            }
        }
    }
    __syncthreads();
    f32x4 o[4][KT];
#pragma unroll
    for (int c = 0; c < 4; c++) {
#pragma unroll
        for (int jt = 0; jt < KT; jt++) o[c][jt] = kZero;
    }
#pragma unroll
    for (int st = 0; st < kLrC / 16; st++) {
        if (st >= ntile) break;
#pragma unroll
        for (int v = 0; v < 4; v++) {
            const int li = 16 * st + 4 * kg + v;
            const float *e = Es + li * KL;
            const float ak = e[wr + ml], av = e[kLrC * KL + wr + ml], aq = e[2 * kLrC * KL + wr + ml];
            const float ay = dy[4 * st + v];
#pragma unroll
            for (int jt = 0; jt < KT; jt++) {
                const float bg = e[3 * kLrC * KL + 16 * jt + ml], bp = e[4 * kLrC * KL + 16 * jt + ml];
                o[0][jt] = mfma4(ak, bg, o[0][jt]);
                o[1][jt] = mfma4(av, bg, o[1][jt]);
                o[2][jt] = mfma4(aq, bg, o[2][jt]);
                o[3][jt] = mfma4(ay, bp, o[3][jt]);
            }
        }
    }
#pragma unroll
    for (int c = 0; c < 4; c++) {
#pragma unroll
        for (int jt = 0; jt < KT; jt++)
            *reinterpret_cast<f32x4 *>(outer + (chunk * 4 + c) * DD + ((size_t)(wave * KT + jt) * 64 + lane) * 4) = o[c][jt];
    }
}

// ── the sweep ────────────────────────────────────────────────────────────────────────────────────────────────────
// f(4 J + 3) ... f(4 J) with the argument as a type, if the tile has tokens there
template <int J, class Fn>
__device__ __forceinline__ void four_down(Fn &f, int nt) {
    if (4 * J < nt) {
        f(std::integral_constant<int, 4 * J + 3>{});
        f(std::integral_constant<int, 4 * J + 2>{});
        f(std::integral_constant<int, 4 * J + 1>{});
        f(std::integral_constant<int, 4 * J>{});
    }
}

// acc += m x_I with x spread over the DPP rows: lane i of row kg holds x_i for the row's lanes.  In assembly because the
// compiler moves a broadcast that two products share into a register of its own first.
template <int I>
__device__ __forceinline__ void fmac_spread(float &acc, float x, float m) {
    asm("v_fmac_f32_dpp %0, %1, %2 row_newbcast:%3 row_mask:0xf bank_mask:0xf" : "+v"(acc) : "v"(x), "v"(m), "n"(I));
}
// Two dots with x at once, two chains each.
template <int N, int I = 0>
__device__ __forceinline__ void dots_spread(const float (&m)[N], const float (&n)[N], float x, float (&dm)[2], float (&dn)[2]) {
    if constexpr (I < N) {
        fmac_spread<I>(dm[I & 1], x, m[I]);
        fmac_spread<I>(dn[I & 1], x, n[I]);
        dots_spread<N, I + 1>(m, n, x, dm, dn);
    }
}

// Sums over the four DPP rows of three values at once, every lane receives them.
__device__ __forceinline__ void across_rows3(float &a, float &b, float &c) {
    float a1 = a, b1 = b, c1 = c;
    asm volatile("s_nop 1\n\tv_permlane32_swap_b32 %0, %1\n\tv_permlane32_swap_b32 %2, %3\n\tv_permlane32_swap_b32 %4, %5"
                 : "+v"(a), "+v"(a1), "+v"(b), "+v"(b1), "+v"(c), "+v"(c1));
    a += a1; b += b1; c += c1;
    a1 = a; b1 = b; c1 = c;
    asm volatile("s_nop 1\n\tv_permlane16_swap_b32 %0, %1\n\tv_permlane16_swap_b32 %2, %3\n\tv_permlane16_swap_b32 %4, %5"
                 : "+v"(a), "+v"(a1), "+v"(b), "+v"(b1), "+v"(c), "+v"(c1));
    a += a1; b += b1; c += c1;
}

// dynamic LDS of the sweep: a tile's arrays; G_L^T, two F, dF' of the second half; dF of the first half; dk and dv
constexpr int sweep_tile_floats(int d) { return 8 * kTB * (d + 4); }
constexpr int sweep_lds_floats(int d) { return sweep_tile_floats(d) + 6 * d * (d + 4) + d / 16 * 8 * 64; }

// What a chunk's tokens add to dF whatever the sweep finds: the lane's part of a wave's 16 rows.
template <int D>
__device__ __forceinline__ void token_sums(f32x4 (&sums)[D / 16], const float *outer, int tid) {
    constexpr int JT = D / 16;
#pragma unroll
    for (int jt = 0; jt < JT; jt++)
        sums[jt] = *reinterpret_cast<const f32x4 *>(outer + ((size_t)((tid >> 6) * JT + jt) * 64 + (tid & 63)) * 4);
}

// A wave's 16 rows of a matrix in LDS from its accumulators.
template <int D>
__device__ __forceinline__ void put_rows(float *m, const f32x4 (&x)[D / 16], int tid) {
    const int lane = tid & 63, row = 16 * (tid >> 6) + 4 * (lane >> 4);
#pragma unroll
    for (int jt = 0; jt < D / 16; jt++) {
#pragma unroll
        for (int v = 0; v < 4; v++) m[(row + v) * (D + 4) + 16 * jt + (lane & 15)] = x[jt][v];
    }
}

// F_c of a chunk boundary, a workgroup half's part of each thread.
template <int D>
__device__ __forceinline__ void request_matrix(f32x4 (&m)[D / 16], const float *f, int tid) {
#pragma unroll
    for (int i = 0; i < D / 16; i++) m[i] = *reinterpret_cast<const f32x4 *>(f + (tid + i * 4 * D) * 4);
}
template <int D>
__device__ __forceinline__ void stage_matrix(float *Fs, const f32x4 (&m)[D / 16], int tid) {
#pragma unroll
    for (int i = 0; i < D / 16; i++) {
        const int e = tid + i * 4 * D;
        *reinterpret_cast<f32x4 *>(Fs + (e / (D / 4)) * (D + 4) + (e % (D / 4)) * 4) = m[i];
    }
}

// One memory across a chunk boundary: accG += F_c^T dF'_c, accN = dF'_c G_L^T.
template <int D>
__device__ __forceinline__ void boundary_products(const float *Fs, const float *Bm, const float *GLT, f32x4 (&accG)[D / 16],
                                                  f32x4 (&accN)[D / 16], int tid) {
    constexpr int KT = D / 16, JT = D / 16, LD = D + 4;
    asm volatile("" : "+v"(tid));   // addresses made of it are not to live across the sweep
    const int wave = tid >> 6, lane = tid & 63, ml = lane & 15, kg = lane >> 4, wr = 16 * wave;
#pragma unroll
    for (int jt = 0; jt < JT; jt++) accN[jt] = kZero;
    // contraction in the order 16 c + 4 kg + v: rows 4 apart put the four kg of a read on different banks
#pragma unroll
    for (int c = 0; c < KT; c++) {
        const f32x4 a2 = *reinterpret_cast<const f32x4 *>(Bm + (wr + ml) * LD + 16 * c + 4 * kg);  // dF'_c
#pragma unroll
        for (int v = 0; v < 4; v++) {
            const int k = 16 * c + 4 * kg + v;
            const float a1 = Fs[k * LD + wr + ml];  // F_c^T
#pragma unroll
            for (int jt = 0; jt < JT; jt++) {
                accG[jt] = mfma4(a1, Bm[k * LD + 16 * jt + ml], accG[jt]);
                accN[jt] = mfma4(a2[v], GLT[k * LD + 16 * jt + ml], accN[jt]);
            }
        }
    }
}

// One workgroup per chain, two waves per 16 rows (above).  Lane (ml, kg) = (lane % 16, lane / 16) holds of every matrix row ml of
// the wave's rows, columns CP kg + i (CP = D / 4): operand and result of the tile products (the contraction index runs
// over (i, kg)), and the coefficients of a product with a vector whose element CP kg + i is broadcast from lane i of
// DPP row kg.  dG is kept a second time by columns (dGT).  Tokens of a tile are result rows in the order sigma, so that
// lane kg owns the columns s = 4 v + kg of Y.
template <int D>
__global__ __launch_bounds__(8 * D) void selfref_bwd_sweep_kernel(
    const float *__restrict__ emb, const float *__restrict__ k_cache, const float *__restrict__ v_cache,
    const float *__restrict__ frozen, const float *__restrict__ gl, const float *__restrict__ tok,
    const float *__restrict__ outer, const float *__restrict__ csv, float *__restrict__ d_emb,
    float *__restrict__ d_mems, int s, int C, int nc) {
    constexpr int CP = D / 4, KT = D / 16, JT = D / 16, NT = 4 * D, NW = D / 16, DD = D * D, V4 = D / 4, LD = D + 4;
    constexpr int TF = sweep_token_floats(D), TILE = kTB * LD;
    enum { A_K, A_U, A_X, A_DG0, A_FX, A_DG, A_W, A_Z, A_COUNT };
    static_assert(A_COUNT == 8);
    extern __shared__ __align__(16) float raw[];
    float *const GLT = raw + sweep_tile_floats(D), *const Fa = GLT + D * LD, *const Fb = Fa + D * LD, *const Bm = Fb + D * LD;
    float *const kept = Bm + D * LD;                 // the gradients of F_q and F_mem between the boundaries
    float *const dkv = kept + 2 * D * LD;            // dk, dv of a tile's tokens: [wave][v][2][lane]
    constexpr int LG = D + 16;                       // rows 4 v + kg of g fall on different banks for the four kg
    __shared__ __align__(16) float tg[kTB * LG];     // g
    __shared__ __align__(16) float gam[kTB * kTB];   // x_t . k_s, s in the order sigma
    __shared__ __align__(16) float sc[kTB][8];       // alpha, theta, sigmoid' / (d keep), softplus' / d, dth0, dp . p
    __shared__ __align__(16) float Sx[NW][kTB], Cx[NW][kTB];
    __shared__ __align__(16) float av[2][D];
    __shared__ float sp[NW];
#define T_(a, t, i) raw[(a) * TILE + (t) * LD + (i)]

    const bool second = __builtin_amdgcn_readfirstlane(threadIdx.x) >= NT;
    const int tid = second ? threadIdx.x - NT : threadIdx.x, r = tid >> 2, cq = tid & 3, wave = tid >> 6, lane = tid & 63;
    const int ml = lane & 15, kg = lane >> 4, wr = 16 * wave, c0 = cq * CP;
    const int s_of = sigma(lane & 15), kg_of = lane >> 4;   // as my_s and kg, for masks that stay in scalar registers
    const size_t b = blockIdx.x, tok0 = b * (size_t)s;

    f32x4 accEA = kZero;
    float dG[CP], dGT[CP], sig = 0.f;
    float *dmb = d_mems + b * 6 * DD;
    if (second) {   // the gradients of F_k and F_v, and as many barriers as the first half meets
        f32x4 dFm[2][JT];
        for (int ci = nc - 1; ci >= 0; ci--) {
            const int t0 = ci * C, L = min(C, s - t0), ntile = (L + kTB - 1) / kTB;
            const size_t chunk = b * nc + ci;
            const float *fz = frozen + chunk * 6 * DD;
            int me = tid;
            asm volatile("" : "+v"(me));
            const int wave = me >> 6, lane = me & 63, ml = lane & 15, kg = lane >> 4;
            if (ci < nc - 1) put_rows<D>(Bm, dFm[0], me);
            lds_barrier();
            if (ci < nc - 1) {
                f32x4 accG[JT], accN[JT], sums[2][JT], Fv[JT], Fm[JT];
                request_matrix<D>(Fv, fz + DD, me);
                request_matrix<D>(Fm, fz + 5 * DD, me);
                token_sums<D>(sums[0], outer + chunk * 4 * DD, me);
                token_sums<D>(sums[1], outer + (chunk * 4 + 1) * DD, me);
#pragma unroll
                for (int i = 0; i < JT; i++) accG[i] = kZero;
#pragma unroll
                for (int c = 0; c < 2; c++) {
                    if (c) {
                        stage_matrix<D>(Fa, Fv, me);
                        stage_matrix<D>(Fb, Fm, me);
                        put_rows<D>(Bm, dFm[1], me);
                        lds_barrier();
                    }
                    boundary_products<D>(Fa, Bm, GLT, accG, accN, me);
#pragma unroll
                    for (int jt = 0; jt < JT; jt++) dFm[c][jt] = accN[jt] + sums[c][jt];
                    lds_barrier();   // every wave has read its matrices
                }
                put_rows<D>(Bm, accG, me);
                lds_barrier();   // the first half adds them up
                lds_barrier();
            } else {
                token_sums<D>(dFm[0], outer + chunk * 4 * DD, me);
                token_sums<D>(dFm[1], outer + (chunk * 4 + 1) * DD, me);
            }
            f32x4 Fk[JT], Fq[JT];
            float G[CP];
            // A tile's share of dF, its dg and the next boundary's matrices wait in registers until the other half is among the
            // tokens of the tile after it, which leave the matrix cores alone; a part of them behind each of four barriers, so
            // that no token waits for this half.
            const int stt = me / V4, sj = (me % V4) * 4;
            float op[4][2], gt[4][JT];
            f32x4 dg;
            auto pending = [&](int tile, auto part) {
                constexpr int v = decltype(part)::value;
#pragma unroll
                for (int jt = 0; jt < JT; jt++) {
                    dFm[0][jt] = mfma4(op[v][0], gt[v][jt], dFm[0][jt]);
                    dFm[1][jt] = mfma4(op[v][1], gt[v][jt], dFm[1][jt]);
                }
                if (v == 0 && tile * kTB + stt < L) *reinterpret_cast<f32x4 *>(d_emb + (tok0 + t0 + tile * kTB + stt) * D + sj) = dg;
                if (v == 0 || ci == 0 || tile != ntile - 1) return;
                if (v == 1) stage_matrix<D>(Fa, Fk, me);
                if (v == 2) stage_matrix<D>(Fb, Fq, me);
                if (v == 3) {
#pragma unroll
                    for (int i = 0; i < CP; i++) GLT[((me & 3) * CP + i) * LD + (me >> 2)] = G[i];
                }
            };
            using std::integral_constant;
            for (int tile = ntile - 1; tile >= 0; tile--) {
                const int nt = min(kTB, L - tile * kTB);
                for (int i = 0; i < 4; i++) lds_barrier();   // top, tile staged, W and Z, the first token
                if (tile < ntile - 1) pending(tile + 1, integral_constant<int, 0>{});
                lds_barrier();
                if (tile < ntile - 1) pending(tile + 1, integral_constant<int, 1>{});
                lds_barrier();
                if (tile < ntile - 1) pending(tile + 1, integral_constant<int, 2>{});
                lds_barrier();
                if (tile < ntile - 1) pending(tile + 1, integral_constant<int, 3>{});
                else if (ci > 0) {   // the next boundary's matrices
                    const float *f = fz - 6 * DD;
                    lds_read<CP>(G, gl + (chunk - 1) * DD + (me >> 2) * D + (me & 3) * CP);
                    request_matrix<D>(Fk, f, me);
                    request_matrix<D>(Fq, f + 2 * DD, me);
                }
                for (int i = 3; i < 4 * ((nt + 3) / 4); i++) lds_barrier();   // the other tokens in whole groups of four; dk, dv
#pragma unroll
                for (int v = 0; v < 4; v++) {
                    op[v][0] = dkv[((wave * 4 + v) * 2) * 64 + lane];
                    op[v][1] = dkv[((wave * 4 + v) * 2 + 1) * 64 + lane];
#pragma unroll
                    for (int jt = 0; jt < JT; jt++) gt[v][jt] = tg[(4 * v + kg) * LG + 16 * jt + ml];
                }
                dg = *reinterpret_cast<const f32x4 *>(&T_(A_DG, stt, sj));
            }
            pending(0, integral_constant<int, 0>{});
            pending(0, integral_constant<int, 1>{});
            pending(0, integral_constant<int, 2>{});
            pending(0, integral_constant<int, 3>{});
        }
#pragma unroll
        for (int c = 0; c < 2; c++) {   // gradients of the initial memories
#pragma unroll
            for (int jt = 0; jt < JT; jt++) {
#pragma unroll
                for (int v = 0; v < 4; v++) dmb[(size_t)c * DD + (wr + 4 * kg + v) * D + 16 * jt + ml] = dFm[c][jt][v];
            }
        }
        __syncthreads();
        __syncthreads();
        return;
    }
#pragma unroll
    for (int i = 0; i < CP; i++) dG[i] = dGT[i] = 0.f;
    if (tid < NW * kTB) (&Sx[0][0])[tid] = 0.f;

    float4 pf_k, pf_v, pf_x, pf_g, pf_dg, pf_fx, pf_gam;
    float pf_s[6];
    pf_k = pf_v = pf_x = pf_g = pf_dg = pf_fx = pf_gam = make_float4(0, 0, 0, 0);
#pragma unroll
    for (int i = 0; i < 6; i++) pf_s[i] = 0.f;
    for (int ci = nc - 1; ci >= 0; ci--) {
        const int t0 = ci * C, L = min(C, s - t0), ntile = (L + kTB - 1) / kTB;
        const size_t chunk = b * nc + ci;
        const float *fz = frozen + chunk * 6 * DD;
        // the thread's place through an opaque copy, once per chunk: addresses made of it are not to live across the sweep
        int me = tid;
        asm volatile("" : "+v"(me));
        const int r = me >> 2, cq = me & 3, wave = me >> 6, lane = me & 63, ml = lane & 15, kg = lane >> 4, wr = 16 * wave,
                  c0 = cq * CP, stt = me / V4, sj = (me % V4) * 4;
        // Inputs of a tile, requested one tile ahead; rows behind the chunk's last token are zeros.
        auto request = [&](int first, int nt) {
            const size_t o = (tok0 + first + stt) * D + sj;
            const float *tp = tok + (tok0 + first + stt) * TF;
            auto two = [&](const float *q) {  // rows of tok are 8 bytes aligned
                const float2 lo = *reinterpret_cast<const float2 *>(q), hi = *reinterpret_cast<const float2 *>(q + 2);
                return make_float4(lo.x, lo.y, hi.x, hi.y);
            };
            // branches: a choice of values is one of addresses to the compiler, and so a flat load, which the LDS barriers of
            // the tokens would wait for
            pf_k = pf_v = pf_x = pf_g = pf_dg = pf_fx = make_float4(0, 0, 0, 0);
            if (stt < nt) {
                pf_k = *reinterpret_cast<const float4 *>(k_cache + o);
                pf_v = *reinterpret_cast<const float4 *>(v_cache + o);
                pf_x = *reinterpret_cast<const float4 *>(emb + o);
                pf_g = two(tp + sj);
                pf_dg = two(tp + D + sj);
                pf_fx = two(tp + 2 * D + sj);
            }
            if (tid < 64) {
                pf_gam = make_float4(0, 0, 0, 0);
                if (tid / 4 < nt) pf_gam = two(tok + (tok0 + first + tid / 4) * TF + 3 * D + 4 * (tid % 4));
            }
            if (tid < kTB) {  // zeros behind the last token: it passes everything on as it is
#pragma unroll
                for (int i = 0; i < 6; i++) pf_s[i] = 0.f;
                if (tid < nt) {
                    const float *e = tok + (tok0 + first + tid) * TF + 3 * D + 16;
#pragma unroll
                    for (int i = 0; i < 6; i++) pf_s[i] = e[i];
                }
            }
        };
        float FTk[CP], FTu[CP];   // rows of F_k^T and (F_k - F_v)^T
        // column sums of F_eta, F_alpha
        float csE = csv[chunk * 2 * D + wr + ml], csA = csv[chunk * 2 * D + D + wr + ml];
        // LDS-only barriers from here on: the requests above and the stores of dg stay under way across them
        if (ci < nc - 1 && kg == 0) { av[0][wr + ml] = accEA[0]; av[1][wr + ml] = accEA[1]; }
        lds_barrier();
        sig = 0.f;
        if (ci < nc - 1) {
            // Chunk boundary: gradients of F'_c = F_c G_L flow into dG_L = sum_c F_c^T dF'_c and dF_c = dF'_c G_L^T, on
            // the matrix cores; the rows of dF_eta, dF_alpha are all equal (rank-1 terms of dG_L).
            float q[CP], G[CP];
            const float e = csv[chunk * 2 * D + r], a = csv[chunk * 2 * D + D + r];
            f32x4 accG[JT];
#pragma unroll
            for (int i = 0; i < JT; i++) accG[i] = kZero;
            f32x4 dF[JT], sums[JT];
#pragma unroll
            for (int c = 0; c < 2; c++) {
                if (c) {
                    put_rows<D>(kept, dF, me);
                    lds_barrier();
                }
                token_sums<D>(sums, outer + (chunk * 4 + 2 + c) * DD, me);
#pragma unroll
                for (int i = 0; i < CP; i++) (c ? FTu : FTk)[i] = Fa[(CP * kg + i) * LD + wr + ml];
                boundary_products<D>(Fb, kept + c * D * LD, GLT, accG, dF, me);
#pragma unroll
                for (int jt = 0; jt < JT; jt++) dF[jt] += sums[jt];
                if (c) request(t0 + (ntile - 1) * kTB, L - (ntile - 1) * kTB);
                lds_barrier();  // every wave has read its matrices
            }
            {   // accE <- G_L accE, accA <- G_L accA: rows 0 and 1 of one more product
                f32x4 accV = kZero;
#pragma unroll
                for (int c = 0; c < KT; c++) {
                    const f32x4 a = ml < 2 ? *reinterpret_cast<const f32x4 *>(&av[ml][16 * c + 4 * kg]) : kZero;
#pragma unroll
                    for (int v = 0; v < 4; v++) accV = mfma4(a[v], GLT[(16 * c + 4 * kg + v) * LD + wr + ml], accV);
                }
                accEA = accV;
            }
            put_rows<D>(kept + D * LD, dF, me);
            put_rows<D>(Fb, accG, me);
            {
                float eE[CP], eA[CP];
                lds_read<CP>(eE, &av[0][c0]);
                lds_read<CP>(eA, &av[1][c0]);
#pragma unroll
                for (int i = 0; i < CP; i++) q[i] = e * eE[i] + a * eA[i];
            }
            lds_barrier();  // both halves' sums are there
            float t[CP], h[CP];
            lds_read<CP>(t, Fb + r * LD + c0);
            lds_read<CP>(h, Bm + r * LD + c0);
#pragma unroll
            for (int i = 0; i < CP; i++) t[i] += h[i] + q[i];
            vec_store<CP>(Fb + r * LD + c0, t);
            // sigma_L = <G_L, dG_L>; then (1-a_t) <G_t, dG_{t+1}> = sigma_{t+1} + th_t u.W_t and
            // sigma_t = that + dg.g + dp.p carry the inner product the gradient of alpha needs
#pragma unroll
            for (int i = 0; i < CP; i++) G[i] = GLT[(c0 + i) * LD + r];
            const float part = wave_allreduce(dotn<CP>(G, t));
            if (lane == 0) sp[wave] = part;
            lds_barrier();
#pragma unroll
            for (int w = 0; w < NW; w++) sig += sp[w];
            lds_read<CP>(dG, Fb + (wr + ml) * LD + CP * kg);
#pragma unroll
            for (int i = 0; i < CP; i++) dGT[i] = Fb[(CP * kg + i) * LD + wr + ml];
        } else {
            request(t0 + (ntile - 1) * kTB, L - (ntile - 1) * kTB);
#pragma unroll
            for (int i = 0; i < CP; i++) {
                const float *f = fz + (CP * kg + i) * D + wr + ml;
                FTk[i] = f[0];
                FTu[i] = f[DD];
            }
            f32x4 sums[2][JT];
            token_sums<D>(sums[0], outer + (chunk * 4 + 2) * DD, me);
            token_sums<D>(sums[1], outer + (chunk * 4 + 3) * DD, me);
            put_rows<D>(kept, sums[0], me);
            put_rows<D>(kept + D * LD, sums[1], me);
        }
#pragma unroll
        for (int i = 0; i < CP; i++) FTu[i] = FTk[i] - FTu[i];
        // arrived here: a wait for them inside the tile loop would be one for the next tile's requests as well
        asm volatile("" : "+v"(csE), "+v"(csA));

        for (int tile = ntile - 1; tile >= 0; tile--) {
            const int tb = t0 + tile * kTB, nt = min(kTB, t0 + L - tb);
            int me = tid;   // and once per tile
            asm volatile("" : "+v"(me));
            const int tid = me, wave = tid >> 6, lane = tid & 63, ml = lane & 15, kg = lane >> 4, wr = 16 * wave,
                      stt = tid / V4, sj = (tid % V4) * 4,      // staging slot: token, column
                      ve = CP * kg + ml % CP,                   // the vector element a lane holds
                      tcol = CP * (ml >> 2) + (ml & 3),         // column of result row ml of block 0; block kt: + 4 kt
                      my_s = sigma(ml);                         // token of operand row ml
            lds_barrier();
            *reinterpret_cast<float4 *>(&T_(A_K, stt, sj)) = pf_k;
            *reinterpret_cast<float4 *>(&T_(A_U, stt, sj)) =
                make_float4(pf_k.x - pf_v.x, pf_k.y - pf_v.y, pf_k.z - pf_v.z, pf_k.w - pf_v.w);
            *reinterpret_cast<float4 *>(&T_(A_X, stt, sj)) = pf_x;
            *reinterpret_cast<float4 *>(&tg[stt * LG + sj]) = pf_g;
            *reinterpret_cast<float4 *>(&T_(A_DG0, stt, sj)) = pf_dg;
            *reinterpret_cast<float4 *>(&T_(A_FX, stt, sj)) = pf_fx;
            *reinterpret_cast<float4 *>(&T_(A_DG, stt, sj)) = make_float4(0, 0, 0, 0);
            if (tid < 64) *reinterpret_cast<float4 *>(&gam[4 * tid]) = pf_gam;
            if (tid < kTB) {
                *reinterpret_cast<f32x4 *>(&sc[tid][0]) = f32x4{pf_s[0], pf_s[1], pf_s[2], pf_s[3]};
                *reinterpret_cast<float2 *>(&sc[tid][4]) = make_float2(pf_s[4], pf_s[5]);
            }
            lds_barrier();

            // W = dG K, Z = dG^T U, Y = F_k^T Z + (F_k - F_v)^T W of the whole tile; T_s = u_s . W_s.  A sum per 16 terms,
            // added up in a tree: one running sum rounds at every term (d_x 1.1 to 1.2 times as far from float64)
            constexpr int NQ = CP / 4;
            f32x4 Wq[NQ], Zq[NQ], Yq[NQ], Y2q[NQ];
            float U[CP], T = 0.f;
#pragma unroll
            for (int q = 0; q < NQ; q++) Wq[q] = Zq[q] = Yq[q] = Y2q[q] = kZero;
            auto tree = [](const f32x4(&a)[NQ]) {
                if constexpr (NQ == 4) return (a[0] + a[1]) + (a[2] + a[3]);
                else if constexpr (NQ == 2) return a[0] + a[1];
                else return a[0];
            };
#pragma unroll
            for (int i = 0; i < CP; i += 4) {
                const f32x4 k4 = *reinterpret_cast<const f32x4 *>(&T_(A_K, my_s, CP * kg + i));
                const f32x4 u4 = *reinterpret_cast<const f32x4 *>(&T_(A_U, my_s, CP * kg + i));
#pragma unroll
                for (int v = 0; v < 4; v++) {
                    U[i + v] = u4[v];
                    Wq[i / 4] = mfma4(k4[v], dG[i + v], Wq[i / 4]);
                    Zq[i / 4] = mfma4(u4[v], dGT[i + v], Zq[i / 4]);
                }
            }
            f32x4 W = tree(Wq), Z = tree(Zq);
#pragma unroll
            for (int v = 0; v < 4; v++) {
                T_(A_W, 4 * v + kg, wr + ml) = W[v];
                T_(A_Z, 4 * v + kg, wr + ml) = Z[v];
            }
            lds_barrier();
#pragma unroll
            for (int i = 0; i < CP; i += 4) {
                const f32x4 w4 = *reinterpret_cast<const f32x4 *>(&T_(A_W, my_s, CP * kg + i));
                const f32x4 z4 = *reinterpret_cast<const f32x4 *>(&T_(A_Z, my_s, CP * kg + i));
#pragma unroll
                for (int v = 0; v < 4; v++) {
                    T = fmaf(U[i + v], w4[v], T);
                    Yq[i / 4] = mfma4(z4[v], FTk[i + v], Yq[i / 4]);
                    Y2q[i / 4] = mfma4(w4[v], FTu[i + v], Y2q[i / 4]);
                }
            }
            f32x4 Y = tree(Yq) + tree(Y2q);
            T = swapadd32(T, T);
            T = swapadd16(T, T);
            if (tile > 0) request(tb - kTB, kTB);

            // a_ts = dg_t . u_s for t = 4 j + kg, and prod_{s<r<t} (1-a_r); the same product over the whole tile above s;
            // prod_{r<t} (1-a_r) for t = 4 j + kg
            float at[4], ct[4], et[4], above = 1.f, below[4], keep_tile = 1.f;
#pragma unroll
            for (int j = 0; j < 4; j++) at[j] = ct[j] = et[j] = below[j] = 0.f;
            // groups of four tokens; the first one ends behind the last token at most
            const int first_j = (nt - 1) >> 2;
            float ybc = lane_from(4 * (ml + 48), first_j == 3 ? Y[3] : first_j == 2 ? Y[2] : first_j == 1 ? Y[1] : Y[0]);
            float uw = lane_value(T, sigma(3) + first_j), pkeep = 1.f, pfx = 0.f, pm = 0.f;
            f32x4 pgam = kZero, s0 = *reinterpret_cast<const f32x4 *>(&sc[4 * first_j + 3][0]);
            float2 s1 = *reinterpret_cast<const float2 *>(&sc[4 * first_j + 3][4]);
            float dg0 = T_(A_DG0, 4 * first_j + 3, wr + ml);

            auto step = [&](auto TT) __attribute__((always_inline)) {
                constexpr int t = decltype(TT)::value, J = t / 4, Q = t % 4;
                const float th = s0[1], keep = 1.f - s0[0], sig0 = s1.y;
                const float dth = s1.x - uw, keepalp = fmaf(-th, dth, sig);
                const float da = -keepalp * s0[2], de = dth * s0[3];
                T_(A_DG, t, wr + ml) = fmaf(da, csA, fmaf(de, csE, fmaf(-th, ybc, dg0)));
                lds_barrier();
                const float dgv = T_(A_DG, t, ve), gv = tg[t * LG + ve];
                __builtin_amdgcn_sched_barrier(0);  // first in the queue: the step's chain starts with them
                const f32x4 ps = *reinterpret_cast<const f32x4 *>(&Sx[wave][4 * kg]);
                const float gml = gam[t * kTB + ml], fx = T_(A_FX, t, wr + ml);
                const f32x4 g4 = *reinterpret_cast<const f32x4 *>(&gam[t * kTB + 4 * kg]);
                if constexpr (t > 0) {
                    s0 = *reinterpret_cast<const f32x4 *>(&sc[t - 1][0]);
                    s1 = *reinterpret_cast<const float2 *>(&sc[t - 1][4]);
                    dg0 = T_(A_DG0, t - 1, wr + ml);
                }
                __builtin_amdgcn_sched_barrier(0);  // what follows runs while the reads are under way
                // tables of the tile's end: the retention of token t counts for the pairs around it
                const float km = s_of < t ? keep : 1.f;
                above *= km;
#pragma unroll
                for (int j = J; j < 4; j++) { ct[j] *= km; below[j] *= keep; }
                keep_tile *= keep;
                const bool mine = kg_of == Q;
                below[J] = mine ? 1.f : below[J];
                ct[J] = mine ? (s_of < t ? 1.f : 0.f) : ct[J];
                et[J] = mine ? (ml == 0 ? de : da) : et[J];
                float yold = 0.f;
                if constexpr (t > 0) {
                    constexpr int J1 = (t - 1) / 4, Q1 = (t - 1) % 4;
#pragma unroll
                    for (int v = 0; v <= J1; v++) {
                        Y[v] = fmaf(pm, pgam[v], fmaf(pfx, ps[v], pkeep * Y[v]));
                        asm volatile("" : "+v"(Y[v]));
                    }
                    yold = keep * lane_from(4 * (ml + 16 * Q1), Y[J1]);
                }
                float gg = row_sum((CP == 16 || ml < CP) ? dgv * gv : 0.f);
                float m2[2] = {0.f, 0.f}, a2[2] = {0.f, 0.f};
                // two wait states, should a vector instruction (a copy of the compiler's) have written dgv last
                float spread = dgv;
                asm("s_nop 1" : "+v"(spread));
                dots_spread<CP>(FTu, U, spread, m2, a2);
                float mv = m2[0] + m2[1], a = a2[0] + a2[1];
                across_rows3(mv, a, gg);
                asm volatile("" ::"v"(ps), "v"(g4));  // whole: an element without a use is not to be overwritten early
                sig = keepalp + gg + sig0;
                T = fmaf(a, gml, keep * T);
                if constexpr (t > 0) {
                    constexpr int P1 = sigma(t - 1);
                    const float a1 = lane_value(a, P1), g1 = lane_value(gml, P1);
                    ybc = fmaf(mv, g1, fmaf(fx, a1, yold));
                    uw = lane_value(T, P1);
                    Sx[wave][ml] = a;
                    pkeep = keep; pfx = fx; pm = mv; pgam = g4;
                }
                at[J] = mine ? a : at[J];
            };
            four_down<3>(step, nt);
            four_down<2>(step, nt);
            four_down<1>(step, nt);
            four_down<0>(step, nt);

            // W_s, Z_s at their own tokens: what the tile started with under the retentions above s, plus the tile's own
            // pairs; dk = -th (Z + W), dv = th W are the operands of the outer products as they stand
            Cx[wave][ml] = above;
            __builtin_amdgcn_wave_barrier();
            const f32x4 top = *reinterpret_cast<const f32x4 *>(&Cx[wave][4 * kg]);
            W *= top;
            Z *= top;
#pragma unroll
            for (int j = 0; j < 4; j++) {
                const int t = 4 * j + kg;
                W = mfma4(ct[j] * gam[t * kTB + ml], T_(A_DG, t, wr + ml), W);
                Z = mfma4(ct[j] * at[j], T_(A_X, t, wr + ml), Z);
            }
#pragma unroll
            for (int v = 0; v < 4; v++) {
                const int t = 4 * v + kg;
                const float th = sc[t][1];
                dkv[((wave * 4 + v) * 2) * 64 + lane] = -th * (Z[v] + W[v]);
                dkv[((wave * 4 + v) * 2 + 1) * 64 + lane] = th * W[v];
            }
            lds_barrier();
#pragma unroll
            for (int v = 0; v < 4; v++) accEA = mfma4(ml < 2 ? et[v] : 0.f, tg[(4 * v + kg) * LG + wr + ml], accEA);
            if (tile > 0) {  // the chunk's first tile has no use for its dG: G_0 = I
                f32x4 n[KT], nT[KT];
#pragma unroll
                for (int kt = 0; kt < KT; kt++) {
#pragma unroll
                    for (int v = 0; v < 4; v++) {
                        n[kt][v] = keep_tile * dG[4 * kt + v];
                        nT[kt][v] = keep_tile * dGT[4 * kt + v];
                    }
                }
#pragma unroll
                for (int j = 0; j < 4; j++) {
                    const int t = 4 * j + kg;
                    const float bg = below[j] * T_(A_DG, t, wr + ml), bx = below[j] * T_(A_X, t, wr + ml);
#pragma unroll
                    for (int kt = 0; kt < KT; kt++) {
                        n[kt] = mfma4(T_(A_X, t, tcol + 4 * kt), bg, n[kt]);
                        nT[kt] = mfma4(T_(A_DG, t, tcol + 4 * kt), bx, nT[kt]);
                    }
                }
#pragma unroll
                for (int kt = 0; kt < KT; kt++) {
#pragma unroll
                    for (int v = 0; v < 4; v++) { dG[4 * kt + v] = n[kt][v]; dGT[4 * kt + v] = nT[kt][v]; }
                }
            }
        }
    }
#pragma unroll
    for (int i = 0; i < JT; i++) {   // gradients of the initial memories, rows of every wave's own
        const int row = wr + 16 * i / JT + lane / (4 * JT), at = lane % (4 * JT) * 4;
        *reinterpret_cast<f32x4 *>(dmb + (size_t)2 * DD + row * D + at) = *reinterpret_cast<const f32x4 *>(kept + row * LD + at);
        *reinterpret_cast<f32x4 *>(dmb + (size_t)5 * DD + row * D + at) =
            *reinterpret_cast<const f32x4 *>(kept + (D + row) * LD + at);
    }
    __syncthreads();
    if (kg == 0) { av[0][wr + ml] = accEA[0]; av[1][wr + ml] = accEA[1]; }
    __syncthreads();
    {
        float eE[CP], eA[CP];
        lds_read<CP>(eE, &av[0][c0]);
        lds_read<CP>(eA, &av[1][c0]);
        vec_store<CP>(dmb + 3 * DD + r * D + c0, eE);
        vec_store<CP>(dmb + 4 * DD + r * D + c0, eA);
    }
#undef T_
}

template <int D>
void launch(const SelfrefSweep &a) {
    constexpr size_t lds = (chunk_lds_floats<D>(0) + PrepareLds<D>::floats) * sizeof(float);
    static_assert(5 * kLrC * (D + 4) <= chunk_lds_floats<D>(0) + PrepareLds<D>::rows, "operands of the outer products");
    static_assert(lds <= 160 * 1024, "LDS");
    check_hip(hipFuncSetAttribute(reinterpret_cast<const void *>(selfref_bwd_prepare_kernel<D>),
                                  hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds), "dynamic LDS size");
    hipLaunchKernelGGL((selfref_bwd_prepare_kernel<D>), dim3(a.batch * a.nc), dim3(4 * D), lds, stream(), a.emb, a.d_y, a.k,
                       a.v, a.q, a.alpha, a.theta, a.amean, a.emean, a.frozen, a.gl, a.tok, a.outer, a.csv, a.s, a.C, a.nc);
    check_launch("selfref_bwd_prepare_kernel");
    constexpr size_t sweep_lds = sweep_lds_floats(D) * sizeof(float);
    check_hip(hipFuncSetAttribute(reinterpret_cast<const void *>(selfref_bwd_sweep_kernel<D>),
                                  hipFuncAttributeMaxDynamicSharedMemorySize, (int)sweep_lds), "dynamic LDS size");
    KernelTimer kt("selfref_bwd_kernel");
    hipLaunchKernelGGL((selfref_bwd_sweep_kernel<D>), dim3(a.batch), dim3(8 * D), sweep_lds, stream(), a.emb, a.k, a.v, a.frozen,
                       a.gl, a.tok, a.outer, a.csv, a.d_emb, a.d_mems, a.s, a.C, a.nc);
    check_launch("selfref_bwd_sweep_kernel");
}

}  // namespace

void selfref_backward_sweep(const SelfrefSweep &a) {
    if (a.d == 16) launch<16>(a);
    else if (a.d == 32) launch<32>(a);
    else launch<64>(a);
}

}  // namespace nlh
