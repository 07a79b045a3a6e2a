// HOPE self-referential memory with self-generated values: the backward for chunks of up to 64 tokens.
//
// Inside a chunk (G, dG as in selfref.hip; W_t = dG_{t+1} k_t, Z_t = dG_{t+1}^T u_t, u = k - v)
//     dk_t = -th_t (Z_t + W_t),  dv_t = th_t W_t,  dth_t = -u_t . W_t,
//     dg_t = F_k^T dk_t + F_v^T dv_t + F_q^T dq_t + de_t csE + da_t csA,   dG_t = (1-a_t) dG_{t+1} + dg_t x_t^T + dp_t q_t^T.
// The part of dG that dp q^T drives depends on nothing the sweep produces, so its W, Z, and with them a first part of
// dk, dv, dth and dg, come from selfref_bwd_prepare_kernel (one workgroup per chunk, the whole chip), as do the outer
// products of those parts that make up dF.  The gradients of F_q and F_mem and their share of dG at the boundaries need nothing
// else: selfref_bwd_scan_kernel, selfref_bwd_share_kernel.  What is left for selfref_bwd_sweep_kernel (one workgroup per chain) is the
// part that dg x^T and the chunk boundary drive, carried as Y_s = F_k^T Z_s + (F_k - F_v)^T W_s:
//     Y_s <- (1-a_t) Y_s + (F_k^T x_t) (dg_t . u_s) + ((F_k - F_v)^T dg_t) (x_t . k_s)      for the earlier tokens s of a tile
//     dg_s = dg0_s - th_s Y_s + de_s csE + da_s csA
// so that a token takes one exchange (dg_t), one product with a matrix and the dots of dg_t with the tile's u_s.
//
// 64 chains of 2048 tokens, head size 64, chunks of 64: preparation 0.29 ms (one workgroup per compute unit for its LDS;
// 0.10 are matrix instructions), scan 0.06 and share 0.03, sweep 1.30 ms: 870 clocks a token (115 instructions of one wave per
// SIMD and the exchange), 6.7 k clocks a tile and 15 k a chunk boundary, most of those matrix instructions.  The sweep that formed w, z, dk, dv and the
// update of dG token by token took 3.16 ms behind 0.23 ms of preparation; without self-generated values it is still the one
// (selfref.hip), since there dh_t comes back as a second vector.
//
// The sweep has two waves for each 16 rows.  The first half does what the tokens wait for; the second half the gradients of F_k
// and F_v, from every tile's dk and dv and across the boundaries, stores dg, and brings the next tile's inputs and the next
// boundary's matrices into LDS while the first is among the tokens.  One wave a SIMD did all of it
// in 1.60 ms (9.5 k clocks a tile, 34 k a boundary, half of either with the matrix cores idle; 774 a token: the second wave
// costs the tokens some issue slots and the registers beyond 256).  With F_q and F_mem in the sweep, each half two
// memories at a boundary and the first half its own inputs, it was 1.45 ms (7.7 k a tile, 26 k a boundary).  A matrix instruction of
// the second half keeps the first from issuing for as long: forming dF across the boundary among the tokens hides its
// latencies, not its instructions.
#include <hip/hip_runtime.h>

#include <type_traits>
#include <utility>

#include "../../include/nl_hecate_ffi.h"
#include "handover.h"
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
// LDS: the chunk's k and u, the table of retentions, the masked scores of x and of q with the earlier k and of dp with the
// earlier u (negative), dp, and what the two waves of a tile add up; then q in the place of k, and dk0, dv0, dq, g, p as
// operands in front of the sums.
template <int D>
struct PrepareLds {
    static constexpr int KL = D + 4;
    static constexpr int wx = 0, wq = wx + kLrC * kWL, wd = wq + kLrC * kWL, dp = wd + kLrC * kWL, sums = dp + kLrC * KL,
                         floats = sums + 4 * kLrC;
};
constexpr int kPrepThr = 512;
// N neighbouring columns, one for each of a wave's column tiles
template <int N>
__device__ __forceinline__ void load_columns(float (&x)[N], const float *p) {
    if constexpr (N == 2) {
        const float2 t = *reinterpret_cast<const float2 *>(p);
        x[0] = t.x; x[1] = t.y;
    } else {
        x[0] = p[0];
    }
}
template <int N>
__device__ __forceinline__ void store_columns(float *p, const float (&x)[N]) {
    if constexpr (N == 2) *reinterpret_cast<float2 *>(p) = make_float2(x[0], x[1]);
    else p[0] = x[0];
}

// A workgroup per chunk, eight waves: two for each tile of 16 tokens, which share its scores by tiles of earlier tokens and its
// results by columns, and for each 16 rows of a D x D result, by columns.  Waves w and w + 4 share a SIMD and take tiles w and
// 3 - w, whose numbers of earlier tokens add up to the same.  One workgroup fills a compute unit's LDS, so its own latencies are
// what bounds it: 82 k clocks a chunk, 31 k of them matrix instructions, 19 k until the chunk is in LDS, 19 k where the
// low-rank products wait and F_k, F_v, F_q are on their way.  2048 chunks at head size 64: 293 us; four waves, one for each tile, whose
// column sums of F_eta and F_alpha were 64 loads one after the other, took 363.
template <int D>
__device__ __forceinline__ void prepare_of(const SelfrefSweep &a, size_t b, int ci, float *lds) {
    const float *const emb = a.emb, *const d_y = a.d_y, *const k_cache = a.k, *const v_cache = a.v, *const q_cache = a.q,
                *const alpha_cache = a.alpha, *const theta_cache = a.theta, *const amean_cache = a.amean, *const emean_cache = a.emean,
                *const frozen = a.frozen;
    float *const gl = a.gl, *const tok = a.tok, *const outer = a.outer, *const csv = a.csv, *const d_mems = a.d_mems;
    const int s = a.s, C = a.C, nc = a.nc;
    constexpr int KT = D / 16, DD = D * D, KL = D + 4, V4 = D / 4;
    constexpr int JH = KT > 1 ? KT / 2 : 1, CG = KT / JH;   // a wave's column tiles; groups of columns
    constexpr int TF = sweep_token_floats(D);
    using P = PrepareLds<D>;
    const ChunkLds<D> m(lds);
    float *Wx = m.tiles + P::wx, *Wq = m.tiles + P::wq, *Wd = m.tiles + P::wd, *DP = m.tiles + P::dp, *sums = m.tiles + P::sums;
    int tid = threadIdx.x;   // an opaque copy: addresses made of it are not to live across the chunks of a workgroup
    asm volatile("" : "+v"(tid));
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6), lane = tid & 63, ml = lane & 15, kg = lane >> 4;
    const size_t chunk = b * nc + ci, tok0 = b * (size_t)s;
    const int t0 = ci * C, L = min(C, s - t0), ntile = (L + kTB - 1) / kTB;
    const float *fz = frozen + chunk * 6 * DD;
    const int half = wave >> 2, tile = half ? 7 - wave : wave, li0 = tile * kTB, nt = min(kTB, L - li0);
    const bool live = tile < ntile, columns = live && half < CG;   // tokens there; columns as well
    // Column ml of this wave's column tile j is column JH ml + j of its share: one load serves both tiles.
    const int cw = 16 * JH * (half < CG ? half : 0) + JH * ml;
    const size_t tk = tok0 + t0 + li0;
    float *out = tok + tk * TF;

    // Requested in the order in which they are waited for.  First the chunk's k and v: row e / V4, columns 4 (e % V4) ..
    constexpr int LOADS = kLrC * V4 / kPrepThr > 0 ? kLrC * V4 / kPrepThr : 1;
    f32x4 k4[LOADS], v4[LOADS];
#pragma unroll
    for (int i = 0; i < LOADS; i++) {
        const int e = tid + i * kPrepThr;
        const size_t o = (tok0 + t0 + min(e / V4, L - 1)) * D + (e % V4) * 4;
        k4[i] = *reinterpret_cast<const f32x4 *>(k_cache + o);
        v4[i] = *reinterpret_cast<const f32x4 *>(v_cache + o);
    }
    float al = 0.f, th = 0.f;
    float amean = 0.f, emean = 0.f;
    if (tid < L) {
        const size_t i = tok0 + t0 + tid;
        al = alpha_cache[i]; th = theta_cache[i]; amean = amean_cache[i]; emean = emean_cache[i];
    }
    f32x4 in[3][KT];   // x, q, dy of the tile's tokens as operands
    float xr[2][4][JH];   // x, q as results: token 4 kg + v, column cw + j
    float fm[4 * KT][JH];   // F_mem, this wave's columns
    if (live) {
        const size_t o = (tk + min(ml, nt - 1)) * D + 4 * kg;
#pragma unroll
        for (int kt = 0; kt < KT; kt++) {
            in[0][kt] = *reinterpret_cast<const f32x4 *>(emb + o + 16 * kt);
            in[1][kt] = *reinterpret_cast<const f32x4 *>(q_cache + o + 16 * kt);
            in[2][kt] = *reinterpret_cast<const f32x4 *>(d_y + o + 16 * kt);
        }
#pragma unroll
        for (int i = 0; i < 4 * KT; i++) load_columns(fm[i], fz + 5 * DD + (16 * (i >> 2) + 4 * kg + (i & 3)) * D + cw);
#pragma unroll
        for (int v = 0; v < 4; v++) {
            const size_t e = (tk + min(4 * kg + v, nt - 1)) * D + cw;
            load_columns(xr[0][v], emb + e);
            load_columns(xr[1][v], q_cache + e);
        }
    }
    // column sums of F_eta, F_alpha: a column's share of the rows per thread
    constexpr int PARTS = kPrepThr / (2 * D), ROWS = D / PARTS;
    float cs[ROWS];
    {
        const int e = tid % (2 * D);
        const float *src = fz + (size_t)(3 + e / D) * DD + tid / (2 * D) * ROWS * D + e % D;
#pragma unroll
        for (int c = 0; c < ROWS; c++) cs[c] = src[c * D];
    }
    __builtin_amdgcn_sched_barrier(0);
#pragma unroll
    for (int i = 0; i < LOADS; i++) {   // rows behind a short chunk's last token enter products times zero
        const int e = tid + i * kPrepThr, li = e / V4, j = (e % V4) * 4;
        if (li < kLrC) {
            *reinterpret_cast<f32x4 *>(m.KC + li * KL + j) = li < L ? k4[i] : kZero;
            *reinterpret_cast<f32x4 *>(m.XC + li * KL + j) = li < L ? k4[i] - v4[i] : kZero;
        }
    }
    if (tid < kLrC) { m.cal[tid] = al; m.cth[tid] = th; }
    if (tid < 4 * kLrC) sums[tid] = 0.f;
    lds_barrier();   // of LDS only: the other requests stay under way

    // rows that no token has are zeros in every operand
#pragma unroll
    for (int i = 0; i < 3; i++) {
#pragma unroll
        for (int kt = 0; kt < KT; kt++) in[i][kt] = live && ml < nt ? in[i][kt] : kZero;
    }
    // products of 16 rows with those of the tile's earlier tokens, a tile's two waves in turn; c: which of the wave's
    auto score = [&](const f32x4(&a)[KT], const float *Lr, f32x4(&acc)[2]) {
#pragma unroll
        for (int c = 0; c < 2; c++) {
            acc[c] = kZero;
            const int st = 2 * c + half;
            if (st > tile) continue;
#pragma unroll
            for (int kt = 0; kt < KT; kt++) {
                const f32x4 l = *reinterpret_cast<const f32x4 *>(Lr + (16 * st + ml) * KL + 16 * kt + 4 * kg);
#pragma unroll
                for (int v = 0; v < 4; v++) acc[c] = mfma4(a[kt][v], l[v], acc[c]);
            }
        }
    };
    // masked, with the retentions in between, to W (negative with sign -1); x_t . k_s of the tile's own tokens to gam as well, in
    // the order sigma
    auto put_scores = [&](const f32x4(&acc)[2], float *W, float sign, float *gam) {
#pragma unroll
        for (int c = 0; c < 2; c++) {
            const int st = 2 * c + half;
            if (st > tile) continue;
#pragma unroll
            for (int v = 0; v < 4; v++) {
                const int tt = 4 * kg + v, li = li0 + tt, s1 = 16 * st + ml;
                const bool on = tt < nt && s1 < li;
                W[li * kWL + s1] = on ? sign * m.CT[li * kLrC + s1] * acc[c][v] : 0.f;
                if (gam && st == tile && tt < nt) gam[(size_t)tt * TF + sigma(ml)] = on ? acc[c][v] : 0.f;
            }
        }
    };
    // sum over this wave's columns of a product of two results, to the half's 64 sums
    auto add_up = [&](float (&x)[4], float *to) {
#pragma unroll
        for (int v = 0; v < 4; v++) {
            x[v] = row_sum(x[v]);
            if (ml == 0) to[half * kLrC + li0 + 4 * kg + v] = x[v];
        }
    };

    f32x4 sx[2], sq[2];
    float dp[4][JH];
#pragma unroll
    for (int v = 0; v < 4; v++) {
#pragma unroll
        for (int j = 0; j < JH; j++) dp[v][j] = 0.f;
    }
    if (live) {
        score(in[0], m.KC, sx);
        score(in[1], m.KC, sq);
    }
    if (columns) {   // dp = F_mem^T dy
#pragma unroll
        for (int j = 0; j < JH; j++) {
            f32x4 acc = kZero;
#pragma unroll
            for (int i = 0; i < 4 * KT; i++) acc = mfma4(in[2][i >> 2][i & 3], fm[i][j], acc);
#pragma unroll
            for (int v = 0; v < 4; v++) dp[v][j] = acc[v];
        }
#pragma unroll
        for (int v = 0; v < 4; v++) store_columns(DP + (li0 + 4 * kg + v) * KL + cw, dp[v]);
    }
#pragma unroll
    for (int n = ROWS / 2; n > 0; n /= 2) {
#pragma unroll
        for (int c = 0; c < n; c++) cs[c] += cs[c + n];
    }
    m.Wt[tid] = cs[0];
    if (wave == 7) chunk_tables<D, false>(m, L, lane);   // the wave with the fewest scores
    lds_barrier();
    f32x4 sd[2];
    if (live) {
        put_scores(sx, Wx, 1.f, out + 3 * D);
        put_scores(sq, Wq, 1.f, nullptr);
        f32x4 a[KT];
#pragma unroll
        for (int kt = 0; kt < KT; kt++) a[kt] = *reinterpret_cast<const f32x4 *>(DP + (li0 + ml) * KL + 16 * kt + 4 * kg);
        score(a, m.XC, sd);
        put_scores(sd, Wd, -1.f, nullptr);
    }
    if (tid < 2 * D) {
        float a = 0.f;
#pragma unroll
        for (int i = 0; i < PARTS; i++) a += m.Wt[i * 2 * D + tid];
        csv[chunk * 2 * D + tid] = a;
    }
    lds_barrier();
    // g = G x, p = G q, dq = G^T dp
    if (columns) {   // A x - sum_s th_s c_ts (scores) R_s for this wave's columns, the three side by side
        f32x4 acc[3][JH];
#pragma unroll
        for (int j = 0; j < JH; j++) acc[0][j] = acc[1][j] = acc[2][j] = kZero;
        for (int st = 0; st <= tile; st++) {
            const int at = (li0 + ml) * kWL + 16 * st + 4 * kg;
            const f32x4 wx = *reinterpret_cast<const f32x4 *>(Wx + at), wq = *reinterpret_cast<const f32x4 *>(Wq + at),
                        wd = *reinterpret_cast<const f32x4 *>(Wd + at), th = *reinterpret_cast<const f32x4 *>(m.cth + 16 * st + 4 * kg);
            float u[4][JH], kk[4][JH];
#pragma unroll
            for (int v = 0; v < 4; v++) {
                load_columns(u[v], m.XC + (16 * st + 4 * kg + v) * KL + cw);
                load_columns(kk[v], m.KC + (16 * st + 4 * kg + v) * KL + cw);
            }
            __builtin_amdgcn_sched_barrier(0);   // all reads ahead of the products
#pragma unroll
            for (int v = 0; v < 4; v++) {
#pragma unroll
                for (int j = 0; j < JH; j++) {
                    acc[0][j] = mfma4(wx[v] * th[v], u[v][j], acc[0][j]);
                    acc[1][j] = mfma4(wq[v] * th[v], u[v][j], acc[1][j]);
                    acc[2][j] = mfma4(-wd[v] * th[v], kk[v][j], acc[2][j]);
                }
            }
        }
        float pp[4];
#pragma unroll
        for (int v = 0; v < 4; v++) {
            const int tt = 4 * kg + v;
            const float A = m.cA[li0 + tt];
            pp[v] = 0.f;
#pragma unroll
            for (int j = 0; j < JH; j++) {
                xr[0][v][j] = tt < nt ? fmaf(A, xr[0][v][j], -acc[0][j][v]) : 0.f;
                xr[1][v][j] = tt < nt ? fmaf(A, xr[1][v][j], -acc[1][j][v]) : 0.f;
                pp[v] = fmaf(dp[v][j], xr[1][v][j], pp[v]);
                dp[v][j] = tt < nt ? fmaf(A, dp[v][j], -acc[2][j][v]) : 0.f;   // dq from here on
            }
            if (tt < nt) store_columns(out + (size_t)tt * TF + cw, xr[0][v]);
        }
        add_up(pp, sums);
    }
    const int rb = wave % KT, wr = 16 * rb, c0 = JH * (wave / KT < CG ? wave / KT : 0);   // D x D results: rows, column tiles
    const bool rows = wave < KT * CG;
    if (ci < nc - 1 && rows) {  // G_L = A_L I - sum_s c_Ls u_s k_s^T
        f32x4 acc[JH];
#pragma unroll
        for (int j = 0; j < JH; j++) acc[j] = kZero;
        for (int k0 = 0; k0 < L; k0 += 16) {   // rows behind the last token are zeros
            float au[4], bk[4][JH];
#pragma unroll
            for (int i = 0; i < 4; i++) {
                const int k = k0 + 4 * i + kg;
                au[i] = m.XC[k * KL + wr + ml] * m.cL[k];
#pragma unroll
                for (int j = 0; j < JH; j++) bk[i][j] = m.KC[k * KL + 16 * (c0 + j) + ml];
            }
            __builtin_amdgcn_sched_barrier(0);
#pragma unroll
            for (int i = 0; i < 4; i++) {
#pragma unroll
                for (int j = 0; j < JH; j++) acc[j] = mfma4(au[i], bk[i][j], acc[j]);
            }
        }
        const float aL = m.cA[L];
#pragma unroll
        for (int j = 0; j < JH; j++) {
#pragma unroll
            for (int v = 0; v < 4; v++) {
                const int r = wr + 4 * kg + v, c = 16 * (c0 + j) + ml;
                gl[chunk * DD + r * D + c] = (r == c ? aL : 0.f) - acc[j][v];
            }
        }
    }
    f32x4 q4[LOADS];   // q in the layout of the first loads
#pragma unroll
    for (int i = 0; i < LOADS; i++) {
        const int e = tid + i * kPrepThr;
        q4[i] = *reinterpret_cast<const f32x4 *>(q_cache + (tok0 + t0 + min(e / V4, L - 1)) * D + (e % V4) * 4);
    }
    // F_k, F_v, F_q, this wave's columns, ahead of their products
    float f[3][4 * KT][JH];
    if (columns) {
#pragma unroll
        for (int c = 0; c < 3; c++) {
#pragma unroll
            for (int i = 0; i < 4 * KT; i++) load_columns(f[c][i], fz + c * DD + (16 * (i >> 2) + 4 * kg + (i & 3)) * D + cw);
        }
    }
    lds_barrier();
    float *Q = m.KC;
#pragma unroll
    for (int i = 0; i < LOADS; i++) {
        const int e = tid + i * kPrepThr, li = e / V4, j = (e % V4) * 4;
        if (li < L) *reinterpret_cast<f32x4 *>(Q + li * KL + j) = q4[i];
    }
    lds_barrier();
    f32x4 dk[JH], dv[JH];
#pragma unroll
    for (int j = 0; j < JH; j++) dk[j] = dv[j] = kZero;
    if (columns) {
        // W_s = sum_t c_ts (q_t . k_s) dp_t, -Z_s = -sum_t c_ts (dp_t . u_s) q_t over the later tokens
        for (int st = tile; st < ntile; st++) {
#pragma unroll
            for (int v = 0; v < 4; v++) {
                const int t = 16 * st + 4 * kg + v;
                const float wq = Wq[t * kWL + li0 + ml], wd = Wd[t * kWL + li0 + ml];
                float p[JH], q[JH];
                load_columns(p, DP + t * KL + cw);
                load_columns(q, Q + t * KL + cw);
#pragma unroll
                for (int j = 0; j < JH; j++) {
                    dv[j] = mfma4(wq, p[j], dv[j]);
                    dk[j] = mfma4(wd, q[j], dk[j]);
                }
            }
        }
        float uw[4] = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
        for (int v = 0; v < 4; v++) {
            const int li = li0 + 4 * kg + v;
            const float th = m.cth[li];
            float u[JH];
            load_columns(u, m.XC + li * KL + cw);
#pragma unroll
            for (int j = 0; j < JH; j++) {
                uw[v] = fmaf(u[j], dv[j][v], uw[v]);
                dk[j][v] = th * (dk[j][v] - dv[j][v]);
                dv[j][v] *= th;
            }
        }
        add_up(uw, sums + 2 * kLrC);
    }
    lds_barrier();
    if (tid < L) {   // the sweep's scalars of a token
        float *o = tok + (tok0 + t0 + tid) * TF + 3 * D + 16;
        const float keep = 1.f - al, sa = sr_sigmoid(amean);
        o[0] = al;
        o[1] = th;
        // sigmoid' of the mean over d keep (the sweep forms keep <G_t, dG_{t+1}>): a saturated gate has no gradient
        o[2] = keep > 0.f ? sa * (1.f - sa) * (1.f / D) / keep : 0.f;
        o[3] = sr_sigmoid(emean) * (1.f / D);  // softplus' of the mean over d
        o[4] = -(sums[2 * kLrC + tid] + sums[3 * kLrC + tid]);
        o[5] = sums[tid] + sums[kLrC + tid];
    }
    float *Es = lds;  // dk, dv, dq, g, p: rows of stride KL, in front of the sums
    if (columns) {
#pragma unroll
        for (int v = 0; v < 4; v++) {
            float *e = Es + (li0 + 4 * kg + v) * KL + cw, k1[JH], v1[JH];
#pragma unroll
            for (int j = 0; j < JH; j++) { k1[j] = dk[j][v]; v1[j] = dv[j][v]; }
            store_columns(e, k1);
            store_columns(e + kLrC * KL, v1);
            store_columns(e + 2 * kLrC * KL, dp[v]);
            store_columns(e + 3 * kLrC * KL, xr[0][v]);
            store_columns(e + 4 * kLrC * KL, xr[1][v]);
        }
    }
    float dy[kLrC / 4];
#pragma unroll
    for (int i = 0; i < kLrC / 4; i++) {
        const int li = 16 * (i >> 2) + 4 * kg + (i & 3);
        dy[i] = li < L ? d_y[(tok0 + t0 + li) * D + wr + ml] : 0.f;
    }
    lds_barrier();
    if (columns) {   // dg0 = F_k^T dk + F_v^T dv + F_q^T dq, and F_k^T x
        f32x4 a[3][KT];
#pragma unroll
        for (int c = 0; c < 3; c++) {
#pragma unroll
            for (int kt = 0; kt < KT; kt++) a[c][kt] = *reinterpret_cast<const f32x4 *>(Es + (c * kLrC + li0 + ml) * KL + 16 * kt + 4 * kg);
        }
        float dg[4][JH], fx[4][JH];
#pragma unroll
        for (int j = 0; j < JH; j++) {
            f32x4 dgk[2] = {kZero, kZero}, dgv[2] = {kZero, kZero}, dgq[2] = {kZero, kZero}, fxk[2] = {kZero, kZero};
#pragma unroll
            for (int i = 0; i < 4 * KT; i++) {
                const int h = i >= 2 * KT;
                dgk[h] = mfma4(a[0][i >> 2][i & 3], f[0][i][j], dgk[h]);
                fxk[h] = mfma4(in[0][i >> 2][i & 3], f[0][i][j], fxk[h]);
                dgv[h] = mfma4(a[1][i >> 2][i & 3], f[1][i][j], dgv[h]);
                dgq[h] = mfma4(a[2][i >> 2][i & 3], f[2][i][j], dgq[h]);
            }
            const f32x4 dg4 = ((dgk[0] + dgk[1]) + (dgv[0] + dgv[1])) + (dgq[0] + dgq[1]), fx4 = fxk[0] + fxk[1];
#pragma unroll
            for (int v = 0; v < 4; v++) { dg[v][j] = dg4[v]; fx[v][j] = fx4[v]; }
        }
#pragma unroll
        for (int v = 0; v < 4; v++) {
            if (4 * kg + v < nt) {
                float *o = out + (size_t)(4 * kg + v) * TF + cw;
                store_columns(o + D, dg[v]);
                store_columns(o + 2 * D, fx[v]);
            }
        }
    }
    if (!rows) return;
    // outer products: dF_k, dF_v, dF_q with g, dF_mem with p; the first two stored as the sweep's lanes hold them, the others
    // as matrices
    f32x4 o[4][JH];
#pragma unroll
    for (int c = 0; c < 4; c++) {
#pragma unroll
        for (int j = 0; j < JH; j++) o[c][j] = kZero;
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
            for (int j = 0; j < JH; j++) {
                const float bg = e[3 * kLrC * KL + 16 * (c0 + j) + ml], bp = e[4 * kLrC * KL + 16 * (c0 + j) + ml];
                o[0][j] = mfma4(ak, bg, o[0][j]);
                o[1][j] = mfma4(av, bg, o[1][j]);
                o[2][j] = mfma4(bg, aq, o[2][j]);
                o[3][j] = mfma4(bp, ay, o[3][j]);
            }
        }
    }
#pragma unroll
    for (int j = 0; j < JH; j++) {
        const int jt = c0 + j;
#pragma unroll
        for (int c = 0; c < 2; c++)
            *reinterpret_cast<f32x4 *>(outer + (chunk * 4 + c) * DD + ((size_t)(rb * KT + jt) * 64 + lane) * 4) = o[c][j];
#pragma unroll
        for (int c = 2; c < 4; c++) {
            const int at = (wr + ml) * D + 16 * jt + 4 * kg;
            if (nc > 1) *reinterpret_cast<f32x4 *>(outer + (chunk * 4 + c) * DD + at) = o[c][j];
            else *reinterpret_cast<f32x4 *>(d_mems + (b * 6 + (c == 2 ? 2 : 5)) * DD + at) = o[c][j];   // no chunk passes them on
        }
    }
}

template <int D>
constexpr size_t prepare_lds_bytes() { return (chunk_lds_floats<D>(0) + PrepareLds<D>::floats) * sizeof(float); }
template <int D>
__global__ __launch_bounds__(kPrepThr) void selfref_bwd_prepare_kernel(SelfrefSweep a) {
    extern __shared__ __align__(16) float lds[];
    prepare_of<D>(a, blockIdx.x / a.nc, blockIdx.x % a.nc, lds);
}

// ── matrices ─────────────────────────────────────────────────────────────────────────────────────────────────────
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

// A matrix by way of registers to LDS, 4 D threads.
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

// acc += F_0^T B_0 + .. + F_(N-1)^T B_(N-1), the wave's 16 rows: contraction in the order 16 c + 4 kg + v, since rows 4 apart put
// the four kg of a read on different banks.  Operands are read two steps ahead: left to the compiler, a read stands right
// before its use.
template <int D, int N>
__device__ __forceinline__ void share_products(const float *const (&F)[N], const float *const (&B)[N], f32x4 (&acc)[D / 16], int wr,
                                               int ml, int kg) {
    constexpr int JT = D / 16, LD = D + 4, STEPS = D / 4;
    float a[3], b[3][JT];
    auto read = [&](int i) __attribute__((always_inline)) {
        const int k = 16 * (i % STEPS >> 2) + 4 * kg + (i & 3);
        a[i % 3] = F[i / STEPS][k * LD + wr + ml];
#pragma unroll
        for (int jt = 0; jt < JT; jt++) b[i % 3][jt] = B[i / STEPS][k * LD + 16 * jt + ml];
    };
    read(0);
    read(1);
#pragma unroll
    for (int i = 0; i < N * STEPS; i++) {
        if (i + 2 < N * STEPS) read(i + 2);
        __builtin_amdgcn_sched_barrier(0);
#pragma unroll
        for (int jt = 0; jt < JT; jt++) acc[jt] = mfma4(a[i % 3], b[i % 3][jt], acc[jt]);
        __builtin_amdgcn_sched_barrier(0);
    }
}
// Part c < KT of acc += B G_L^T, the wave's 16 rows, which are all it needs of B.
template <int D>
__device__ __forceinline__ void pass_part(const float *Bm, const float *GLT, f32x4 (&acc)[D / 16], int c, int wr, int ml, int kg) {
    constexpr int JT = D / 16, LD = D + 4;
    const f32x4 a = *reinterpret_cast<const f32x4 *>(Bm + (wr + ml) * LD + 16 * c + 4 * kg);
#pragma unroll
    for (int v = 0; v < 4; v++) {
        const int k = 16 * c + 4 * kg + v;
#pragma unroll
        for (int jt = 0; jt < JT; jt++) acc[jt] = mfma4(a[v], GLT[k * LD + 16 * jt + ml], acc[jt]);
    }
}

// ── the gradients of F_q and F_mem ───────────────────────────────────────────────────────────────────────────────
// Nothing of the sweep reaches them: dF_c <- dF'_c G_L^T + what the chunk's tokens add, chunk by chunk backwards, a row by
// itself.  A wave takes 16 rows of one of the two through a chain; its lane (ml, kg) holds row ml, columns 16 kt + 4 kg + v, operand and
// result of the product at once, and G_L comes straight from memory, two chunks ahead.  The matrices of `outer` become dF_c in place.
// 64 chains of 32 chunks, head size 64: 62 us, matrix instructions 27 of them.
template <int D>
__global__ __launch_bounds__(64) void selfref_bwd_scan_kernel(const float *__restrict__ gl, float *__restrict__ outer,
                                                              float *__restrict__ d_mems, int nc, int batch) {
    constexpr int KT = D / 16, DD = D * D;
    const int lane = threadIdx.x, ml = lane & 15, kg = lane >> 4;
    const size_t b = blockIdx.x % batch;   // the waves of a chain share an XCD's L2
    const int c = blockIdx.x / batch & 1, row0 = 16 * (blockIdx.x / batch >> 1);
    float *rows = outer + (b * nc * 4 + 2 + c) * DD + (row0 + ml) * D + 4 * kg;
    const float *g = gl + b * nc * DD + ml * D + 4 * kg;
    f32x4 f[KT], G[2][KT][KT], sums[2][KT];
    auto request = [&](int ci, int set) __attribute__((always_inline)) {
#pragma unroll
        for (int kt = 0; kt < KT; kt++) {
            sums[set][kt] = *reinterpret_cast<const f32x4 *>(rows + (size_t)ci * 4 * DD + 16 * kt);
#pragma unroll
            for (int jt = 0; jt < KT; jt++) G[set][kt][jt] = *reinterpret_cast<const f32x4 *>(g + (size_t)ci * DD + 16 * jt * D + 16 * kt);
        }
    };
    // Loads and stores stand on every path: the memory counter is in order, and behind a branch a wait would be for all of them.
    auto step = [&](int ci, int set) __attribute__((always_inline)) {
        f32x4 acc[KT];
#pragma unroll
        for (int jt = 0; jt < KT; jt++) acc[jt] = kZero;
#pragma unroll
        for (int kt = 0; kt < KT; kt++) {
#pragma unroll
            for (int v = 0; v < 4; v++) {
#pragma unroll
                for (int jt = 0; jt < KT; jt++) acc[jt] = mfma4(G[set][kt][jt][v], f[kt][v], acc[jt]);
            }
        }
#pragma unroll
        for (int jt = 0; jt < KT; jt++) f[jt] = acc[jt] + sums[set][jt];
        __builtin_amdgcn_sched_barrier(0);
        request(max(ci - 2, 0), set);
#pragma unroll
        for (int jt = 0; jt < KT; jt++) *reinterpret_cast<f32x4 *>(rows + (size_t)ci * 4 * DD + 16 * jt) = f[jt];
        __builtin_amdgcn_sched_barrier(0);
    };
#pragma unroll
    for (int kt = 0; kt < KT; kt++) f[kt] = *reinterpret_cast<const f32x4 *>(rows + (size_t)(nc - 1) * 4 * DD + 16 * kt);
    request(max(nc - 2, 0), 0);
    request(max(nc - 3, 0), 1);
    int ci = nc - 2;
    for (; ci >= 1; ci -= 2) {
        step(ci, 0);
        step(ci - 1, 1);
    }
    if (ci == 0) step(0, 0);
    float *out = d_mems + (b * 6 + (c ? 5 : 2)) * DD + (row0 + ml) * D + 4 * kg;
#pragma unroll
    for (int jt = 0; jt < KT; jt++) *reinterpret_cast<f32x4 *>(out + 16 * jt) = f[jt];
}

// Their share of dG_L at the end of every chunk but a chain's last: F_q^T dF'_q + F_mem^T dF'_mem, in place of the next chunk's
// dF_q and in the order of the sweep's lanes.  A workgroup per chunk, one memory after the other.  26 us for 1984 chunks at
// head size 64: 80 KB a chunk, 14 us of matrix instructions.
template <int D>
__global__ __launch_bounds__(4 * D) void selfref_bwd_share_kernel(const float *__restrict__ frozen, float *__restrict__ outer, int nc) {
    constexpr int JT = D / 16, DD = D * D, LD = D + 4;
    __shared__ __align__(16) float Fs[D * LD], Bm[D * LD];
    const int tid = threadIdx.x, wave = tid >> 6, lane = tid & 63, ml = lane & 15, kg = lane >> 4, wr = 16 * wave;
    const size_t chunk = blockIdx.x / (nc - 1) * nc + blockIdx.x % (nc - 1);
    const float *fz = frozen + chunk * 6 * DD;
    float *df = outer + ((chunk + 1) * 4 + 2) * DD;
    f32x4 acc[JT], f[2][JT], d[2][JT];
    request_matrix<D>(f[0], fz + 2 * DD, tid);
    request_matrix<D>(d[0], df, tid);
    request_matrix<D>(f[1], fz + 5 * DD, tid);
    request_matrix<D>(d[1], df + DD, tid);
#pragma unroll
    for (int jt = 0; jt < JT; jt++) acc[jt] = kZero;
#pragma unroll
    for (int c = 0; c < 2; c++) {
        if (c) __syncthreads();
        stage_matrix<D>(Fs, f[c], tid);
        stage_matrix<D>(Bm, d[c], tid);
        __syncthreads();
        share_products<D, 1>({Fs}, {Bm}, acc, wr, ml, kg);
    }
#pragma unroll
    for (int jt = 0; jt < JT; jt++) *reinterpret_cast<f32x4 *>(df + ((size_t)(wave * JT + jt) * 64 + lane) * 4) = acc[jt];
}

// ── the sweep ────────────────────────────────────────────────────────────────────────────────────────────────────
template <class Fn, int... I>
__device__ __forceinline__ void for_each(Fn &f, std::integer_sequence<int, I...>) {
    (f(std::integral_constant<int, I>{}), ...);
}
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

// dynamic LDS of the sweep: a tile's inputs, twice; dg; G_L^T; F and dF' of k and v; dk and dv
constexpr int sweep_tile_floats(int d) { return kTB * (5 * (d + 4) + d + 16); }
constexpr int sweep_lds_floats(int d) { return 2 * sweep_tile_floats(d) + kTB * (d + 4) + 5 * d * (d + 4) + d / 16 * 8 * 64; }

// One workgroup per chain, two waves per 16 rows (above).  Lane (ml, kg) = (lane % 16, lane / 16) holds of every matrix row ml of
// the wave's rows, columns CP kg + i (CP = D / 4): operand and result of the tile products (the contraction index runs
// over (i, kg)), and the coefficients of a product with a vector whose element CP kg + i is broadcast from lane i of
// DPP row kg.  dG is kept a second time by columns (dGT).  Tokens of a tile are result rows in the order sigma, so that
// lane kg owns the columns s = 4 v + kg of Y.
// FOLLOWED: what a chunk needs comes from workgroups that work beside this one (selfref_backward_kernel): sh counts the chunks whose
// share of dG_L is there (from the end of the chain), pr is 1 for a prepared chunk of the chain; done tells of the chunks whose dg is
// stored.  The second half asks a chunk ahead, so that nobody waits for the answer, and tells behind a wait that it has anyway.
template <int D, bool FOLLOWED>
__device__ __forceinline__ void sweep_of(const SelfrefSweep &args, size_t b, float *raw, const unsigned *pr, const unsigned *sh,
                                         unsigned *done) {
    const float *const emb = args.emb, *const k_cache = args.k, *const v_cache = args.v, *const frozen = args.frozen,
                *const gl = args.gl, *const tok = args.tok, *const outer = args.outer, *const csv = args.csv;
    float *const d_emb = args.d_emb, *const d_mems = args.d_mems;
    const int s = args.s, C = args.C, nc = args.nc;
    constexpr int CP = D / 4, KT = D / 16, JT = D / 16, NT = 4 * D, NW = D / 16, DD = D * D, V4 = D / 4, LD = D + 4;
    constexpr int TF = sweep_token_floats(D), TILE = kTB * LD;
    constexpr int LG = D + 16;                       // rows 4 v + kg of g fall on different banks for the four kg
    enum { A_K, A_U, A_X, A_DG0, A_FX };             // and g behind them
    constexpr int SET = sweep_tile_floats(D);
    static_assert(SET >= D * LD, "dG_L in the place of a tile's inputs");
    float *const DG = raw + 2 * SET, *const GLT = DG + TILE, *const Fa = GLT + D * LD, *const Fb = Fa + D * LD;   // G_L^T, F_k, F_v
    float *const Ba = Fb + D * LD, *const Bb = Ba + D * LD;   // dF'_k, dF'_v
    float *const dkv = Bb + D * LD;                  // dk, dv of a tile's tokens: [wave][v][2][lane]
    __shared__ __align__(16) float gams[2][kTB * kTB];   // x_t . k_s, s in the order sigma
    __shared__ __align__(16) float scs[2][kTB][8];       // alpha, theta, sigmoid' / (d keep), softplus' / d, dth0, dp . p
    __shared__ __align__(16) float Sx[NW][kTB], Cx[NW][kTB];
    __shared__ __align__(16) float av[2][D], av1[2][D];   // accE, accA at a boundary, before and behind it
    __shared__ float sp[NW];
#define T_(a, t, i) set[(a) * TILE + (t) * LD + (i)]
#define DG_(t, i) DG[(t) * LD + (i)]

    const bool second = __builtin_amdgcn_readfirstlane(threadIdx.x) >= NT;
    const int tid = second ? threadIdx.x - NT : threadIdx.x, r = tid >> 2, cq = tid & 3, wave = tid >> 6, lane = tid & 63;
    const int ml = lane & 15, kg = lane >> 4, wr = 16 * wave, c0 = cq * CP;
    const int s_of = sigma(lane & 15), kg_of = lane >> 4;   // as my_s and kg, for masks that stay in scalar registers
    const size_t tok0 = b * (size_t)s;

    if (FOLLOWED) {   // the last two chunks and the share between them
        if (threadIdx.x < 64) {
            while (!told(pr + nc - 1, 1) || !told(pr + nc - 2, 1) || !told(sh, 1)) __builtin_amdgcn_s_sleep(8);
        }
        __syncthreads();
        __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "agent");
    }

    f32x4 accEA = kZero;
    float dG[CP], dGT[CP], sig = 0.f;
    float *dmb = d_mems + b * 6 * DD;
    if (second) {   // the gradients of F_k and F_v, and as many barriers as the first half meets
        f32x4 dFm[2][JT];
        // Inputs of a tile: requested while the tile two before it is worked on, and in LDS while the tile before it is, in the
        // set that that one does not use.  Rows behind a chunk's last token are zeros.
        float4 pf_k, pf_v, pf_x, pf_g, pf_dg, pf_fx, pf_gam;
        float pf_s[6];
        int pf_ci = nc - 1, pf_tile = (s - (nc - 1) * C - 1) / kTB, pf_nt = 0;   // the tile to request; tokens of the one requested
        // No branch around the loads: the memory counter is in order, and behind a branch a wait would be for all of them.
        auto request = [&](int me) __attribute__((always_inline)) {
            const int first = pf_ci * C + pf_tile * kTB, last = min(pf_ci * C + C, s) - 1, stt = me / V4, sj = (me % V4) * 4;
            pf_nt = min(kTB, last + 1 - first);
            const size_t at = tok0 + min(first + stt, last), o = at * D + sj;
            const float *tp = tok + at * TF;
            auto two = [&](const float *q) {  // rows of tok are 8 bytes aligned
                const float2 lo = *reinterpret_cast<const float2 *>(q), hi = *reinterpret_cast<const float2 *>(q + 2);
                return make_float4(lo.x, lo.y, hi.x, hi.y);
            };
            pf_k = *reinterpret_cast<const float4 *>(k_cache + o);
            pf_v = *reinterpret_cast<const float4 *>(v_cache + o);
            pf_x = *reinterpret_cast<const float4 *>(emb + o);
            pf_g = two(tp + sj);
            pf_dg = two(tp + D + sj);
            pf_fx = two(tp + 2 * D + sj);
            pf_gam = two(tok + (tok0 + min(first + (me >> 2 & 15), last)) * TF + 3 * D + 4 * (me & 3));
            const float *e = tok + (tok0 + min(first + (me & 15), last)) * TF + 3 * D + 16;
#pragma unroll
            for (int i = 0; i < 6; i++) pf_s[i] = e[i];
            if (pf_tile > 0) pf_tile--;
            else if (pf_ci > 0) { pf_ci--; pf_tile = (C - 1) / kTB; }   // behind the last tile: it again, not used
        };
        auto stage = [&](int buf, int me) __attribute__((always_inline)) {
            float *set = raw + buf * SET;
            const int stt = me / V4, sj = (me % V4) * 4;
            auto in = [&](const float4 &x, int t) { return t < pf_nt ? x : make_float4(0, 0, 0, 0); };
            const float4 k = in(pf_k, stt), v = in(pf_v, stt);
            *reinterpret_cast<float4 *>(&T_(A_K, stt, sj)) = k;
            *reinterpret_cast<float4 *>(&T_(A_U, stt, sj)) = make_float4(k.x - v.x, k.y - v.y, k.z - v.z, k.w - v.w);
            *reinterpret_cast<float4 *>(&T_(A_X, stt, sj)) = in(pf_x, stt);
            *reinterpret_cast<float4 *>(&T_(A_DG0, stt, sj)) = in(pf_dg, stt);
            *reinterpret_cast<float4 *>(&T_(A_FX, stt, sj)) = in(pf_fx, stt);
            *reinterpret_cast<float4 *>(set + 5 * TILE + stt * LG + sj) = in(pf_g, stt);
            if (me < 64) *reinterpret_cast<float4 *>(&gams[buf][4 * me]) = in(pf_gam, me >> 2);
            if (me < kTB) {   // zeros behind the last token: it passes everything on as it is
                float x[6];
#pragma unroll
                for (int i = 0; i < 6; i++) x[i] = me < pf_nt ? pf_s[i] : 0.f;
                *reinterpret_cast<f32x4 *>(&scs[buf][me][0]) = f32x4{x[0], x[1], x[2], x[3]};
                *reinterpret_cast<float2 *>(&scs[buf][me][4]) = make_float2(x[4], x[5]);
            }
        };
        request(tid);
        stage(0, tid);
        request(tid);
        int stored = 0, whole = 0, told_of = 0;   // chunks whose dg was stored before now, before the tile before; as the others know
        for (int ci = nc - 1, buf = 0; ci >= 0; ci--) {
            const int t0 = ci * C, L = min(C, s - t0), ntile = (L + kTB - 1) / kTB;
            const size_t chunk = b * nc + ci;
            const float *fz = frozen + chunk * 6 * DD;
            unsigned ask_p = 1, ask_s = 1;   // answers of the chunk before the one before this
            int me = tid;
            asm volatile("" : "+v"(me));
            const int wave = me >> 6, lane = me & 63, ml = lane & 15, kg = lane >> 4;
            if (ci < nc - 1) {
                put_rows<D>(Ba, dFm[0], me);
                put_rows<D>(Bb, dFm[1], me);
            }
            lds_barrier();
            if (FOLLOWED) __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "agent");
            if (ci < nc - 1) {
                // accE <- G_L accE, accA <- G_L accA: rows 0 and 1 of one more product
                f32x4 accV[KT];
#pragma unroll
                for (int c = 0; c < KT; c++) {
                    const f32x4 a = ml < 2 ? *reinterpret_cast<const f32x4 *>(&av[ml][16 * c + 4 * kg]) : kZero;
                    accV[c] = kZero;
#pragma unroll
                    for (int v = 0; v < 4; v++) accV[c] = mfma4(a[v], GLT[(16 * c + 4 * kg + v) * LD + 16 * wave + ml], accV[c]);
                }
#pragma unroll
                for (int c = 1; c < KT; c++) accV[0] += accV[c];
                if (kg == 0) { av1[0][16 * wave + ml] = accV[0][0]; av1[1][16 * wave + ml] = accV[0][1]; }
                lds_barrier();   // dG_L is there
            } else {
                token_sums<D>(dFm[0], outer + chunk * 4 * DD, me);
                token_sums<D>(dFm[1], outer + (chunk * 4 + 1) * DD, me);
            }
            // Across the boundary dF_c = dF'_c G_L^T + what the tokens add: nobody waits for it, so it is formed while the other
            // half is among the tokens of the chunk's last tile, a part behind a barrier.
            f32x4 across[JT], sums[JT];
            auto pass = [&](auto part) {
                constexpr int c = decltype(part)::value / KT, q = decltype(part)::value % KT;
                if (q == 0) {
                    token_sums<D>(sums, outer + (chunk * 4 + c) * DD, me);
#pragma unroll
                    for (int jt = 0; jt < JT; jt++) across[jt] = kZero;
                }
                pass_part<D>(c ? Bb : Ba, GLT, across, q, 16 * wave, ml, kg);
                if (q == KT - 1) {
#pragma unroll
                    for (int jt = 0; jt < JT; jt++) dFm[c][jt] = across[jt] + sums[jt];
                }
            };
            f32x4 Fk[JT], Fv[JT];
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
                if (v == 2) stage_matrix<D>(Fb, Fv, me);
                if (v == 3) {
#pragma unroll
                    for (int i = 0; i < CP; i++) GLT[((me & 3) * CP + i) * LD + (me >> 2)] = G[i];
                }
            };
            using std::integral_constant;
            for (int tile = ntile - 1; tile >= 0; tile--, buf ^= 1) {
                const int nt = min(kTB, L - tile * kTB);
                const float *set = raw + buf * SET, *tg = set + 5 * TILE;
                for (int i = 0; i < 3; i++) lds_barrier();   // top, W and Z, the first token
                stage(buf ^ 1, me);
                if (FOLLOWED) {   // no load is under way here, and stores of the tile before have arrived
                    stores_arrived();
                    if (wave == 0 && (whole >= told_of + kTellChunks || (whole > told_of && whole >= nc - kTellChunks))) {
                        told_of = whole;
                        tell(done, told_of);
                    }
                    whole = stored;
                    if (tile == 0 && ci > 1) {
                        ask_p = __hip_atomic_load(pr + ci - 2, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
                        ask_s = __hip_atomic_load(sh, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
                    }
                }
                request(me);
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
                    request_matrix<D>(Fv, f + DD, me);
                }
                int left = 4 * ((nt + 3) / 4) - 3;   // the other tokens in whole groups of four; dk, dv
                if (tile == ntile - 1 && ci < nc - 1) {
                    const bool spread = left > 2 * KT;
                    auto next = [&](auto part) __attribute__((always_inline)) {
                        if (spread) lds_barrier();
                        pass(part);
                    };
                    for_each(next, std::make_integer_sequence<int, 2 * KT>{});
                    left -= spread ? 2 * KT : 0;
                }
                for (int i = 0; i < left; i++) lds_barrier();
#pragma unroll
                for (int v = 0; v < 4; v++) {
                    op[v][0] = dkv[((wave * 4 + v) * 2) * 64 + lane];
                    op[v][1] = dkv[((wave * 4 + v) * 2 + 1) * 64 + lane];
#pragma unroll
                    for (int jt = 0; jt < JT; jt++) gt[v][jt] = tg[(4 * v + kg) * LG + 16 * jt + ml];
                }
                dg = *reinterpret_cast<const f32x4 *>(DG + stt * LD + sj);
            }
            pending(0, integral_constant<int, 0>{});
            pending(0, integral_constant<int, 1>{});
            pending(0, integral_constant<int, 2>{});
            pending(0, integral_constant<int, 3>{});
            stored++;
            // the chunk after the next needs its preparation and its share; the other half meets this one at the next barrier
            if (FOLLOWED && ci > 1 && (!ask_p || ask_s < (unsigned)(nc - ci + 1))) {
                while (!told(pr + ci - 2, 1) || !told(sh, nc - ci + 1)) __builtin_amdgcn_s_sleep(2);
            }
        }
#pragma unroll
        for (int c = 0; c < 2; c++) {   // gradients of the initial memories
#pragma unroll
            for (int jt = 0; jt < JT; jt++) {
#pragma unroll
                for (int v = 0; v < 4; v++) dmb[(size_t)c * DD + (wr + 4 * kg + v) * D + 16 * jt + ml] = dFm[c][jt][v];
            }
        }
        if (FOLLOWED) stores_arrived();
        __syncthreads();
        if (FOLLOWED && tid < 64) tell(done, nc);
        __syncthreads();
        return;
    }
#pragma unroll
    for (int i = 0; i < CP; i++) dG[i] = dGT[i] = 0.f;
    if (tid < NW * kTB) (&Sx[0][0])[tid] = 0.f;

    // A chunk's share of dG_L and column sums of F_eta, F_alpha, requested in the last tile of the chunk behind it.
    f32x4 share[JT], csr[2];
    float cs1[2];
    auto ahead = [&](size_t chunk, int me, bool behind) __attribute__((always_inline)) {
        const int row = 16 * (me >> 6);
        if (behind) token_sums<D>(share, outer + ((chunk + 1) * 4 + 2) * DD, me);   // of F_q and F_mem
        const float *c = csv + chunk * 2 * D + row;
#pragma unroll
        for (int i = 0; i < 2; i++) csr[i] = *reinterpret_cast<const f32x4 *>(c + i * D + 4 * (me >> 4 & 3));
        cs1[0] = c[me & 15];
        cs1[1] = c[D + (me & 15)];
    };
    ahead(b * nc + nc - 1, tid, false);
    for (int ci = nc - 1, buf = 0; ci >= 0; ci--) {
        const int t0 = ci * C, L = min(C, s - t0), ntile = (L + kTB - 1) / kTB;
        const size_t chunk = b * nc + ci;
        const float *fz = frozen + chunk * 6 * DD;
        // the thread's place through an opaque copy, once per chunk: addresses made of it are not to live across the sweep
        int me = tid;
        asm volatile("" : "+v"(me));
        const int wave = me >> 6, lane = me & 63, ml = lane & 15, kg = lane >> 4, wr = 16 * wave;
        float FTk[CP], FTu[CP];   // rows of F_k^T and (F_k - F_v)^T
        float csE = cs1[0], csA = cs1[1];
        // LDS-only barriers from here on: requests and the stores of dg stay under way across them
        if (ci < nc - 1 && kg == 0) { av[0][wr + ml] = accEA[0]; av[1][wr + ml] = accEA[1]; }
        lds_barrier();
        if (FOLLOWED) __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "agent");
        sig = 0.f;
        if (ci < nc - 1) {
            // Chunk boundary: gradients of F'_c = F_c G_L flow into dG_L = sum_c F_c^T dF'_c and dF_c = dF'_c G_L^T, on
            // the matrix cores; the rows of dF_eta, dF_alpha are all equal (rank-1 terms of dG_L).
            f32x4 accG[JT];
#pragma unroll
            for (int i = 0; i < JT; i++) accG[i] = kZero;
            share_products<D, 2>({Fa, Fb}, {Ba, Bb}, accG, wr, ml, kg);
#pragma unroll
            for (int i = 0; i < CP; i++) {
                FTk[i] = Fa[(CP * kg + i) * LD + wr + ml];
                FTu[i] = Fb[(CP * kg + i) * LD + wr + ml];
            }
            // sigma_L = <G_L, dG_L>; then (1-a_t) <G_t, dG_{t+1}> = sigma_{t+1} + th_t u.W_t and
            // sigma_t = that + dg.g + dp.p carry the inner product the gradient of alpha needs
            float part[JT];
#pragma unroll
            for (int jt = 0; jt < JT; jt++) {
                const float eE = av[0][16 * jt + ml], eA = av[1][16 * jt + ml];
                const f32x4 G = *reinterpret_cast<const f32x4 *>(GLT + (16 * jt + ml) * LD + wr + 4 * kg);
#pragma unroll
                for (int v = 0; v < 4; v++) share[jt][v] += accG[jt][v] + (csr[0][v] * eE + csr[1][v] * eA);
                part[jt] = (G[0] * share[jt][0] + G[1] * share[jt][1]) + (G[2] * share[jt][2] + G[3] * share[jt][3]);
            }
#pragma unroll
            for (int jt = 1; jt < JT; jt++) part[0] += part[jt];
            float *const dGL = raw + (buf ^ 1) * SET;   // the set of the tile before is idle here
            put_rows<D>(dGL, share, me);
            const float whole = wave_allreduce(part[0]);
            if (lane == 0) sp[wave] = whole;
            lds_barrier();
            accEA = kZero;   // rows 0 and 1 count
            if (kg == 0) { accEA[0] = av1[0][wr + ml]; accEA[1] = av1[1][wr + ml]; }
#pragma unroll
            for (int w = 0; w < NW; w++) sig += sp[w];
            lds_read<CP>(dG, dGL + (wr + ml) * LD + CP * kg);
#pragma unroll
            for (int i = 0; i < CP; i++) dGT[i] = dGL[(CP * kg + i) * LD + wr + ml];
        } else {
#pragma unroll
            for (int i = 0; i < CP; i++) {
                const float *f = fz + (CP * kg + i) * D + wr + ml;
                FTk[i] = f[0];
                FTu[i] = f[DD];
            }
        }
#pragma unroll
        for (int i = 0; i < CP; i++) FTu[i] = FTk[i] - FTu[i];
        // arrived here: a wait for them inside the tile loop would be one for the next tile's requests as well
        asm volatile("" : "+v"(csE), "+v"(csA));

        for (int tile = ntile - 1; tile >= 0; tile--, buf ^= 1) {
            const int nt = min(kTB, L - tile * kTB);
            float *const set = raw + buf * SET, *const tg = set + 5 * TILE;
            const float *const gam = gams[buf], (*const sc)[8] = scs[buf];
            float *const Ws = raw + (buf ^ 1) * SET, *const Zs = Ws + TILE;   // until the next tile's inputs come
            int me = tid;   // and once per tile
            asm volatile("" : "+v"(me));
            const int tid = me, wave = tid >> 6, lane = tid & 63, ml = lane & 15, kg = lane >> 4, wr = 16 * wave,
                      stt = tid / V4, sj = (tid % V4) * 4,      // staging slot: token, column
                      ve = CP * kg + ml % CP,                   // the vector element a lane holds
                      tcol = CP * (ml >> 2) + (ml & 3),         // column of result row ml of block 0; block kt: + 4 kt
                      my_s = sigma(ml);                         // token of operand row ml
            lds_barrier();
            if (nt < kTB) *reinterpret_cast<float4 *>(DG + stt * LD + sj) = make_float4(0, 0, 0, 0);   // dg behind the last token

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
                Ws[(4 * v + kg) * LD + wr + ml] = W[v];
                Zs[(4 * v + kg) * LD + wr + ml] = Z[v];
            }
            lds_barrier();
#pragma unroll
            for (int i = 0; i < CP; i += 4) {
                const f32x4 w4 = *reinterpret_cast<const f32x4 *>(Ws + my_s * LD + CP * kg + i);
                const f32x4 z4 = *reinterpret_cast<const f32x4 *>(Zs + my_s * LD + CP * kg + i);
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
            if (tile == 0 && ci > 0) ahead(chunk - 1, me, true);

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
                DG_(t, wr + ml) = fmaf(da, csA, fmaf(de, csE, fmaf(-th, ybc, dg0)));
                lds_barrier();
                const float dgv = DG_(t, ve), gv = tg[t * LG + ve];
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
                W = mfma4(ct[j] * gam[t * kTB + ml], DG_(t, wr + ml), W);
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
                    const float bg = below[j] * DG_(t, wr + ml), bx = below[j] * T_(A_X, t, wr + ml);
#pragma unroll
                    for (int kt = 0; kt < KT; kt++) {
                        n[kt] = mfma4(T_(A_X, t, tcol + 4 * kt), bg, n[kt]);
                        nT[kt] = mfma4(DG_(t, tcol + 4 * kt), bx, nT[kt]);
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
#undef DG_
}

template <int D>
__global__ __launch_bounds__(8 * D) void selfref_bwd_sweep_kernel(SelfrefSweep a) {
    extern __shared__ __align__(16) float raw[];
    sweep_of<D, false>(a, blockIdx.x, raw, nullptr, nullptr, nullptr);
}

// ── all of it at once ────────────────────────────────────────────────────────────────────────────────────────────
// A chain's gradients of F_q and F_mem and their share of dG_L, as selfref_bwd_scan_kernel and selfref_bwd_share_kernel, chunk by
// chunk as the chunks are prepared.  8 D threads: a wave has 16 rows of one of the two, and 16 rows and half of the columns of a share.
template <int D>
constexpr int passed_lds_floats() { return 4 * D * (D + 4); }
template <int D>
__device__ __forceinline__ void passed_of(const SelfrefSweep &a, size_t b, float *lds, const unsigned *prepared, unsigned *shares) {
    constexpr int KT = D / 16, DD = D * D, LD = D + 4, NW = D / 16, JH = KT / 2, STEPS = D / 4;
    static_assert(KT % 2 == 0, "two waves for 16 rows of a share");
    const int tid = threadIdx.x, wave = tid >> 6, lane = tid & 63, ml = lane & 15, kg = lane >> 4, nc = a.nc;
    const int c = wave / NW, row0 = 16 * (wave % NW);
    float *const Fs = lds, *const Bm = lds + 2 * D * LD;   // F_q, F_mem; dF'_q, dF'_mem
    float *const rows = a.outer + (b * nc * 4 + 2 + c) * DD + (row0 + ml) * D + 4 * kg;
    const float *const g = a.gl + b * nc * DD + ml * D + 4 * kg;
    f32x4 f[KT], G[KT][KT], sums[KT], F[KT];
    auto request_F = [&](int ci) {   // half the threads for each matrix
#pragma unroll
        for (int i = 0; i < KT; i++)
            F[i] = *reinterpret_cast<const f32x4 *>(a.frozen + ((b * nc + ci) * 6 + (c ? 5 : 2)) * DD + (tid % (4 * D) + i * 4 * D) * 4);
    };
    request_F(nc - 2);
    wait_told(prepared + nc - 1, 1, 1);
#pragma unroll
    for (int kt = 0; kt < KT; kt++) f[kt] = *reinterpret_cast<const f32x4 *>(rows + (size_t)(nc - 1) * 4 * DD + 16 * kt);
    for (int ci = nc - 2; ci >= 0; ci--) {
        stage_matrix<D>(Fs + c * D * LD, F, tid % (4 * D));
#pragma unroll
        for (int kt = 0; kt < KT; kt++) *reinterpret_cast<f32x4 *>(Bm + c * D * LD + (row0 + ml) * LD + 16 * kt + 4 * kg) = f[kt];
        __syncthreads();
        request_F(max(ci - 1, 0));
        {   // the same sums in the same order as a workgroup that takes one memory after the other
            f32x4 acc[JH];
#pragma unroll
            for (int j = 0; j < JH; j++) acc[j] = kZero;
            for (int m = 0; m < 2; m++) {
                const float *Fm = Fs + m * D * LD + row0 + ml, *B = Bm + m * D * LD + 16 * JH * c + ml;
#pragma unroll
                for (int i = 0; i < STEPS; i++) {
                    const int k = 16 * (i >> 2) + 4 * kg + (i & 3);
#pragma unroll
                    for (int j = 0; j < JH; j++) acc[j] = mfma4(Fm[k * LD], B[k * LD + 16 * j], acc[j]);
                }
            }
            float *share = a.outer + ((b * nc + ci + 1) * 4 + 2) * DD;
#pragma unroll
            for (int j = 0; j < JH; j++)
                *reinterpret_cast<f32x4 *>(share + ((size_t)(wave % NW * KT + JH * c + j) * 64 + lane) * 4) = acc[j];
        }
        stores_arrived();
        wait_told(prepared + ci, 1, 1);   // everybody's part of the share has arrived
        if (wave == 0) tell(shares, nc - 1 - ci);
#pragma unroll
        for (int kt = 0; kt < KT; kt++) {
            sums[kt] = *reinterpret_cast<const f32x4 *>(rows + (size_t)ci * 4 * DD + 16 * kt);
#pragma unroll
            for (int jt = 0; jt < KT; jt++) G[kt][jt] = *reinterpret_cast<const f32x4 *>(g + (size_t)ci * DD + 16 * jt * D + 16 * kt);
        }
        f32x4 acc[KT];
#pragma unroll
        for (int jt = 0; jt < KT; jt++) acc[jt] = kZero;
#pragma unroll
        for (int kt = 0; kt < KT; kt++) {
#pragma unroll
            for (int v = 0; v < 4; v++) {
#pragma unroll
                for (int jt = 0; jt < KT; jt++) acc[jt] = mfma4(G[kt][jt][v], f[kt][v], acc[jt]);
            }
        }
#pragma unroll
        for (int jt = 0; jt < KT; jt++) f[jt] = acc[jt] + sums[jt];
    }
    float *out = a.d_mems + (b * 6 + (c ? 5 : 2)) * DD + (row0 + ml) * D + 4 * kg;
#pragma unroll
    for (int jt = 0; jt < KT; jt++) *reinterpret_cast<f32x4 *>(out + 16 * jt) = f[jt];
}

// Counters: the numbers drawn, by workgroups and for the chunks of the first and the last ones; a chain's shares, its chunks with dg; a
// flag for each prepared chunk.
struct BackwardCounters {
    unsigned *drawn;
    int batch, nc;
    __host__ __device__ unsigned *next(int i) const { return drawn + (1 + i) * kTellStride; }
    __host__ __device__ unsigned *shares(size_t b) const { return drawn + (3 + b) * kTellStride; }
    __host__ __device__ unsigned *swept(size_t b) const { return drawn + (3 + batch + b) * kTellStride; }
    __host__ __device__ unsigned *prepared(size_t b) const { return drawn + (3 + 2 * (size_t)batch) * kTellStride + b * nc; }
    size_t words() const { return (3 + 2 * (size_t)batch) * kTellStride + (size_t)batch * nc; }
};
// The sweeps leave most of the compute units idle, need one prepared chunk after the other, from the end, and their dg becomes d_x
// chunk by chunk.  So one launch has workgroups that prepare chunks, in the order in which they are needed; for each chain one that
// takes the gradients of F_q and F_mem through it, and the sweep; and those that form d_x, which start as the first ones end.  The
// order of the numbers (handover.h) is that order.  A workgroup fills a compute unit's LDS.
// 64 chains of 2048 tokens, head size 64, chunks of 64: 1.49 ms for 0.29 + 0.06 + 0.03 + 1.29 + 0.06 of five launches.  The
// preparation ends at 0.69 ms, a sweep starts at 0.05 and is slower than alone by 5 % (its neighbours' code and traffic), the last
// d_x is 8 us behind the last sweep.  With the chunks dealt out beforehand the last d_x was 170 us behind: some workgroups of the last
// kind find no place before the sweeps end.  Of 256 registers a lane six values are spilled (20 bytes of scratch; the sweep by itself
// spills four).
template <int D>
__global__ __launch_bounds__(8 * D) void selfref_backward_kernel(SelfrefSweep a, BackwardCounters n, int preparers) {
    static_assert(8 * D == kPrepThr, "the same workgroup for all");
    extern __shared__ __align__(16) float raw[];
    int role = draw(n.drawn);
    const int tasks = a.batch * a.nc;
    if (role < preparers) {
        for (int task = draw(n.next(0)); task < tasks; task = draw(n.next(0))) {
            const int ci = a.nc - 1 - task / a.batch;
            const size_t b = task % a.batch;
            prepare_of<D>(a, b, ci, raw);
            stores_arrived();
            __syncthreads();
            if (threadIdx.x < 64) tell(n.prepared(b) + ci, 1);
        }
        return;
    }
    role -= preparers;
    if (role < a.batch) {
        passed_of<D>(a, role, raw, n.prepared(role), n.shares(role));
        return;
    }
    role -= a.batch;
    if (role < a.batch) {
        sweep_of<D, true>(a, role, raw, n.prepared(role), n.shares(role), n.swept(role));
        return;
    }
    if (threadIdx.x >= 4 * D) return;
    for (int task = draw(n.next(1)); task < tasks; task = draw(n.next(1))) {
        const int ci = a.nc - 1 - task / a.batch;
        const size_t b = task % a.batch;
        dx_of_chunk<D, true>(raw, a.k, a.v, a.alpha, a.theta, a.d_emb, nullptr, b, ci, a.s, a.C,
                             [&] { wait_told(n.swept(b), 1, a.nc - ci); });
        __syncthreads();   // the chunk's LDS is free
    }
}

template <int D>
bool launch_together(const SelfrefSweep &a) {
    const int cus = compute_units();
    BackwardCounters n{nullptr, a.batch, a.nc};
    const Counters counters(43, n.words());
    if (!counters.at) return false;
    n.drawn = counters.at;
    constexpr size_t sweep = sweep_lds_floats(D) * sizeof(float), lds = sweep > prepare_lds_bytes<D>() ? sweep : prepare_lds_bytes<D>();
    static_assert(lds >= kAloneFloats * sizeof(float) && lds >= passed_lds_floats<D>() * sizeof(float) &&
                  lds >= chunk_lds_floats<D>(2) * sizeof(float), "LDS");
    const long long tasks = (long long)a.batch * a.nc, rest = cus - 2 * a.batch;
    const int others = (int)(tasks < rest ? tasks : rest);
    check_hip(hipFuncSetAttribute(reinterpret_cast<const void *>(selfref_backward_kernel<D>), hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds),
              "dynamic LDS size");
    KernelTimer kt("selfref_backward_kernel");
    hipLaunchKernelGGL((selfref_backward_kernel<D>), dim3(2 * a.batch + 2 * others), dim3(8 * D), lds, counters.on, a, n,
                       others);
    check_launch("selfref_backward_kernel");
    return true;
}

template <int D>
bool launch(const SelfrefSweep &a) {
    constexpr size_t lds = prepare_lds_bytes<D>();
    static_assert(5 * kLrC * (D + 4) <= chunk_lds_floats<D>(0) + PrepareLds<D>::sums, "operands of the outer products");
    static_assert(lds <= 160 * 1024, "LDS");
    if constexpr (8 * D == kPrepThr) {
        // Together where the chunks are more than the chip prepares in two rounds, beside chains that leave at least half of it to
        // them.  Otherwise the preparation is over before the sweep is far, and what a sweep does here besides (0.9 us a chunk, and
        // its first chunks to wait for) costs more than the launches behind each other.  Apart / together: 64 chains of 2048 tokens
        // 1734 / 1484 us in chunks of 64 and 2081 / 1887 in chunks of 32, of 512 tokens 430 / 420 and 509 / 488; 24 of 1400 1.05, 32 of
        // 1000 1.03, 48 of 400 1.03 times as fast; 16 of 1000 (256 chunks) 0.98, 64 of 200 0.87.  Chunks have two tiles at least, since
        // the inputs of a tile are requested two tiles ahead and those of one chunk ahead are there.
        const int cus = compute_units();
        if (a.C >= 2 * kTB && 4 * a.batch <= cus && (long long)a.batch * a.nc >= 2 * cus && launch_together<D>(a)) return true;
    }
    check_hip(hipFuncSetAttribute(reinterpret_cast<const void *>(selfref_bwd_prepare_kernel<D>),
                                  hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds), "dynamic LDS size");
    hipLaunchKernelGGL((selfref_bwd_prepare_kernel<D>), dim3(a.batch * a.nc), dim3(kPrepThr), lds, stream(), a);
    check_launch("selfref_bwd_prepare_kernel");
    if (a.nc > 1) {
        hipLaunchKernelGGL((selfref_bwd_scan_kernel<D>), dim3(2 * (D / 16) * a.batch), dim3(64), 0, stream(), a.gl, a.outer, a.d_mems,
                           a.nc, a.batch);
        check_launch("selfref_bwd_scan_kernel");
        hipLaunchKernelGGL((selfref_bwd_share_kernel<D>), dim3(a.batch * (a.nc - 1)), dim3(4 * D), 0, stream(), a.frozen, a.outer,
                           a.nc);
        check_launch("selfref_bwd_share_kernel");
    }
    constexpr size_t sweep_lds = sweep_lds_floats(D) * sizeof(float);
    check_hip(hipFuncSetAttribute(reinterpret_cast<const void *>(selfref_bwd_sweep_kernel<D>),
                                  hipFuncAttributeMaxDynamicSharedMemorySize, (int)sweep_lds), "dynamic LDS size");
    KernelTimer kt("selfref_bwd_kernel");
    hipLaunchKernelGGL((selfref_bwd_sweep_kernel<D>), dim3(a.batch), dim3(8 * D), sweep_lds, stream(), a);
    check_launch("selfref_bwd_sweep_kernel");
    return false;
}

}  // namespace

bool selfref_backward_sweep(const SelfrefSweep &a) {
    return a.d == 16 ? launch<16>(a) : a.d == 32 ? launch<32>(a) : launch<64>(a);
}

}  // namespace nlh
