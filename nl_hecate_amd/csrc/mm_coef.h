// Gate coefficients of the chunkwise matrix forms on the fp32 matrix cores: the vectors a, beta, h and the table
// c of one chunk of up to 64 tokens, built in LDS by the first waves of a 512-thread workgroup.
#pragma once
#include <hip/hip_runtime.h>

#include "mm_tiles.h"

namespace nlh {
namespace mmt {

// Gate coefficients of one chunk (L <= 64 tokens), all in LDS.
struct Coef {
    float al[CW], th[CW], et[CW];   // gates (eta = 0 for the Delta rule), zero beyond L
    float a[CW], beta[CW], h[CW];   // a_t, beta_t, h_t
    float cl[CW], bl[CW];           // c[L-1,j], bb[j,L-1]
};

// Gates of token (lane % 64) of a chunk, one register each; zero beyond L (eta = 0 without S).
struct Gates { float al, th, et; };
__device__ __forceinline__ Gates fetch_gates(const float *alpha, const float *theta, const float *eta, int L,
                                             bool has_s) {
    const int t = threadIdx.x & 63;
    Gates g;
    g.al = t < L ? alpha[t] : 0.f;
    g.th = t < L ? theta[t] : 0.f;
    g.et = (t < L && has_s) ? eta[t] : 0.f;
    return g;
}
__device__ __forceinline__ void load_gates(Coef &cf, const Gates &g) {
    const int t = threadIdx.x;
    if (t < CW) { cf.al[t] = g.al; cf.th[t] = g.th; cf.et[t] = g.et; }
}

__device__ __forceinline__ float lane_bcast(float x, int lane) {
    return __builtin_bit_cast(float, __builtin_amdgcn_readlane(__builtin_bit_cast(int, x), lane));
}

// The gates of a token as a map of the weights that an earlier term has in (M, S): keep M + eta S, eta S; a run of tokens composes
// to an upper triangular map (chunk_coef.h has the algebra).  T: type of the recurrences.  In float every composition
// rounds; float64 leaves the rounding of what is kept.
template <class T>
struct GateMap { T R, X, H; };   // [[R, X], [0, H]]
template <class T>
__device__ __forceinline__ GateMap<T> after(const GateMap<T> &l, const GateMap<T> &e) {   // l behind e
    return {l.R * e.R, fma(l.R, e.X, l.X * e.H), l.H * e.H};
}
// value of the lane of the same 16-lane row that DPP control CTRL names, `fill` where there is none
template <int CTRL, class T>
__device__ __forceinline__ T row_moved(T x, T fill) {
    if constexpr (sizeof(T) == 8) {
        const long long u = __builtin_bit_cast(long long, x), f = __builtin_bit_cast(long long, fill);
        const unsigned lo = __builtin_amdgcn_update_dpp((int)f, (int)u, CTRL, 0xF, 0xF, false);
        const unsigned hi = __builtin_amdgcn_update_dpp((int)(f >> 32), (int)(u >> 32), CTRL, 0xF, 0xF, false);
        return __builtin_bit_cast(T, (long long)(((unsigned long long)hi << 32) | lo));
    } else {
        return __builtin_bit_cast(T, __builtin_amdgcn_update_dpp(__builtin_bit_cast(int, fill), __builtin_bit_cast(int, x), CTRL,
                                                                 0xF, 0xF, false));
    }
}
template <int CTRL, class T>
__device__ __forceinline__ GateMap<T> row_moved(const GateMap<T> &m) {
    return {row_moved<CTRL>(m.R, T(1)), row_moved<CTRL>(m.X, T(0)), row_moved<CTRL>(m.H, T(1))};
}
template <class T>
__device__ __forceinline__ T lane_of(T x, int lane) {
    if constexpr (sizeof(T) == 8) {
        const long long u = __builtin_bit_cast(long long, x);
        const unsigned lo = __builtin_amdgcn_readlane((int)u, lane), hi = __builtin_amdgcn_readlane((int)(u >> 32), lane);
        return __builtin_bit_cast(T, (long long)(((unsigned long long)hi << 32) | lo));
    } else {
        return lane_bcast(x, lane);
    }
}

// The vectors of a chunk (wave 0) and, where Cc is given, column j of c in lane j: Cc[t][j] (stride LDM; entries outside
// j <= t < L are zero), tokens 16 w .. 16 w + 15 by wave w < 4.  Needs a barrier afterwards.
// Every wave composes the maps inside the four blocks of 16 tokens by scans and starts its own block's recurrence, 16 steps,
// from what an earlier token's weight has become by then.  One wave that took the recurrence through all 64 tokens was the
// others' wait: 7 to 9 k clocks of the 27 k (outputs), 32 k (local backward) and 63 k (gradients) that a chunk of float tokens takes.
template <class T = float>
__device__ __forceinline__ void coefficients(Coef &cf, const Gates &g, int L, float *Cc) {
    const int j = threadIdx.x & 63, w = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), J = j >> 4;
    if (w >= (Cc ? 4 : 1)) return;
    const bool jv = j < L;
    const T keep = T(1) - T(g.al), et = T(g.et);   // 1 and 0 beyond L
    using M = GateMap<T>;
    const M id = {T(1), T(0), T(1)}, own = jv ? M{keep, et, et} : id;
    M hd = own;   // the block's tokens up to j
    hd = after(hd, row_moved<0x111>(hd));
    hd = after(hd, row_moved<0x112>(hd));
    hd = after(hd, row_moved<0x114>(hd));
    hd = after(hd, row_moved<0x118>(hd));
    M sf = own;   // the block's tokens from j on
    sf = after(row_moved<0x101>(sf), sf);
    sf = after(row_moved<0x102>(sf), sf);
    sf = after(row_moved<0x104>(sf), sf);
    sf = after(row_moved<0x108>(sf), sf);
    const M tl = row_moved<0x101>(sf);   // behind j
    M blk[4];
#pragma unroll
    for (int b = 0; b < 4; b++) blk[b] = {lane_of(hd.R, 16 * b + 15), lane_of(hd.X, 16 * b + 15), lane_of(hd.H, 16 * b + 15)};
    if (w == 0) {
        const M pre2 = after(blk[1], blk[0]), pre3 = after(blk[2], pre2), post1 = after(blk[3], blk[2]), post0 = after(post1, blk[1]);
        const M pf = after(hd, J == 0 ? id : J == 1 ? blk[0] : J == 2 ? pre2 : pre3);
        const M sx = after(J == 3 ? id : J == 2 ? blk[3] : J == 1 ? post1 : post0, tl);
        cf.a[j] = jv ? (float)pf.R : 0.f;
        cf.beta[j] = jv ? (float)pf.X : 0.f;
        cf.h[j] = jv ? (float)pf.H : 0.f;
        cf.cl[j] = jv ? (float)(sx.R + sx.X) : 0.f;
        cf.bl[j] = jv ? (float)sx.H : 0.f;
    }
    if (!Cc) return;
    // whole blocks between j's and this wave's
    const M between = w == 3 ? (J == 0 ? after(blk[2], blk[1]) : J == 1 ? blk[2] : id) : w == 2 && J == 0 ? blk[1] : id;
    const M start = after(between, tl);
    T b = J < w ? start.H : T(1), c = J < w ? start.R + start.X : T(1);
    float *out = Cc + 16 * w * LDM + j;
#pragma unroll
    for (int u = 0; u < 16; u++) {
        const int t = 16 * w + u;
        const T kp = lane_of(keep, t), e = lane_of(et, t);
        const bool behind = t > j;
        b *= behind ? e : T(1);
        c = behind ? fma(kp, c, b) : c;
        out[u * LDM] = (jv && t >= j && t < L) ? (float)c : 0.f;
    }
}

}  // namespace mmt
}  // namespace nlh
