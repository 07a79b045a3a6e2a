// Gate coefficients of one chunk of the frozen-M0 chunkwise Titans / Delta rule, computed inside
// the kernels that use them (no table in HBM).
//
// With keep_t = 1 - alpha_t and the per-token map g_t = [[keep_t, eta_t], [0, eta_t]] acting on
// (weight in M, weight in S) of an earlier rank-1 term, a range of tokens composes to an upper
// triangular 2x2 map G(a..b) = g_b ... g_a = [[R, X], [0, H]] (R = prod keep, H = prod eta).  The
// coefficients of chunkwise_mm.hip are entries of such maps:
//   a_t = R(0..t), beta_t = X(0..t), h_t = H(0..t)
//   r[j][t] = R(j+1..t), bb[j][t] = H(j+1..t), c[t][j] = R(j+1..t) + X(j+1..t)      (j <= t)
//   cl_j = c[L-1][j], bl_j = bb[j][L-1], rl_j = r[j][L-1]
// Tokens beyond a short chunk's length L carry the identity map, so "L-1" is always token 63.
// A chunk is cut into four blocks of 16 tokens (one DPP row of a wave each).  One wave scans the
// maps inside the blocks (prefixes "head", suffixes "tail") and across them; every other quantity
// is a product of at most three maps, without a division (a saturated gate, keep = 0 or eta = 0,
// is an ordinary value):
//   tokens j < t in different blocks J < T:  G(j+1..t) = head_t . mid(J,T) . tail_j
//     => c[t][j] = A.R zc_j + A.X zh_j,  bb[j][t] = A.H zh_j,  r[j][t] = A.R zr_j,  A = head_t . mid(J,T)
//   tokens in the same block: a 16-step recurrence per lane (coef_diag_*).
#pragma once
#include <hip/hip_runtime.h>

#include <algorithm>

#include "lane_ops.h"
#include "runtime.h"

namespace nlh {
namespace {

// Chunks that a wave of the coefficient passes walks over: up to four once there are sixteen waves for every compute unit
// (their loads then run under the chunk before), one where there are fewer (four sequences of eight chunks:
// 13 us in eight waves, 5 in 32).
inline int coef_chunks_per_wave(int chunks) { return std::clamp(chunks / (16 * compute_units()), 1, 4); }

typedef float cf32x4 __attribute__((ext_vector_type(4)));

struct Map3 { float R, X, H; };   // [[R, X], [0, H]]
__device__ __forceinline__ Map3 map_identity() { return Map3{1.f, 0.f, 1.f}; }
// later . earlier
__device__ __forceinline__ Map3 compose(const Map3 &l, const Map3 &e) {
    return Map3{l.R * e.R, fmaf(l.R, e.X, l.X * e.H), l.H * e.H};
}

// Everything the consumers read, in LDS (one per chunk in flight).
struct ChunkCoef {
    float keep[64], eta[64], th[64];   // gates; beyond L: 1, 0, 0  (the scan itself uses the identity map there)
    float hR[64], hX[64], hH[64];      // head_t = G(16 T .. t)
    float zc[64], zh[64], zr[64];      // tail_j = G(j+1 .. 16 J + 15):  R + X, H, R
    float a[64], beta[64], h[64];      // G(0 .. t)
    float cl[64], bl[64], rl[64];      // G(j+1 .. 63): R + X, H, R
    float mid[6][4];                   // mid(J,T) for (0,1) (0,2) (0,3) (1,2) (1,3) (2,3): R, X, H, unused
    float last[4];                     // a_63, beta_63, h_63 (= a_L, beta_L, h_L), unused
};
__device__ __forceinline__ int mid_index(int J, int T) { return J == 0 ? T - 1 : (J == 1 ? T + 1 : 5); }

// value of lane (i - n) of the same 16-lane row, `fill` where that lane does not exist
template <int N>
__device__ __forceinline__ float row_shr(float x, float fill) {
    return __builtin_bit_cast(float, __builtin_amdgcn_update_dpp(__builtin_bit_cast(int, fill),
                                                                 __builtin_bit_cast(int, x), 0x110 + N, 0xF, 0xF, false));
}
// value of lane (i + n) of the same row
template <int N>
__device__ __forceinline__ float row_shl(float x, float fill) {
    return __builtin_bit_cast(float, __builtin_amdgcn_update_dpp(__builtin_bit_cast(int, fill),
                                                                 __builtin_bit_cast(int, x), 0x100 + N, 0xF, 0xF, false));
}
template <int N>
__device__ __forceinline__ Map3 map_shr(const Map3 &m) { return Map3{row_shr<N>(m.R, 1.f), row_shr<N>(m.X, 0.f), row_shr<N>(m.H, 1.f)}; }
template <int N>
__device__ __forceinline__ Map3 map_shl(const Map3 &m) { return Map3{row_shl<N>(m.R, 1.f), row_shl<N>(m.X, 0.f), row_shl<N>(m.H, 1.f)}; }
__device__ __forceinline__ float coef_readlane(float x, int lane) {
    return __builtin_bit_cast(float, __builtin_amdgcn_readlane(__builtin_bit_cast(int, x), lane));
}

// One whole wave, lane = token of the chunk; alpha, theta, eta are that token's gates (any value
// beyond L).  Fills cc; the caller orders it against the readers with a barrier.
__device__ __forceinline__ void coef_scan(ChunkCoef &cc, float alpha, float theta, float eta, int L) {
    const int t = threadIdx.x & 63;
    const bool in = t < L;
    const float keep = in ? 1.f - alpha : 1.f, et = in ? eta : 0.f;
    cc.keep[t] = keep;
    cc.eta[t] = et;
    cc.th[t] = in ? theta : 0.f;
    const Map3 g = in ? Map3{keep, et, et} : map_identity();
    // prefixes inside the block: head_t = g_t ... g_(16 T)
    Map3 hd = g;
    hd = compose(hd, map_shr<1>(hd));
    hd = compose(hd, map_shr<2>(hd));
    hd = compose(hd, map_shr<4>(hd));
    hd = compose(hd, map_shr<8>(hd));
    // suffixes inside the block: sf_j = g_(16 J + 15) ... g_j; tail_j = sf_(j+1)
    Map3 sf = g;
    sf = compose(map_shl<1>(sf), sf);
    sf = compose(map_shl<2>(sf), sf);
    sf = compose(map_shl<4>(sf), sf);
    sf = compose(map_shl<8>(sf), sf);
    const Map3 tl = map_shl<1>(sf);
    // whole blocks (uniform values)
    Map3 blk[4];
#pragma unroll
    for (int b = 0; b < 4; b++)
        blk[b] = Map3{coef_readlane(hd.R, 16 * b + 15), coef_readlane(hd.X, 16 * b + 15), coef_readlane(hd.H, 16 * b + 15)};
    const Map3 m02 = blk[1], m13 = blk[2], m03 = compose(blk[2], blk[1]);
    const Map3 pre1 = blk[0], pre2 = compose(blk[1], blk[0]), pre3 = compose(blk[2], pre2);
    const Map3 post2 = blk[3], post1 = compose(blk[3], blk[2]), post0 = compose(post1, blk[1]);
    const int T = t >> 4;
    const Map3 pre = T == 0 ? map_identity() : (T == 1 ? pre1 : (T == 2 ? pre2 : pre3));
    const Map3 post = T == 3 ? map_identity() : (T == 2 ? post2 : (T == 1 ? post1 : post0));
    const Map3 pf = compose(hd, pre), sx = compose(post, tl);
    cc.hR[t] = hd.R; cc.hX[t] = hd.X; cc.hH[t] = hd.H;
    cc.zc[t] = tl.R + tl.X; cc.zh[t] = tl.H; cc.zr[t] = tl.R;
    cc.a[t] = pf.R; cc.beta[t] = pf.X; cc.h[t] = pf.H;
    cc.cl[t] = sx.R + sx.X; cc.bl[t] = sx.H; cc.rl[t] = sx.R;
    if (t == 63) { cc.last[0] = pf.R; cc.last[1] = pf.X; cc.last[2] = pf.H; cc.last[3] = 0.f; }
    if (t < 6) {
        const Map3 id = map_identity();
        const Map3 m = t == 1 ? m02 : (t == 2 ? m03 : (t == 4 ? m13 : id));
        cc.mid[t][0] = m.R; cc.mid[t][1] = m.X; cc.mid[t][2] = m.H; cc.mid[t][3] = 0.f;
    }
}

// Which of c, bb, r a tile function returns.
enum CoefKind { COEF_C = 0, COEF_BB = 1, COEF_R = 2 };

// Tile (T, J) in "token-major" order: element i of lane l is the coefficient between
// t = 16 T + 4 (l / 16) + i (row) and j = 16 J + l % 16 (column); zero unless j <= t < L.
template <int KIND>
__device__ __forceinline__ cf32x4 coef_tile_tj(const ChunkCoef &cc, int T, int J, int L) {
    const int l = threadIdx.x & 63, g = l >> 4, c16 = l & 15;
    cf32x4 out = {0.f, 0.f, 0.f, 0.f};
    if (J > T) return out;
    const int j = 16 * J + c16;
    if (J < T) {
        const float *md = cc.mid[mid_index(J, T)];
        const float mR = md[0], mX = md[1], mH = md[2];
        const float zc = cc.zc[j], zh = cc.zh[j], zr = cc.zr[j];
        const cf32x4 hR = *reinterpret_cast<const cf32x4 *>(cc.hR + 16 * T + 4 * g);
        const cf32x4 hX = *reinterpret_cast<const cf32x4 *>(cc.hX + 16 * T + 4 * g);
        const cf32x4 hH = *reinterpret_cast<const cf32x4 *>(cc.hH + 16 * T + 4 * g);
#pragma unroll
        for (int i = 0; i < 4; i++) {
            const float aR = hR[i] * mR;
            float x;
            if (KIND == COEF_C) x = fmaf(aR, zc, fmaf(hR[i], mX, hX[i] * mH) * zh);
            else if (KIND == COEF_BB) x = hH[i] * mH * zh;
            else x = aR * zr;
            out[i] = (16 * T + 4 * g + i < L && j < L) ? x : 0.f;
        }
        return out;
    }
    // same block: run the recurrence from token j upwards, keep the steps this lane owns
    float b = 1.f, c = 1.f, r = 1.f;
#pragma unroll
    for (int u = 0; u < 16; u++) {
        const float kp = cc.keep[16 * T + u], et = cc.eta[16 * T + u];
        const bool after = u > c16;
        if (KIND != COEF_R) b *= after ? et : 1.f;
        if (KIND == COEF_C) c = after ? fmaf(kp, c, b) : c;
        if (KIND == COEF_R) r *= after ? kp : 1.f;
        if ((u >> 2) == g) {
            const float x = KIND == COEF_C ? c : (KIND == COEF_BB ? b : r);
            out[u & 3] = (u >= c16 && 16 * T + u < L && j < L) ? x : 0.f;
        }
    }
    return out;
}

// Tile (J, T) in "source-major" order: element i of lane l is the coefficient between
// j = 16 J + 4 (l / 16) + i (row) and t = 16 T + l % 16 (column); zero unless j <= t < L.
template <int KIND>
__device__ __forceinline__ cf32x4 coef_tile_jt(const ChunkCoef &cc, int J, int T, int L) {
    const int l = threadIdx.x & 63, g = l >> 4, c16 = l & 15;
    cf32x4 out = {0.f, 0.f, 0.f, 0.f};
    if (J > T) return out;
    const int t = 16 * T + c16;
    if (J < T) {
        const float *md = cc.mid[mid_index(J, T)];
        const float mR = md[0], mX = md[1], mH = md[2];
        const float hR = cc.hR[t], hX = cc.hX[t], hH = cc.hH[t];
        const float aR = hR * mR, aX = fmaf(hR, mX, hX * mH), aH = hH * mH;
        const cf32x4 zc = *reinterpret_cast<const cf32x4 *>(cc.zc + 16 * J + 4 * g);
        const cf32x4 zh = *reinterpret_cast<const cf32x4 *>(cc.zh + 16 * J + 4 * g);
        const cf32x4 zr = *reinterpret_cast<const cf32x4 *>(cc.zr + 16 * J + 4 * g);
#pragma unroll
        for (int i = 0; i < 4; i++) {
            float x;
            if (KIND == COEF_C) x = fmaf(aR, zc[i], aX * zh[i]);
            else if (KIND == COEF_BB) x = aH * zh[i];
            else x = aR * zr[i];
            out[i] = (t < L && 16 * J + 4 * g + i < L) ? x : 0.f;
        }
        return out;
    }
    // same block: four recurrences (sources j = 4 g + i), each from j + 1 up to this lane's t
    float b[4] = {1.f, 1.f, 1.f, 1.f}, c[4] = {1.f, 1.f, 1.f, 1.f}, r[4] = {1.f, 1.f, 1.f, 1.f};
#pragma unroll
    for (int u = 1; u < 16; u++) {
        const float kp = cc.keep[16 * T + u], et = cc.eta[16 * T + u];
#pragma unroll
        for (int i = 0; i < 4; i++) {
            const bool on = u > 4 * g + i && u <= c16;
            if (KIND != COEF_R) b[i] *= on ? et : 1.f;
            if (KIND == COEF_C) c[i] = on ? fmaf(kp, c[i], b[i]) : c[i];
            if (KIND == COEF_R) r[i] *= on ? kp : 1.f;
        }
    }
#pragma unroll
    for (int i = 0; i < 4; i++) {
        const float x = KIND == COEF_C ? c[i] : (KIND == COEF_BB ? b[i] : r[i]);
        out[i] = (4 * g + i <= c16 && t < L && 16 * J + 4 * g + i < L) ? x : 0.f;
    }
    return out;
}


// ── Coefficient tables written to HBM by a pre-pass (one wave per chunk) ──
// The vectors of a chunk from two scans of composed maps instead of 64-step loops:
//   a, beta, h = R, X, H of G(0..t);  cl, bl = R + X, H of G(t+1..63)   (tokens beyond L: identity map)
// and what its table is formed from: head_t, tail_t, and the maps of the two middle blocks.
struct ChunkVectors {
    float a, beta, h, cl, bl;
    Map3 head, tail, mid1, mid2;
};
__device__ __forceinline__ ChunkVectors coef_vectors(float keep, float et, bool in) {
    const int t = threadIdx.x & 63;
    const Map3 g = in ? Map3{keep, et, et} : map_identity();
    Map3 hd = g;
    hd = compose(hd, map_shr<1>(hd));
    hd = compose(hd, map_shr<2>(hd));
    hd = compose(hd, map_shr<4>(hd));
    hd = compose(hd, map_shr<8>(hd));
    Map3 sf = g;
    sf = compose(map_shl<1>(sf), sf);
    sf = compose(map_shl<2>(sf), sf);
    sf = compose(map_shl<4>(sf), sf);
    sf = compose(map_shl<8>(sf), sf);
    const Map3 tl = map_shl<1>(sf);
    Map3 blk[4];
#pragma unroll
    for (int b = 0; b < 4; b++)
        blk[b] = Map3{coef_readlane(hd.R, 16 * b + 15), coef_readlane(hd.X, 16 * b + 15), coef_readlane(hd.H, 16 * b + 15)};
    const Map3 pre1 = blk[0], pre2 = compose(blk[1], blk[0]), pre3 = compose(blk[2], pre2);
    const Map3 post2 = blk[3], post1 = compose(blk[3], blk[2]), post0 = compose(post1, blk[1]);
    const int T = t >> 4;
    const Map3 pre = T == 0 ? map_identity() : (T == 1 ? pre1 : (T == 2 ? pre2 : pre3));
    const Map3 post = T == 3 ? map_identity() : (T == 2 ? post2 : (T == 1 ? post1 : post0));
    const Map3 pf = compose(hd, pre), sx = compose(post, tl);
    return ChunkVectors{pf.R, pf.X, pf.H, sx.R + sx.X, sx.H, hd, tl, blk[1], blk[2]};
}

// The table scale_j c[t][j] of one chunk, tile by tile of 16 x 16, without a recurrence over its 64 tokens: tiles below the diagonal are head_t . mid . tail_j, two multiply-adds an entry, and the four tiles on it one
// recurrence of 16 steps, a lane per column, whose gates come from the neighbouring lanes.  What bounds the pre-passes then is
// the 10 KB that a chunk's ten tiles take in HBM: 8192 chunks in 19 and 18 us, 5.2 TB/s (27 and 37 when a lane walked down its
// column, 64 steps, in 18 KB of LDS that let eight waves onto a compute unit), 16384 in 42 and 41 (50 and 64).
constexpr int kDiagLd = 20;   // row stride (floats) of the diagonal tiles
struct ChunkTable {
    float hR[64], hX[64];             // head_t, zero beyond L
    float zc[64], zh[64];             // tail_j times the column's factor
    float diag[(64 + 16) * kDiagLd];  // [t][j % 16]; the last 16 rows take what runs past the chunk's end
};
// once per wave, before the first chunk: the part above the diagonal of the first tile, which no chunk writes
__device__ __forceinline__ void chunk_table_clear(ChunkTable &ct) {
    for (int e = threadIdx.x & 63; e < 16 * kDiagLd; e += 64) ct.diag[e] = 0.f;
}
// value of lane (i + N) of the same 16-lane row, zero behind its end
template <int N>
__device__ __forceinline__ float row_ahead(float x) {
    return __builtin_bit_cast(float, __builtin_amdgcn_update_dpp(0, __builtin_bit_cast(int, x), 0x100 + N, 0xF, 0xF, true));
}
template <int I>
__device__ __forceinline__ void diag_steps(float *dst, float keep, float et, float b, float c) {
    if constexpr (I < 16) {
        b *= row_ahead<I>(et);
        c = fmaf(row_ahead<I>(keep), c, b);
        dst[I * kDiagLd] = c;
        diag_steps<I + 1>(dst, keep, et, b, c);
    }
}
// One wave, lane = token; keep and et are zero or the identity's beyond L, scale zero there.
// A lane whose block has ended goes on with gates of zero: it writes zeros, and they land in the part of the next tile that is
// above the diagonal (token j + i of the next block, column j: i < 16 leaves it above), which needs them.
__device__ __forceinline__ void chunk_table_build(ChunkTable &ct, const ChunkVectors &cv, float keep, float et, float scale, int L) {
    const int t = threadIdx.x & 63;
    const bool in = t < L;
    wave_lds_order();   // the chunk before has been read
    ct.hR[t] = in ? cv.head.R : 0.f;
    ct.hX[t] = in ? cv.head.X : 0.f;
    ct.zc[t] = scale * (cv.tail.R + cv.tail.X);
    ct.zh[t] = scale * cv.tail.H;
    float *dst = ct.diag + t * kDiagLd + (t & 15);
    dst[0] = scale;
    diag_steps<1>(dst, in ? keep : 0.f, in ? et : 0.f, scale, scale);
    wave_lds_order();
}
// what stands between blocks J and T > J
template <int T, int J>
__device__ __forceinline__ Map3 map_between(const ChunkVectors &cv) {
    if constexpr (T == 2 && J == 0) return cv.mid1;
    else if constexpr (T == 3 && J == 1) return cv.mid2;
    else if constexpr (T == 3 && J == 0) return compose(cv.mid2, cv.mid1);
    else return map_identity();
}
// Tile (T, J <= T): element i of lane l at t = 16 T + l % 16, j = 16 J + 4 (l / 16) + i (BY_TOKEN = false), or at
// t = 16 T + 4 (l / 16) + i, j = 16 J + l % 16 (BY_TOKEN = true).
template <bool BY_TOKEN, int T, int J>
__device__ __forceinline__ cf32x4 chunk_table_tile(const ChunkTable &ct, const ChunkVectors &cv) {
    const int l = threadIdx.x & 63, one = l & 15, four = 4 * (l >> 4);
    auto four_of = [&](const float *p) { return *reinterpret_cast<const cf32x4 *>(p + four); };
    if constexpr (T == J) {
        const float *p = ct.diag + 16 * T * kDiagLd;
        if constexpr (!BY_TOKEN) return four_of(p + one * kDiagLd);
        p += four * kDiagLd + one;
        return cf32x4{p[0], p[kDiagLd], p[2 * kDiagLd], p[3 * kDiagLd]};
    } else {
        const Map3 m = map_between<T, J>(cv);
        cf32x4 out;
        if constexpr (BY_TOKEN) {
            const cf32x4 hR = four_of(ct.hR + 16 * T), hX = four_of(ct.hX + 16 * T);
            const float zc = ct.zc[16 * J + one], zh = ct.zh[16 * J + one];
            const float pc = fmaf(m.R, zc, m.X * zh), ph = m.H * zh;   // mid . tail: (R + X, H) of it is (pc, ph)
#pragma unroll
            for (int i = 0; i < 4; i++) out[i] = fmaf(hR[i], pc, hX[i] * ph);
        } else {
            const float hR = ct.hR[16 * T + one], hX = ct.hX[16 * T + one];
            const float aR = hR * m.R, aX = fmaf(hR, m.X, hX * m.H);
            const cf32x4 zc = four_of(ct.zc + 16 * J), zh = four_of(ct.zh + 16 * J);
#pragma unroll
            for (int i = 0; i < 4; i++) out[i] = fmaf(aR, zc[i], aX * zh[i]);
        }
        return out;
    }
}
// f(T, J, tile) for the ten tiles on or below the diagonal
template <bool BY_TOKEN, int T, int J, class F>
__device__ __forceinline__ void chunk_table_tiles(const ChunkTable &ct, const ChunkVectors &cv, F &&f) {
    f(T, J, chunk_table_tile<BY_TOKEN, T, J>(ct, cv));
    if constexpr (J < T) chunk_table_tiles<BY_TOKEN, T, J + 1>(ct, cv, f);
    else if constexpr (T < 3) chunk_table_tiles<BY_TOKEN, T + 1, 0>(ct, cv, f);
}

}  // namespace
}  // namespace nlh
