// Frozen-M0 chunkwise Titans / Delta rule on bf16 tokens with the memory resident on chip.
//
// Semantics are those of core/kernels/titans_chunkwise_forward.cu / _backward.cu with
// error_clip and the M-norm projection off (see chunkwise_mm.hip for the matrix form:
// coefficients r, bb, c, a, beta, h and W[t][j] = -theta_j c[t][j]).
//
// One workgroup owns one chain (batch element x head) and walks its chunks in order.  The
// fp32 master copy of M and S lives in registers (accumulator layout of the matrix cores),
// a bf16 hi/lo split of it in LDS as the operand of the products of the next chunk, so a
// state never travels through HBM between chunks; HBM sees each token once (k, v, q in,
// y out) plus one state snapshot per chunk for the backward.  Per chunk, with
// E = K M0^T - V,  P = Q K^T:
//   Y  = a.(Q M0^T) + beta.(Q S0^T) + (W.P) E
//   M' = a_L M0 + beta_L S0 + (E.wM)^T K        S' = h_L S0 + (E.wS)^T K
// All products run on v_mfma_f32_16x16x32_bf16.  k, v, q are exact in bf16; every fp32
// operand (states, E, W.P) enters as a hi + lo pair of bf16 (16 mantissa bits), the
// accumulation is fp32.
//
// Eight waves compute, one 16x32 output strip each per product.  The coefficients depend on
// the gates only: a chunk-parallel kernel runs their 64-step scalar recurrences up front and
// leaves W in the accumulator order of the chain kernel, which prefetches one chunk ahead.
#include <hip/hip_runtime.h>
#include <stdint.h>

#include "bf16_tiles.h"
#include "chunk_coef.h"
#include "chunkwise_chain.h"
#include "lane_ops.h"
#include "runtime.h"

namespace nlh {
namespace {

constexpr int kChainThr = 512;     // 8 waves for 32 rows of a chain

// Work split of the eight waves: a 64x64 product is four 32x32 blocks (2x2 tiles of 16x16; an
// A or B operand read from LDS then serves two tiles).  Wave w works on block bi = w%4 with
// origin (32 (bi/2), 32 (bi%2)); waves 0..3 (group X) compute E and then Y, waves 4..7
// (group Y) compute W.P and then the state update, and hold the fp32 master state.
//
// Per-chunk coefficients in HBM, written by cw_coef_kernel:
//   table [chunk][block bi][rt][ct][lane l][r]: W[t][j] = -theta_j c[t][j] (zero outside j <= t < L)
//         at j = 32 (bi/2) + 16 rt + 4 (l/16) + r, t = 32 (bi%2) + 16 ct + l%16: the order in which
//         lane l of a group-Y wave holds P^T; tiles entirely above the diagonal are neither
//         written nor read
//   vecs  [chunk][kVecFloats]: a_t, beta_t, wM_j = -theta_j c[L-1][j], wS_j = -theta_j bb[j][L-1],
//         then a_L, beta_L, h_L, one unused float and four zeros
constexpr int kTableFloats = CW * CW;
constexpr int kVecFloats = 4 * CW + 16;
__device__ __forceinline__ bool tile_live(int bi, int rt, int ct) { return 2 * (bi & 1) + ct >= 2 * (bi >> 1) + rt; }

// Coefficients of one chunk from its gates: one wave per chunk, lane = token.  The vectors come from two scans
// of composed maps, the table tile by tile in the consumers' order (chunk_table_tiles), as 16-byte stores of consecutive lanes.
template <bool HAS_S>
__global__ __launch_bounds__(64) void cw_coef_kernel(const float *__restrict__ alpha,
                                                     const float *__restrict__ theta,
                                                     const float *__restrict__ eta, float *__restrict__ table,
                                                     float *__restrict__ vecs, int s, int C, int nc, int nchunks, int per_wave) {
    __shared__ __align__(16) ChunkTable ct;
    chunk_table_clear(ct);
    const int j = threadIdx.x, first = blockIdx.x * per_wave, last = min(nchunks, first + per_wave);
    auto gates_of = [&](int chunk) {
        const int chain = chunk / nc, t0 = (chunk % nc) * C;
        return fetch_gates<HAS_S>(alpha, theta, eta, (size_t)chain * s + t0, min(C, s - t0));
    };
    // a wave walks over a few chunks with the next chunk's gates in flight: a wave per chunk would spend most of
    // its life waiting for its three loads
    Gates gn = gates_of(first);
    for (int chunk = first; chunk < last; chunk++) {
        const int L = min(C, s - (chunk % nc) * C);
        const Gates g = gn;
        gn = gates_of(min(chunk + 1, last - 1));
        const bool jv = j < L;
        const float keep = 1.f - g.al, et = g.et, nth = -g.th;   // 1, 0, 0 beyond L
        const ChunkVectors cv = coef_vectors(keep, et, jv);
        float *vo = vecs + (size_t)chunk * kVecFloats;
        vo[j] = jv ? cv.a : 0.f;
        vo[CW + j] = jv ? cv.beta : 0.f;
        vo[2 * CW + j] = nth * cv.cl;
        vo[3 * CW + j] = nth * cv.bl;
        if (j == 63) { vo[4 * CW] = cv.a; vo[4 * CW + 1] = cv.beta; vo[4 * CW + 2] = cv.h; }   // the values at token L - 1
        if (j < 4) vo[4 * CW + 4 + j] = 0.f;   // zero pad: what tiles of W above the diagonal read
        chunk_table_build(ct, cv, keep, et, nth, L);
        float *out = table + (size_t)chunk * kTableFloats;
        chunk_table_tiles<false, 0, 0>(ct, cv, [&](int T, int J, const cf32x4 &w) __attribute__((always_inline)) {
            const int tile = ((J >> 1) * 2 + (T >> 1)) * 4 + (J & 1) * 2 + (T & 1);   // (bi, rt, ct) of the layout above
            *reinterpret_cast<cf32x4 *>(out + (tile * 64 + j) * 4) = w;
        });
    }
}

// Pipeline of one chunk step.  Every global load of chunk c+1 (tokens, W, coefficient vectors)
// is issued at the top of step c and first touched at the bottom of step c, after the matrix
// work and before the stores of step c, so no wait inside a step ever meets a load in flight
// or a store just issued.  The requests and their landing are unconditional (past the end they
// repeat the last chunk): memory waits are placed per program point, not per path.
//
// The rows of M and S never mix, so a chain is split over two workgroups of 32 rows each
// (chain_half_of_block: both halves of a chain share an XCD's L2 and are dispatched together
// for K, Q and W).  Waves 0..3 (group X): E, then Y^T, one 16-token strip each.  Waves 4..7
// (group Y): one 32x32 block of W.P each, then one 16-column strip of the transposed state
// update; they hold the fp32 master state.
// H = 2: one workgroup of sixteen waves has both halves, eight waves each, and its group Y waves a 32 x 16 block of W.P; K, Q and W
// are fetched, and W.P formed, once, and four waves on a SIMD hide each other's latencies.  256 chains of 4096 tokens: 393 -> 313 us.
// TRACK: also leaves the per-token error norms and the chunk-start state norms of ChainTracks behind.
template <bool HAS_S, bool TRACK, int H>
__global__ __launch_bounds__(H *kChainThr) void cw_chain_fwd_kernel(
    const u16 *__restrict__ k, const u16 *__restrict__ v, const u16 *__restrict__ q,
    const float *__restrict__ table, const float *__restrict__ vecs, const float *m_initial, const float *s_initial,
    float *__restrict__ m_states, float *__restrict__ s_states,
    float *__restrict__ y, int s, int C, int nc, int batch, HeadRows yr, ChainTracks tr, ChainFinal fin) {
    constexpr int HMAT = 32 * H * 64;   // this workgroup's rows of a matrix
    constexpr int CT = 2 / H;           // 16-token tiles of a group Y wave's block of P^T
    extern __shared__ __align__(16) unsigned char smem_raw[];
    u16 *Kr = reinterpret_cast<u16 *>(smem_raw);   // K [t][c]
    u16 *Kt0 = Kr + kPerm, *Kt1 = Kt0 + kPerm;       // K^T [c][t] of this chunk / V [t][i] until K^T of the next lands
    u16 *Qr0 = Kt1 + kPerm, *Qr1 = Qr0 + kPerm;      // Q [t][c], alternating between chunks
    u16 *WPh = Qr1 + kPerm, *WPl = WPh + kPerm;      // W.P [t][j]
    u16 *Mh = WPl + kPerm, *Ml = Mh + HMAT;         // chunk-start M [i][c], this workgroup's rows, hi / lo
    u16 *Sh = Ml + HMAT, *Sl = Sh + HMAT;          // chunk-start S
    u16 *Eh = Sl + HMAT, *El = Eh + HMAT;          // E^T [i][t]
    u16 *EMh = El + HMAT, *EMl = EMh + HMAT;       // (E.wM)^T
    u16 *ESh = EMl + HMAT, *ESl = ESh + HMAT;      // (E.wS)^T
    float *cvec = reinterpret_cast<float *>(ESl + HMAT);   // a, beta, wM, wS [64] each, then a_L, beta_L, h_L

    const int tid = threadIdx.x, w = H == 1 ? tid >> 6 : __builtin_amdgcn_readfirstlane(tid >> 6), l = tid & 63, g = l >> 4, r16 = l & 15, first_l = l;
    int chain, half;   // of the wave's rows
    if (H == 1) chain_half_of_block(batch, chain, half);
    else { chain = blockIdx.x; half = (w >> 2) & 1; }
    const int i0 = 32 * half, il = H == 1 ? 0 : i0;   // first row; and in LDS
    const bool grpX = w < 4 * H;
    const int bi = w & 3, bm = 32 * (bi >> 1), bn = 32 * (bi & 1);   // group Y: 32x32 block of P^T; group X: strip bi
    const size_t chain_tok = (size_t)chain * s;
    const size_t state0 = (size_t)chain * (nc + 1) * HD * HD;
    const size_t y_off = yr.offset(chain);

    // -V enters E = K M0^T - V as one more step of the product: A = V (rows t, this half's 32
    // columns as contraction), B = -identity: column 16 ct + l%16 meets contraction index 8 (l/16) + e.
    bf16x8 negI[2];
#pragma unroll
    for (int ct = 0; ct < 2; ct++) {
        const int hit = 16 * ct + r16 - 8 * g;   // element of this lane's eight that is -1 (bf16 0xBF80), if in 0..7
        uint4 bits;
        bits.x = (hit == 0 ? 0xBF80u : 0u) | (hit == 1 ? 0xBF800000u : 0u);
        bits.y = (hit == 2 ? 0xBF80u : 0u) | (hit == 3 ? 0xBF800000u : 0u);
        bits.z = (hit == 4 ? 0xBF80u : 0u) | (hit == 5 ? 0xBF800000u : 0u);
        bits.w = (hit == 6 ? 0xBF80u : 0u) | (hit == 7 ? 0xBF800000u : 0u);
        negI[ct] = __builtin_bit_cast(bf16x8, bits);
    }

    // Registers of the next chunk.  K, Q: row st_t, 8-element block st_cb (16 rows x 64 bytes per
    // wave instruction), with sixteen waves K by the first eight and Q by the others.  V: row vt, columns from vcb of this workgroup's,
    // eight by each of the first 256 threads, or four by each of 1024.  Group Y:
    // W at the accumulator positions of its P^T block.  Threads 0..259: one float of the vectors.
    const int st_t = 16 * (w & 3) + (l & 15), st_cb = 4 * ((w >> 2) & 1) + (l >> 4);
    const int vt = H == 1 ? (tid >> 2) & 63 : tid >> 4, vcb = H == 1 ? (tid & 3) * 8 : (tid & 15) * 4;
    const bool has_k = H == 1 || w < 8, has_q = H == 1 || w >= 8;
    const int ct0 = H == 1 ? 0 : half;   // group Y: first 16-token tile of its block
    uint4 sk, sq, sv;   // with sixteen waves sk is K or Q
    f32x4 wn[2][CT], wc[2][CT];
    float vn = 0.f;
    auto fetch = [&](int c) {
        const int L = min(C, s - c * C);
        const size_t tok = chain_tok + (size_t)c * C;
        const size_t o = (tok + min(st_t, L - 1)) * HD + st_cb * 8;
        if (H == 1) {
            sk = *reinterpret_cast<const uint4 *>(k + o);
            sq = *reinterpret_cast<const uint4 *>(q + o);
        } else {
            sk = *reinterpret_cast<const uint4 *>((has_k ? k : q) + o);
        }
        const u16 *vp = v + (tok + min(vt, L - 1)) * HD + (i0 - il) + vcb;
        if (H == 1) {
            sv = *reinterpret_cast<const uint4 *>(vp);
        } else {
            const uint2 x = *reinterpret_cast<const uint2 *>(vp);
            sv = make_uint4(x.x, x.y, 0, 0);
        }
        const size_t chunk = (size_t)chain * nc + c;
        const float *tb = table + chunk * kTableFloats, *vo = vecs + chunk * kVecFloats;
#pragma unroll
        for (int rt = 0; rt < 2; rt++)
#pragma unroll
            for (int ct = 0; ct < CT; ct++)
                wn[rt][ct] = *reinterpret_cast<const f32x4 *>(
                    (!grpX && tile_live(bi, rt, ct0 + ct)) ? tb + (((bi * 2 + rt) * 2 + ct0 + ct) * 64 + l) * 4 : vo + 4 * CW + 4);
        vn = vo[min(tid, 4 * CW + 3)];
    };
    auto land = [&](int c) {   // wait for the loads here; zero the rows beyond a short chunk
        const int L = min(C, s - c * C);
        if (st_t >= L) { sk = make_uint4(0, 0, 0, 0); if (H == 1) sq = sk; }
        if (vt >= L) sv = make_uint4(0, 0, 0, 0);
#pragma unroll
        for (int rt = 0; rt < 2; rt++)
#pragma unroll
            for (int ct = 0; ct < CT; ct++) wc[rt][ct] = wn[rt][ct];
        // V and the vectors are written to LDS later, behind the stores of this step: pin their
        // arrival to this point
        asm volatile("" : "+v"(sv.x), "+v"(sv.y), "+v"(sv.z), "+v"(sv.w), "+v"(vn));
    };
    auto commit_rows = [&](u16 *dst, const uint4 &x) { *reinterpret_cast<uint4 *>(dst + bf_at(st_t, st_cb * 8)) = x; };
    auto commit_kt = [&](u16 *Kt) {
        const unsigned kw[4] = {sk.x, sk.y, sk.z, sk.w};
#pragma unroll
        for (int i = 0; i < 4; i++) {
            Kt[bf_at(st_cb * 8 + 2 * i, st_t)] = (u16)(kw[i] & 0xffffu);
            Kt[bf_at(st_cb * 8 + 2 * i + 1, st_t)] = (u16)(kw[i] >> 16);
        }
    };
    auto commit_v = [&](u16 *dst) {
        if (H == 2) *reinterpret_cast<uint2 *>(dst + bf_at(vt, vcb)) = make_uint2(sv.x, sv.y);
        else if (tid < 256) *reinterpret_cast<uint4 *>(dst + bf_at(vt, vcb)) = sv;
    };
    auto commit_tokens = [&](u16 *Q, u16 *Kt) {
        if (has_k) commit_rows(Kr, sk);
        if (has_q) commit_rows(Q, H == 1 ? sq : sk);   // whole rows first: K^T leaves in single elements
        if (has_k) commit_kt(Kt);
    };
    auto commit_vecs = [&]() {
        if (tid < 4 * CW + 4) cvec[tid] = vn;
    };

    // fp32 master state (group Y), transposed strip:
    //   Mm[ct][r] = M[i = i0 + 16 ct + l%16][c = 16 bi + 4 (l/16) + r]
    // Group X has no state; it borrows the same registers as accumulators of M0 Q^T and S0 Q^T.
    f32x4 Mm[2], Sm[2];
    auto publish_state = [&](int slot) {   // -> HBM snapshot
#pragma unroll
        for (int ct = 0; ct < 2; ct++) {
            const size_t o = state0 + (size_t)slot * HD * HD + (i0 + 16 * ct + r16) * HD + 16 * bi + 4 * g;
            *reinterpret_cast<f32x4 *>(m_states + o) = Mm[ct];
            if (HAS_S) *reinterpret_cast<f32x4 *>(s_states + o) = Sm[ct];
        }
    };
    auto stage_state = [&]() {             // -> LDS operands of the next chunk
#pragma unroll
        for (int ct = 0; ct < 2; ct++) {
            const int off = bf_at(il + 16 * ct + r16, 16 * bi + 4 * g);
            split_store(Mh, Ml, off, Mm[ct]);
            if (HAS_S) split_store(Sh, Sl, off, Sm[ct]);
        }
    };

    fetch(0);
    if (!grpX) {
#pragma unroll
        for (int ct = 0; ct < 2; ct++) {
            const size_t o = (size_t)chain * HD * HD + (i0 + 16 * ct + r16) * HD + 16 * bi + 4 * g;
            Mm[ct] = *reinterpret_cast<const f32x4 *>(m_initial + o);
            Sm[ct] = HAS_S ? *reinterpret_cast<const f32x4 *>(s_initial + o) : zero4();
        }
        publish_state(0);
        stage_state();
    }
    land(0);
    commit_tokens(Qr0, Kt0);
    commit_v(Kt1);
    commit_vecs();
    __syncthreads();

    for (int c = 0; c < nc; c++) {
        const int t0 = c * C, L = min(C, s - t0);
        const size_t tok = chain_tok + t0;
        // The thread's place through an opaque copy, once per chunk: with sixteen waves the LDS addresses made of it do not fit
        // the registers across the sequence.
        int me = first_l;
        if (H == 2) asm volatile("" : "+v"(me));
        const int l = me, g = l >> 4, r16 = l & 15;
        // this chunk: Q in Qc, K^T in Kc, V in Kn (until K^T of the next chunk replaces it)
        u16 *Qc = (c & 1) ? Qr1 : Qr0, *Kc = (c & 1) ? Kt1 : Kt0;
        u16 *Qn = (c & 1) ? Qr0 : Qr1, *Kn = (c & 1) ? Kt0 : Kt1;
        fetch(min(c + 1, nc - 1));
        if (TRACK && !grpX) {   // sums of squares of this wave's part of the chunk-start states
            float msq = 0.f, ssq = 0.f;
#pragma unroll
            for (int ct = 0; ct < 2; ct++)
#pragma unroll
                for (int e = 0; e < 4; e++) {
                    msq = fmaf(Mm[ct][e], Mm[ct][e], msq);
                    if (HAS_S) ssq = fmaf(Sm[ct][e], Sm[ct][e], ssq);
                }
            msq = wave_allreduce(msq);
            ssq = wave_allreduce(ssq);
            if (l == 0)
                *reinterpret_cast<float2 *>(tr.nrm + ((((size_t)chain * nc + c) * 2 + half) * 4 + bi) * 2) = make_float2(msq, ssq);
        }
        // ── first half: E^T, (E.wM)^T, (E.wS)^T (group X) and W.P (group Y) ──
        if (grpX) {
            // E[t][i]: rows t = 16 bi .., columns i = 16 ct ..
            const bf16x8 aK[2] = {ld_perm(Kr, 16 * bi, 0, l), ld_perm(Kr, 16 * bi, 1, l)};
            const bf16x8 aV = ld_perm(Kn, 16 * bi, H == 1 ? 0 : half, l);
            const f32x4 wm = *reinterpret_cast<const f32x4 *>(cvec + 2 * CW + 16 * bi + 4 * g);
            const f32x4 wsv = *reinterpret_cast<const f32x4 *>(cvec + 3 * CW + 16 * bi + 4 * g);
            f32x4 esq = zero4();
#pragma unroll
            for (int ct = 0; ct < 2; ct++) {
                f32x4 e = zero4();
#pragma unroll
                for (int ks = 0; ks < 2; ks++) {
                    e = mfma32(aK[ks], ld_perm(Mh, il + 16 * ct, ks, l), e);
                    e = mfma32(aK[ks], ld_perm(Ml, il + 16 * ct, ks, l), e);
                }
                e = mfma32(aV, negI[ct], e);
                if (TRACK) esq += e * e;
                const int off = bf_at(il + 16 * ct + r16, 16 * bi + 4 * g);   // [i][t .. t+3]
                split_store(Eh, El, off, e);
                split_store(EMh, EMl, off, e * wm);
                if (HAS_S) split_store(ESh, ESl, off, e * wsv);
            }
            if (TRACK) {   // a lane holds tokens 16 bi + 4 g .. + 3 of rows 16 ct + l % 16: sum over the 16 lanes of the group
#pragma unroll
                for (int e = 0; e < 4; e++) esq[e] = group_allreduce<16>(esq[e]);
                if (r16 == 0)
                    *reinterpret_cast<f32x4 *>(tr.e2 + (((size_t)chain * 2 + half) * nc + c) * CW + 16 * bi + 4 * g) = esq;
            }
        } else {
            bf16x8 aK[2][2];
#pragma unroll
            for (int rt = 0; rt < 2; rt++)
#pragma unroll
                for (int ks = 0; ks < 2; ks++) aK[rt][ks] = ld_perm(Kr, bm + 16 * rt, ks, l);
            f32x4 acc[2][CT];
#pragma unroll
            for (int rt = 0; rt < 2; rt++)
#pragma unroll
                for (int ct = 0; ct < CT; ct++) acc[rt][ct] = zero4();
#pragma unroll
            for (int ks = 0; ks < 2; ks++)
#pragma unroll
                for (int ct = 0; ct < CT; ct++) {
                    const bf16x8 bq = ld_perm(Qc, bn + 16 * (ct0 + ct), ks, l);
#pragma unroll
                    for (int rt = 0; rt < 2; rt++)     // P^T[j][t]: rows j, columns t
                        acc[rt][ct] = mfma32(aK[rt][ks], bq, acc[rt][ct]);
                }
#pragma unroll
            for (int rt = 0; rt < 2; rt++)
#pragma unroll
                for (int ct = 0; ct < CT; ct++)         // [t][j .. j+3]
                    split_store(WPh, WPl, bf_at(bn + 16 * (ct0 + ct) + r16, bm + 16 * rt + 4 * g),
                                wc[rt][ct] * acc[rt][ct]);
        }
        __syncthreads();
        // ── second half: Y^T (group X) and the state update (group Y) ──
        f32x4 y2[2] = {zero4(), zero4()};   // group X: E^T (W.P)^T, then the finished Y^T; group Y: unused
        if (grpX) {
            // Y^T[i][t]: rows i = 16 rt .., columns t = 16 bi ..: a lane ends up with four consecutive
            // i of one token
            f32x4(&y0)[2] = Mm, (&y1)[2] = Sm;
            y0[0] = y0[1] = y1[0] = y1[1] = zero4();
#pragma unroll
            for (int ks = 0; ks < 2; ks++) {
                const bf16x8 bQ = ld_perm(Qc, 16 * bi, ks, l), bWh = ld_perm(WPh, 16 * bi, ks, l), bWl = ld_perm(WPl, 16 * bi, ks, l);
#pragma unroll
                for (int rt = 0; rt < 2; rt++) {
                    const bf16x8 eh = ld_perm(Eh, il + 16 * rt, ks, l);
                    y0[rt] = mfma32(ld_perm(Mh, il + 16 * rt, ks, l), bQ, y0[rt]);
                    y0[rt] = mfma32(ld_perm(Ml, il + 16 * rt, ks, l), bQ, y0[rt]);
                    y2[rt] = mfma32(eh, bWh, y2[rt]);
                    y2[rt] = mfma32(eh, bWl, y2[rt]);
                    y2[rt] = mfma32(ld_perm(El, il + 16 * rt, ks, l), bWh, y2[rt]);
                    if (HAS_S) {
                        y1[rt] = mfma32(ld_perm(Sh, il + 16 * rt, ks, l), bQ, y1[rt]);
                        y1[rt] = mfma32(ld_perm(Sl, il + 16 * rt, ks, l), bQ, y1[rt]);
                    }
                }
            }
            const float at = cvec[16 * bi + r16], bt = cvec[CW + 16 * bi + r16];
#pragma unroll
            for (int rt = 0; rt < 2; rt++) y2[rt] += at * y0[rt] + bt * y1[rt];
        } else {
            // transposed state strip: rows c = 16 bi .., columns i = 16 ct ..
            f32x4 am[2] = {zero4(), zero4()}, as[2] = {zero4(), zero4()};
#pragma unroll
            for (int ks = 0; ks < 2; ks++) {
                const bf16x8 aKt = ld_perm(Kc, 16 * bi, ks, l);
#pragma unroll
                for (int ct = 0; ct < 2; ct++) {
                    am[ct] = mfma32(aKt, ld_perm(EMh, il + 16 * ct, ks, l), am[ct]);
                    am[ct] = mfma32(aKt, ld_perm(EMl, il + 16 * ct, ks, l), am[ct]);
                    if (HAS_S) {
                        as[ct] = mfma32(aKt, ld_perm(ESh, il + 16 * ct, ks, l), as[ct]);
                        as[ct] = mfma32(aKt, ld_perm(ESl, il + 16 * ct, ks, l), as[ct]);
                    }
                }
            }
            const float aL = cvec[4 * CW], betaL = cvec[4 * CW + 1], hL = cvec[4 * CW + 2];
#pragma unroll
            for (int ct = 0; ct < 2; ct++) {
                Mm[ct] = aL * Mm[ct] + betaL * Sm[ct] + am[ct];
                if (HAS_S) Sm[ct] = hL * Sm[ct] + as[ct];
            }
        }
        // tokens of the next chunk land: K and V of this one are no longer read
        land(min(c + 1, nc - 1));
        commit_tokens(Qn, Kn);
        // results of this chunk leave
        if (grpX) {
            const int t = 16 * bi + r16;
            if (t < L) {
#pragma unroll
                for (int rt = 0; rt < 2; rt++)
                    *reinterpret_cast<f32x4 *>(y + y_off + (size_t)(t0 + t) * yr.row_stride + i0 + 16 * rt + 4 * g) = y2[rt];
            }
        } else {
            publish_state(c + 1);
        }
        __syncthreads();
        if (!grpX) stage_state();
        commit_v(Kc);   // K^T of this chunk is no longer read
        commit_vecs();
        __syncthreads();
    }
    if (!grpX && fin.m) {   // may be the initial states: this thread has read its part of those
#pragma unroll
        for (int ct = 0; ct < 2; ct++) {
            const size_t o = (size_t)chain * HD * HD + (i0 + 16 * ct + r16) * HD + 16 * bi + 4 * g;
            *reinterpret_cast<f32x4 *>(fin.m + o) = Mm[ct];
            if (HAS_S) *reinterpret_cast<f32x4 *>(fin.s + o) = Sm[ct];
        }
    }
}

constexpr size_t chain_fwd_lds(int h) { return (7 * kPerm + 10 * 32 * h * 64) * sizeof(u16) + (4 * CW + 4) * sizeof(float); }

template <bool HAS_S, bool TRACK, int H>
void launch_chain(const u16 *k, const u16 *v, const u16 *q, const float *table, const float *vecs, const float *m_initial,
                  const float *s_initial, float *m_states, float *s_states, float *y, int seq_len, int chunk_size, int nc, int batch,
                  const HeadRows &yr, const ChainTracks &tr, const ChainFinal &fin) {
    static bool attr_set = false;
    if (!attr_set) {
        check_hip(hipFuncSetAttribute(reinterpret_cast<const void *>(cw_chain_fwd_kernel<HAS_S, TRACK, H>),
                                      hipFuncAttributeMaxDynamicSharedMemorySize, (int)chain_fwd_lds(H)), "dynamic LDS size");
        attr_set = true;
    }
    KernelTimer kt("cw_chain_fwd_kernel");
    hipLaunchKernelGGL((cw_chain_fwd_kernel<HAS_S, TRACK, H>), dim3(2 / H * batch), dim3(H * kChainThr), chain_fwd_lds(H), stream(), k, v, q,
                       table, vecs, m_initial, s_initial, m_states, s_states, y, seq_len, chunk_size, nc, batch, yr, tr, fin);
}

template <bool HAS_S>
void launch_forward(const char *fn, const u16 *k, const u16 *v, const u16 *q, const float *alpha, const float *theta,
                    const float *eta, const float *m_initial, const float *s_initial, float *m_states,
                    float *s_states, float *y, int seq_len, int batch, int chunk_size, const HeadRows &yr,
                    const ChainTracks *tracks, const ChainFinal &fin) {
    const ErrorScope es;
    const int nc = ceil_div(seq_len, chunk_size), nchunks = batch * nc;
    float *table = scratch(3, (size_t)nchunks * kTableFloats * sizeof(float));
    float *vecs = scratch(4, (size_t)nchunks * kVecFloats * sizeof(float));
    if (es.failed()) return;
    {
        KernelTimer kt("cw_coef_kernel");
        hipLaunchKernelGGL(cw_coef_kernel<HAS_S>, dim3(ceil_div(nchunks, coef_chunks_per_wave(nchunks))), dim3(64), 0, stream(), alpha, theta, eta,
                           table, vecs, seq_len, chunk_size, nc, nchunks,
                           coef_chunks_per_wave(nchunks));
    }
    check_launch("cw_coef_kernel");
    const ChainTracks tr = tracks ? *tracks : ChainTracks{nullptr, nullptr};
    const bool whole = chain_in_one_workgroup(batch);
    auto launch = tracks ? (whole ? launch_chain<HAS_S, true, 2> : launch_chain<HAS_S, true, 1>)
                         : (whole ? launch_chain<HAS_S, false, 2> : launch_chain<HAS_S, false, 1>);
    launch(k, v, q, table, vecs, m_initial, s_initial, m_states, s_states, y, seq_len, chunk_size, nc, batch, yr, tr, fin);
    check_launch(fn);
}

}  // namespace

bool chunkwise_chain_forward_bf16(const char *fn, const uint16_t *k, const uint16_t *v, const uint16_t *q,
                                  const float *alpha, const float *theta, const float *eta, const float *m_initial,
                                  const float *s_initial, float *m_states, float *s_states, float *y, int seq_len,
                                  int d, int batch, int chunk_size, bool has_s, const HeadRows *y_rows,
                                  const ChainTracks *tracks, const ChainFinal *final_states) {
    if (d != HD || chunk_size < 1 || chunk_size > CW || seq_len <= 0 || batch <= 0) return false;
    const HeadRows yr = y_rows ? *y_rows : head_major_rows(seq_len, HD);
    const ChainFinal fin = final_states ? *final_states : ChainFinal{nullptr, nullptr};
    if (has_s)
        launch_forward<true>(fn, k, v, q, alpha, theta, eta, m_initial, s_initial, m_states, s_states, y, seq_len,
                             batch, chunk_size, yr, tracks, fin);
    else
        launch_forward<false>(fn, k, v, q, alpha, theta, nullptr, m_initial, nullptr, m_states, nullptr, y, seq_len,
                              batch, chunk_size, yr, tracks, fin);
    return true;
}

}  // namespace nlh
