// Backward of the frozen-M0 chunkwise Titans / Delta rule on bf16 tokens: the adjoint scan.
//
// dMo, dSo are the adjoints of a chunk's end state; walking the chunks of a chain backwards,
//   dE  = (W.P)^T dY + wM.(K dMo^T) + wS.(K dSo^T)          [token j][row i]
//   dM0 = a_L dMo + (a.dY)^T Q + dE^T K
//   dS0 = beta_L dMo + h_L dSo + (beta.dY)^T Q
// with P = Q K^T, W[t][j] = -theta_j c[t][j], wM_j = -theta_j c[L-1][j], wS_j = -theta_j bb[j][L-1]
// (the adjoint of the chunk map of chunkwise_mm.hip, written without its 64x64 transfer
// matrices).  The rows of dM, dS never mix, so a chain is split over two workgroups of 32 rows
// each; each walks all chunks with its rows of dM and dS in registers (fp32) and, as bf16
// hi + lo pairs, in LDS as operands of the next step.  HBM sees k, q, dY and the coefficient
// table once per step and receives one adjoint snapshot per chunk, in bf16: dm_snap[chain][c] is the
// adjoint of the state at the start of chunk c (slot num_chunks = 0), rounded as the gradient pass
// would round it; slot 0, the gradient of the initial state, leaves in fp32 (dm_first).
//
// Where that takes the fewer rounds (chunkwise_chain.h), one workgroup of sixteen waves has all rows of a chain (H = 2): K, Q
// and the coefficients are fetched, and W.P formed, once, and four waves on a SIMD hide each other's
// latencies.  256 chains of 4096 tokens: 282 -> 243 us.
//
// Every fp32 operand enters the bf16 matrix cores as a hi + lo pair: this path is recurrent.
#include <hip/hip_runtime.h>
#include <stdint.h>

#include "bf16_tiles.h"
#include "chunkwise_chain.h"
#include "chunkwise_grads.h"
#include "runtime.h"

namespace nlh {
namespace {

// Element (token, row) of a [token][32 H rows] bf16 matrix.  32 rows: 64 bytes a token, their halves exchanged with the token's bit 3,
// so that the tokens 0..3 and 8..11 that a transposing read takes together fall on different banks.
template <int H>
__device__ __forceinline__ int dy_at(int t, int i) {
    return H == 2 ? bf_at(t, i) : t * 32 + ((((i >> 3) ^ ((t >> 2) & 2))) << 3) + (i & 7);
}
template <int H>
__device__ __forceinline__ bf16x8 ld_dy_tr(const u16 *X, int row0, int ks, int l) {   // as ld_op_tr
    const int sl = l & 15, k = 32 * ks + 8 * (l >> 4) + (sl >> 2), n = row0 + 4 * (sl & 3);
    return tr_pair(X + dy_at<H>(k, n), X + dy_at<H>(k + 4, n));
}
constexpr int kCvec = 5 * CW + 8;

// The staged inputs of a chunk are K [j][c], Q [t][c], dY, a.dY, beta.dY hi / lo [t][i], and the vectors a, beta, cl, bl, theta
// [64] each, .., h_L.  They exist twice, so that the next step's copy is written while this step's is still in use; with all rows in
// one workgroup dY's exist once: dY is used by a step's first phase only and written in the second for the next step, a.dY and
// beta.dY by the second only and written in the first.
template <int H>
struct AdjointLds {
    static constexpr int HMAT = 32 * H * 64, DYM = 64 * 32 * H, LATE = 2 * kPerm + (H == 1 ? 6 * DYM : 0);
    static constexpr size_t bytes = (2 * kPerm + 6 * HMAT + 2 * LATE + (H == 2 ? 6 * DYM : 0)) * sizeof(u16) + 2 * kCvec * sizeof(float);
};

template <bool HAS_S, int H>
__global__ __launch_bounds__(H *kTileThr) void cw_adjoint_chain_kernel(
    const u16 *__restrict__ k, const u16 *__restrict__ q, const float *__restrict__ d_y,
    const float *__restrict__ tab_b, const float *__restrict__ vecs, u16 *__restrict__ dm_snap,
    u16 *__restrict__ ds_snap, float *__restrict__ dm_first, float *__restrict__ ds_first, int s, int C, int nc, int batch, int tab_floats, int vec_floats, HeadRows dyr) {
    constexpr int HMAT = AdjointLds<H>::HMAT, DYM = AdjointLds<H>::DYM, LATE = AdjointLds<H>::LATE;
    extern __shared__ __align__(16) unsigned char smem_raw[];
    u16 *WPh = reinterpret_cast<u16 *>(smem_raw), *WPl = WPh + kPerm;   // (W.P)^T [j][t]
    u16 *dMh = WPl + kPerm, *dMl = dMh + HMAT;                          // dMo [i][c]
    u16 *dSh = dMl + HMAT, *dSl = dSh + HMAT;                          // dSo [i][c]
    u16 *dEh = dSl + HMAT, *dEl = dEh + HMAT;                          // dE^T [i][j]
    u16 *late = dEl + HMAT, *const dys = late + 2 * LATE;   // dys: dY's, where they exist once
    float *cvecs = reinterpret_cast<float *>(dys + (H == 2 ? 6 * DYM : 0));
    const int tid = threadIdx.x, w = H == 1 ? tid >> 6 : __builtin_amdgcn_readfirstlane(tid >> 6), l = tid & 63, first_l = l;
    auto dy_of = [&](int par) { return H == 2 ? dys : late + par * LATE + 2 * kPerm; };
    int chain = blockIdx.x, half = 0;
    if (H == 1) chain_half_of_block(batch, chain, half);
    const int i0 = 32 * half;
    const size_t chain_tok = (size_t)chain * s, state0 = (size_t)chain * (nc + 1) * HD * HD;
    const size_t dy_off = dyr.offset(chain);
    const int st_t = 16 * (w & 3) + (l & 15), st_cb = 4 * ((w >> 2) & 1) + (l >> 4);   // bf16 tile: row, 8-element block
    const bool has_k = H == 1 || w < 8;                                           // sixteen waves: K by the first eight, Q by the others
    const int yt = tid / (8 * H), yg = tid % (8 * H);                             // dY tile: row t, 4-element block

    // zero what is never written again: tiles of (W.P)^T above the diagonal
    for (int e = tid; e < kPerm / 2; e += H * kTileThr) {
        reinterpret_cast<unsigned *>(WPh)[e] = 0u;
        reinterpret_cast<unsigned *>(WPl)[e] = 0u;
    }

    // registers of the next step (chunk c - 1)
    uint4 nK, nQ;
    f32x4 ndY, dYc = zero4();            // dYc, ac, bc: of a chunk that is staged in part
    float na = 0.f, nb = 0.f, nvec = 0.f, ac = 0.f, bc = 0.f;
    constexpr int PT = 2 / H;            // tiles of P of a wave: (tt, jt0) .. in one row
    const int tt = w / (2 * H), jt0 = PT * (w % (2 * H));
    auto fetch = [&](int c) {
        const int L = min(C, s - c * C);
        const size_t tok = chain_tok + (size_t)c * C;
        const size_t row = tok + min(st_t, L - 1);
        nK = *reinterpret_cast<const uint4 *>((has_k ? k : q) + row * HD + st_cb * 8);
        if (H == 1) nQ = *reinterpret_cast<const uint4 *>(q + row * HD + st_cb * 8);
        ndY = *reinterpret_cast<const f32x4 *>(d_y + dy_off + (size_t)(c * C + min(yt, L - 1)) * dyr.row_stride + i0 +
                                               yg * 4);
        const size_t chunk = (size_t)chain * nc + c;
        const float *vo = vecs + chunk * vec_floats;
        na = vo[yt];
        nb = vo[CW + yt];
        nvec = vo[min(tid, 5 * CW + 7)];
    };
    // The coefficient tiles are used by the first phase of a step only; the next step's are requested right
    // after that use, into the same registers (a value that had to outlive the next request would be copied at
    // the bottom of the loop, behind a wait for that request).
    f32x4 ctab[PT];
    auto fetch_tab = [&](int c) {
        const size_t chunk = (size_t)chain * nc + c;
        const float *vo = vecs + chunk * vec_floats, *tb = tab_b + chunk * tab_floats;
#pragma unroll
        for (int x = 0; x < PT; x++) {
            const int jt = jt0 + x, bi = 2 * (tt >> 1) + (jt >> 1);
            ctab[x] = *reinterpret_cast<const f32x4 *>(
                jt <= tt ? tb + (((bi * 2 + (tt & 1)) * 2 + (jt & 1)) * 64 + l) * 4 : vo + 5 * CW);
        }
    };
    // Registers -> LDS, everything in the order it arrives (rows = tokens): the products that contract over
    // tokens read their operands through ld_op_tr.  Called during the step before, into the copy that step
    // does not use.
    auto commit_scaled = [&](u16 *dY, const f32x4 &x, float a, float b) {   // a.dY, beta.dY
        const int off = dy_at<H>(yt, yg * 4);
        split_store(dY + 2 * DYM, dY + 3 * DYM, off, a * x);
        if (HAS_S) split_store(dY + 4 * DYM, dY + 5 * DYM, off, b * x);
    };
    auto commit_plain = [&](u16 *dY, const f32x4 &x) { split_store(dY, dY + DYM, dy_at<H>(yt, yg * 4), x); };
    auto commit = [&](int c, int par) {
        const int L = min(C, s - c * C);
        u16 *Kr = late + par * LATE, *Qr = Kr + kPerm;
        if (st_t >= L) { nK = make_uint4(0, 0, 0, 0); if (H == 1) nQ = nK; }
        if (yt >= L) ndY = zero4();
        *reinterpret_cast<uint4 *>((has_k ? Kr : Qr) + bf_at(st_t, st_cb * 8)) = nK;
        if (H == 1) {
            *reinterpret_cast<uint4 *>(Qr + bf_at(st_t, st_cb * 8)) = nQ;
            commit_plain(dy_of(par), ndY);
            commit_scaled(dy_of(par), ndY, na, nb);
        } else {   // what is left of the chunk before, and this one's to wait for its turn
            commit_scaled(dys, dYc, ac, bc);
            dYc = ndY;
            ac = na;
            bc = nb;
        }
        if (tid < kCvec) cvecs[par * kCvec + tid] = nvec;
    };

    // fp32 master: transposed tile rows c = 16 (w/2) + 4 (l/16) + r, column i = 16 (w%2) + l%16
    const int rt = w / (2 * H), ct = w % (2 * H);
    f32x4 dM = zero4(), dS = zero4();
    // The snapshot a later pass reads is the bf16 value that this scan itself uses as the hi operand: it leaves
    // from the LDS copy at the top of the next step, as whole 128-byte rows (from the accumulator layout a wave
    // would store 32-byte pieces of 16 different lines).  The gradient of the initial state (slot 0) leaves in fp32.
    auto publish = [&](int slot, int l) {
        const int g = l >> 4, r16 = l & 15;
        const int e = (i0 + 16 * ct + r16) * HD + 16 * rt + 4 * g, off = bf_at(16 * ct + r16, 16 * rt + 4 * g);
        split_store(dMh, dMl, off, dM);
        if (HAS_S) split_store(dSh, dSl, off, dS);
        if (slot == 0) {
            *reinterpret_cast<f32x4 *>(dm_first + (size_t)chain * HD * HD + e) = dM;
            if (HAS_S) *reinterpret_cast<f32x4 *>(ds_first + (size_t)chain * HD * HD + e) = dS;
        }
    };
    auto store_snapshot = [&](int slot) {   // the first half of the threads: a row piece of dMo, the others: of dSo
        const int which = tid / (256 * H), row = tid % (256 * H) >> 3, c8 = (tid & 7) * 8;
        if (which && !HAS_S) return;
        const uint4 x = *reinterpret_cast<const uint4 *>((which ? dSh : dMh) + bf_at(row, c8));
        *reinterpret_cast<uint4 *>((which ? ds_snap : dm_snap) + state0 + (size_t)slot * HD * HD + (i0 + row) * HD + c8) = x;
    };

    // (W.P)^T of chunk c from its staged K, Q (copy par): this wave's two tiles of P[t][j].  It does not depend
    // on the scan, so it is computed a step ahead, in the shadow of the step's last phase.
    auto weights = [&](int par, int l) {
        const int g = l >> 4, r16 = l & 15;
        const float *cvec = cvecs + par * kCvec;
        const u16 *Kr = late + par * LATE, *Qr = Kr + kPerm;
        const bf16x8 aq[2] = {ld_perm(Qr, 16 * tt, 0, l), ld_perm(Qr, 16 * tt, 1, l)};
#pragma unroll
        for (int x = 0; x < PT; x++) {
            const int jt = jt0 + x;
            if (jt <= tt) {
                f32x4 p = zero4();
#pragma unroll
                for (int ks = 0; ks < 2; ks++) p = mfma32(aq[ks], ld_perm(Kr, 16 * jt, ks, l), p);
                const float nth = -cvec[4 * CW + 16 * jt + r16];
                split_store(WPh, WPl, bf_at(16 * jt + r16, 16 * tt + 4 * g), nth * ctab[x] * p);   // [j][t .. t+3]
            }
        }
    };

    // Two barriers per step.  First phase: the next chunk's inputs go to LDS (requested a step earlier), the ones
    // after that are requested, dE.  Second phase: dM0, dS0, the next chunk's (W.P)^T, the new state to LDS.
    fetch(nc - 1);
    fetch_tab(nc - 1);
    publish(nc, l);
    commit(nc - 1, (nc - 1) & 1);
    if (H == 2) commit_plain(dys, dYc);
    fetch(max(nc - 2, 0));
    __syncthreads();
    weights((nc - 1) & 1, l);
    fetch_tab(max(nc - 2, 0));
    __syncthreads();
    for (int c = nc - 1; c >= 0; c--) {
        const int L = min(C, s - c * C), par = c & 1;
        const float *cvec = cvecs + par * kCvec;
        const u16 *Kr = late + par * LATE, *Qr = Kr + kPerm;
        const u16 *dYh = dy_of(par), *dYl = dYh + DYM, *dYah = dYl + DYM, *dYal = dYah + DYM, *dYbh = dYal + DYM, *dYbl = dYbh + DYM;
        // The lane through an opaque copy, once per chunk: with sixteen waves the LDS addresses made of it do not fit the registers
        // across the sequence.
        int me = first_l;
        if (H == 2) asm volatile("" : "+v"(me));
        const int l = me, g = l >> 4, r16 = l & 15;
        store_snapshot(c + 1);
        commit(max(c - 1, 0), par ^ 1);
        fetch(max(c - 2, 0));
        // ── dE[j][i]: tile rows j = 16 rt.., columns i = 16 ct.. ──
        {
            f32x4 e1 = zero4(), e2 = zero4(), e3 = zero4();
#pragma unroll
            for (int ks = 0; ks < 2; ks++) {
                const bf16x8 wh = ld_perm(WPh, 16 * rt, ks, l), wl = ld_perm(WPl, 16 * rt, ks, l), ak = ld_perm(Kr, 16 * rt, ks, l);
                const bf16x8 yh = ld_dy_tr<H>(dYh, 16 * ct, ks, l), yl = ld_dy_tr<H>(dYl, 16 * ct, ks, l);
                e1 = mfma32(wh, yh, e1);
                e1 = mfma32(wl, yh, e1);
                e1 = mfma32(wh, yl, e1);
                e2 = mfma32(ak, ld_perm(dMh, 16 * ct, ks, l), e2);
                e2 = mfma32(ak, ld_perm(dMl, 16 * ct, ks, l), e2);
                if (HAS_S) {
                    e3 = mfma32(ak, ld_perm(dSh, 16 * ct, ks, l), e3);
                    e3 = mfma32(ak, ld_perm(dSl, 16 * ct, ks, l), e3);
                }
            }
            const int j4 = 16 * rt + 4 * g;
            const f32x4 th = *reinterpret_cast<const f32x4 *>(cvec + 4 * CW + j4);
            const f32x4 cl = *reinterpret_cast<const f32x4 *>(cvec + 2 * CW + j4);
            const f32x4 bl = *reinterpret_cast<const f32x4 *>(cvec + 3 * CW + j4);
            split_store(dEh, dEl, bf_at(16 * ct + r16, j4), e1 - th * (cl * e2 + bl * e3));   // [i][j .. j+3]
        }
        __syncthreads();
        // ── dM0^T, dS0^T: tile rows c = 16 rt.., columns i = 16 ct.. ──
        {
            f32x4 am = zero4(), as = zero4();
#pragma unroll
            for (int ks = 0; ks < 2; ks++) {
                const bf16x8 aq = ld_perm_tr(Qr, 16 * rt, ks, l), ak = ld_perm_tr(Kr, 16 * rt, ks, l);   // Q^T, K^T
                am = mfma32(aq, ld_dy_tr<H>(dYah, 16 * ct, ks, l), am);
                am = mfma32(aq, ld_dy_tr<H>(dYal, 16 * ct, ks, l), am);
                am = mfma32(ak, ld_perm(dEh, 16 * ct, ks, l), am);
                am = mfma32(ak, ld_perm(dEl, 16 * ct, ks, l), am);
                if (HAS_S) {
                    as = mfma32(aq, ld_dy_tr<H>(dYbh, 16 * ct, ks, l), as);
                    as = mfma32(aq, ld_dy_tr<H>(dYbl, 16 * ct, ks, l), as);
                }
            }
            const float aL = cvec[L - 1], betaL = cvec[CW + L - 1], hL = cvec[5 * CW + 4];
            const f32x4 dMn = aL * dM + am;
            if (HAS_S) dS = betaL * dM + hL * dS + as;
            dM = dMn;
        }
        publish(c, l);
        if (H == 2) commit_plain(dys, dYc);
        // (W.P)^T of the next step's chunk (staged during this step's first phase), then the tiles after it
        weights(par ^ 1, l);
        fetch_tab(max(c - 2, 0));
        __syncthreads();
    }
}

template <bool HAS_S, int H>
void launch_adjoint(const u16 *k, const u16 *q, const float *d_y, const float *tab_b, const float *vecs, u16 *dm_snap, u16 *ds_snap,
                    float *dm_first, float *ds_first, int seq_len, int chunk_size, int nc, int batch, const HeadRows &dyr) {
    static bool attr_set = false;
    if (!attr_set) {
        check_hip(hipFuncSetAttribute(reinterpret_cast<const void *>(cw_adjoint_chain_kernel<HAS_S, H>),
                                      hipFuncAttributeMaxDynamicSharedMemorySize, (int)AdjointLds<H>::bytes), "dynamic LDS size");
        attr_set = true;
    }
    KernelTimer kt("cw_adjoint_chain_kernel");
    hipLaunchKernelGGL((cw_adjoint_chain_kernel<HAS_S, H>), dim3(2 / H * batch), dim3(H * kTileThr), AdjointLds<H>::bytes, stream(), k, q,
                       d_y, tab_b, vecs, dm_snap, ds_snap, dm_first, ds_first, seq_len, chunk_size, nc, batch,
                       (int)chunkwise_grads_table_floats(), (int)chunkwise_grads_vec_floats(), dyr);
}

}  // namespace

bool chunkwise_adjoint_bf16(const uint16_t *k, const uint16_t *q, const float *d_y, const float *tab_b,
                            const float *vecs, uint16_t *dm_snap, uint16_t *ds_snap, float *dm_first,
                            float *ds_first, int seq_len, int batch, int chunk_size, bool has_s,
                            const HeadRows *dy_rows) {
    const ErrorScope es;
    const int nc = ceil_div(seq_len, chunk_size);
    const HeadRows dyr = dy_rows ? *dy_rows : head_major_rows(seq_len, HD);
    if (es.failed()) return true;
    const bool whole = adjoint_in_one_workgroup(batch, nc);
    auto launch = has_s ? (whole ? launch_adjoint<true, 2> : launch_adjoint<true, 1>)
                        : (whole ? launch_adjoint<false, 2> : launch_adjoint<false, 1>);
    launch(k, q, d_y, tab_b, vecs, dm_snap, has_s ? ds_snap : nullptr, dm_first, has_s ? ds_first : nullptr, seq_len, chunk_size, nc, batch,
           dyr);
    check_launch("cw_adjoint_chain_kernel");
    return true;
}

}  // namespace nlh
