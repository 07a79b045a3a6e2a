// Tables of one chunk shared by the chunk-parallel kernels of the HOPE self-referential memory, its gate
// functions and the entry of the chain-resident forward (selfref_chain.hip).
#pragma once
#include <hip/hip_runtime.h>

namespace nlh {

constexpr int kTB = 16;  // tokens staged in LDS at a time
using f32x4 = float __attribute__((ext_vector_type(4)));

__device__ __forceinline__ f32x4 mfma4(float a, float b, f32x4 c) {
    return __builtin_amdgcn_mfma_f32_16x16x4f32(a, b, c, 0, 0, 0);
}
__device__ __forceinline__ float lane_from(int byte_addr, float x) {
    return __builtin_bit_cast(float, __builtin_amdgcn_ds_bpermute(byte_addr, __builtin_bit_cast(int, x)));
}
__device__ __forceinline__ float lane_value(float x, int lane) {
    return __builtin_bit_cast(float, __builtin_amdgcn_readlane(__builtin_bit_cast(int, x), lane));
}
// The order in which a tile's 16 tokens are rows of a matrix product: result row 4 kg + v is token 4 v + kg.  Its own
// inverse.
__host__ __device__ constexpr int sigma(int t) { return 4 * (t & 3) + (t >> 2); }

// core/src/tensor.rs:202-207, 221-227.  The gates sit on the per-token critical path of the forward,
// so exp, log and the reciprocal are the hardware approximations (v_exp_f32, v_log_f32, v_rcp_f32: about
// one ulp each, three orders of magnitude inside the parity bar) instead of the library routines.
__device__ __forceinline__ float sr_sigmoid(float x) {
    if (x >= 15.f) return 1.f;
    if (x <= -15.f) return 0.f;
    return __builtin_amdgcn_rcpf(1.f + __expf(-x));
}
__device__ __forceinline__ float sr_softplus(float x) {
    if (x >= 15.f) return x;
    if (x <= -15.f) return 0.f;
    return __logf(1.f + __expf(x));
}

// Chunks of up to kLrC tokens use the explicit form of the shared factors,
//     G_t = A_t I - sum_{s<t} c_ts u_s k_s^T,   H_t = sum_{s<t} c_ts v_s k_s^T,
//     A_t = prod_{r<t} (1-a_r),   c_ts = th_s prod_{s<r<t} (1-a_r),
// so that no G_t, H_t is ever written to memory: products G_t^T y, H_t^T y of a
// tile of tokens become two small LDS-resident matrix products, and the inner
// product <G_t, dG_{t+1}> + <H_t, dH_{t+1}> the alpha gradient needs follows
// from a scalar recurrence (see the reverse sweep).
constexpr int kLrC = 64;

constexpr int kWL = kLrC + 4;

// LDS of the chunk-parallel kernels: the chunk's keys KC and u = k - v (or v) XC, rows of stride D + 4;
// the table c_ts; one tile of products Wt; gates and the vectors c_L, A (kLrC + 1 entries).
template <int D>
struct ChunkLds {
    static constexpr int KL = D + 4;
    float *KC, *XC, *CT, *Wt, *cal, *cth, *cL, *cA, *tiles;
    __device__ explicit ChunkLds(float *base) {
        KC = base; XC = KC + kLrC * KL; CT = XC + kLrC * KL; Wt = CT + kLrC * kLrC;
        cal = Wt + kTB * kWL; cth = cal + kLrC; cL = cth + kLrC; cA = cL + kLrC; tiles = cA + 2 * kLrC;
    }
};

// A chunk's tables from its keys and gates, one wave.  Without THETA the table holds prod_{s<r<t} (1-a_r) alone.
template <int D, bool THETA>
__device__ __forceinline__ void chunk_tables(const ChunkLds<D> &m, int L, int lane) {
    // Lane s builds column s of c downwards, c_{t,s} = th_s prod_{s<r<t} (1-a_r), so that a row's writes fall on 64
    // banks; the retentions come from the lanes that hold them, and A_t is their running product.
    const bool on = lane < L;
    const float th = on ? m.cth[lane] : 0.f, keep = on ? 1.f - m.cal[lane] : 1.f, head = THETA ? th : 1.f;
    float P = 1.f, A = 1.f, mine = 1.f;
#pragma unroll
    for (int t = 0; t < kLrC; t++) {  // retention 1 behind the last token: P and A stay as they are
        const float k = __builtin_bit_cast(float, __builtin_amdgcn_readlane(__builtin_bit_cast(int, keep), t));
        const bool behind = lane < t;
        m.CT[t * kLrC + lane] = behind ? head * P : 0.f;
        P *= behind ? k : 1.f;
        mine = lane == t ? A : mine;
        A *= k;
    }
    m.cL[lane] = on ? th * P : 0.f;
    if (on) m.cA[lane] = mine;
    if (lane == 0) m.cA[L] = A;
}
// Stages the chunk [t0, t0 + L) and builds its tables; ends with a barrier.
template <int D, bool SG>
__device__ __forceinline__ void chunk_setup(const ChunkLds<D> &m, const float *__restrict__ k_cache,
                                            const float *__restrict__ v_cache, const float *__restrict__ alpha_cache,
                                            const float *__restrict__ theta_cache, size_t tok0, int t0, int L, int tid) {
    constexpr int NT = 4 * D, V4 = D / 4, KL = D + 4;
    for (int e = tid; e < L * V4; e += NT) {
        const int li = e / V4, j = (e % V4) * 4;
        const size_t o = (tok0 + t0 + li) * D + j;
        const float4 k4 = *reinterpret_cast<const float4 *>(k_cache + o);
        const float4 v4 = *reinterpret_cast<const float4 *>(v_cache + o);
        *reinterpret_cast<float4 *>(m.KC + li * KL + j) = k4;
        *reinterpret_cast<float4 *>(m.XC + li * KL + j) =
            SG ? make_float4(k4.x - v4.x, k4.y - v4.y, k4.z - v4.z, k4.w - v4.w) : v4;
    }
    // rows behind a short chunk's last token enter the products of lowrank_tile times zero
    for (int e = L * KL + tid; e < kLrC * KL; e += NT) { m.KC[e] = 0.f; m.XC[e] = 0.f; }
    for (int e = tid; e < L; e += NT) { m.cal[e] = alpha_cache[tok0 + t0 + e]; m.cth[e] = theta_cache[tok0 + t0 + e]; }
    __syncthreads();
    if (tid < 64) chunk_tables<D, true>(m, L, tid);
    __syncthreads();
}

template <int D>
constexpr int chunk_lds_floats(int tiles) { return 2 * kLrC * (D + 4) + kLrC * kLrC + kTB * kWL + 5 * kLrC + tiles * kTB * (D + 4); }

// out_t = [A_t a1_t] + sum_{s<t} c_ts R_s ([l2_s . a2_t] - [l1_s . a1_t]) for the tokens of one tile, written
// to dst[tt * dst_stride + j]; t = li0 + tt is the token's index in its chunk, the a1 terms exist with
// HAS1, the a2 term with HAS2.  With L1 = u, R = k this is G_t^T a1 (plus H_t^T a2 for L2 = v); with
// L1 = k, R = u it is G_t a1; with L2 = k, R = v it is H_t a2.  Two products on the fp32 matrix cores:
// S = a2 L2^T - a1 L1^T (tokens x earlier tokens; wave w takes the earlier tokens 16 w ..), masked and
// scaled by c into Wt, then Wt R (wave w takes columns 16 w ..).  Tile rows have stride TL, the chunk
// arrays KL, Wt kWL (all = 4 mod 64, so the operand reads of a wave fall on 64 banks).  Rows of the
// chunk arrays behind the chunk's last token are read (times zero) and must be finite.  Called by
// every thread of the workgroup; one barrier inside, the caller synchronises before Wt, the tile or
// dst (when it is in LDS) are touched again.
template <int D, bool HAS1, bool HAS2>
__device__ __forceinline__ void lowrank_tile(const float *a1, const float *L1, const float *a2, const float *L2,
                                             const float *R, int li0, int nt, const float *CT, const float *cA,
                                             float *Wt, float *dst, size_t dst_stride, int tid) {
    constexpr int TL = D + 4, KL = D + 4, NW = D / 16;
    const int lane = tid & 63, wave = tid >> 6, ml = lane & 15, kg = lane >> 4;
    const int nprev = li0 + nt - 1;  // earlier tokens any token of the tile sees
    for (int st = wave; st < kLrC / 16; st += NW) {
        f32x4 acc = f32x4{0.f, 0.f, 0.f, 0.f};
        if (16 * st < nprev) {
#pragma unroll
            for (int k0 = 0; k0 < D; k0 += 4) {
                if (HAS1)
                    acc = __builtin_amdgcn_mfma_f32_16x16x4f32(-a1[ml * TL + k0 + kg],
                                                               L1[(16 * st + ml) * KL + k0 + kg], acc, 0, 0, 0);
                if (HAS2)
                    acc = __builtin_amdgcn_mfma_f32_16x16x4f32(a2[ml * TL + k0 + kg],
                                                               L2[(16 * st + ml) * KL + k0 + kg], acc, 0, 0, 0);
            }
        }
#pragma unroll
        for (int v = 0; v < 4; v++) {
            const int tt = 4 * kg + v, li = li0 + tt, s1 = 16 * st + ml;
            Wt[tt * kWL + s1] = (tt < nt && s1 < li) ? CT[li * kLrC + s1] * acc[v] : 0.f;
        }
    }
    __syncthreads();
    f32x4 o = f32x4{0.f, 0.f, 0.f, 0.f};
    // all of Wt's columns: those behind the tile's last token are zero, and a fixed trip count lets the
    // operand reads of the whole product be issued ahead of the first matrix instruction
#pragma unroll
    for (int k0 = 0; k0 < kLrC; k0 += 4)
        o = __builtin_amdgcn_mfma_f32_16x16x4f32(Wt[ml * kWL + k0 + kg], R[(k0 + kg) * KL + 16 * wave + ml], o, 0, 0, 0);
#pragma unroll
    for (int v = 0; v < 4; v++) {
        const int tt = 4 * kg + v, j = 16 * wave + ml;
        if (tt < nt) dst[(size_t)tt * dst_stride + j] = HAS1 ? fmaf(cA[li0 + tt], a1[tt * TL + j], o[v]) : o[v];
    }
}

// Chunk-parallel last pass of the backward: d_x_t = G_t^T dg_t + H_t^T dh_t of one chunk, in place on d_emb, which
// holds dg [B, s, D] on entry (dh likewise in its own buffer without self-generated values).  4 D threads; ready() is called
// between what needs no dg and the rest.
template <int D, bool SG, class Ready>
__device__ __forceinline__ void dx_of_chunk(float *lds, const float *k_cache, const float *v_cache, const float *alpha_cache,
                                            const float *theta_cache, float *d_emb, const float *dh, size_t b, int ci, int s, int C,
                                            Ready ready) {
    constexpr int V4 = D / 4, TL = D + 4;
    const ChunkLds<D> m(lds);
    float *tDG = m.tiles, *tDH = tDG + kTB * TL;
    int tid = threadIdx.x;   // an opaque copy: addresses made of it are not to live across the chunks of a workgroup
    asm volatile("" : "+v"(tid));
    const size_t tok0 = b * (size_t)s;
    const int t0 = ci * C, L = min(C, s - t0);
    chunk_setup<D, SG>(m, k_cache, v_cache, alpha_cache, theta_cache, tok0, t0, L, tid);
    ready();
    const int stt = tid / V4, sj = (tid % V4) * 4;
    const int ntile = (L + kTB - 1) / kTB;
    for (int tile = 0; tile < ntile; tile++) {
        const int tb = t0 + tile * kTB, nt = min(kTB, t0 + L - tb);
        __syncthreads();
        if (stt < nt) {
            const size_t o = (tok0 + tb + stt) * D + sj;
            *reinterpret_cast<float4 *>(tDG + stt * TL + sj) = *reinterpret_cast<const float4 *>(d_emb + o);
            if (!SG) *reinterpret_cast<float4 *>(tDH + stt * TL + sj) = *reinterpret_cast<const float4 *>(dh + o);
        }
        __syncthreads();
        lowrank_tile<D, true, !SG>(tDG, SG ? m.XC : m.KC, tDH, m.XC, m.KC, tb - t0, nt, m.CT, m.cA, m.Wt,
                                   d_emb + (tok0 + tb) * D, (size_t)D, tid);
    }
}

// Forward for chunks of up to kLrC tokens at head sizes 16, 32 and 64; arguments as in
// selfref_chunkwise_forward_f32_rocm, nc chunks of C tokens.  Scratch memory only where it is free to take.
struct SelfrefForward {
    float *mems;
    const float *emb;
    float *y, *k, *v, *q, *alpha, *theta, *amean, *emean, *frozen;
    int s, d, batch, C, nc;
    bool sg;
};
void selfref_forward_chain(const SelfrefForward &a);

// Backward under self-generated values for the same chunks and head sizes, up to dg (in d_emb) and d_mems; the last
// pass, d_x = G^T dg, is the caller's unless it returns true.  gl: [chunks, d, d] scratch; tok: [tokens, 3 d + 16 + 6]; outer: [chunks, 4, d, d];
// csv: [chunks, 2, d].
struct SelfrefSweep {
    const float *emb, *d_y, *k, *v, *q, *alpha, *theta, *amean, *emean, *frozen;
    float *d_emb, *d_mems, *gl, *tok, *outer, *csv;
    int s, d, batch, C, nc;
};
constexpr int sweep_token_floats(int d) { return 3 * d + 16 + 6; }
bool selfref_backward_sweep(const SelfrefSweep &a);

}  // namespace nlh
