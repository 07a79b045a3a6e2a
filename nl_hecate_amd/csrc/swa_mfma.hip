// Sliding-window attention on the bf16 matrix cores for head sizes 64 and 32, no
// persistent prefix, window <= 512 (the production shapes).  Contract and mask
// are those of core/kernels/swa_forward.cu / swa_backward.cu; other shapes stay
// on the wave-per-query kernels of swa.hip.
//
// All products are v_mfma_f32_16x16x32_bf16 steps (a 16x16x16 step costs the same
// cycles for half the work), so every operand is 8 consecutive contraction
// elements per lane: lane (r = l % 16, g = l / 16) supplies row r, contraction
// elements 8 g .. 8 g + 7 of a 32-wide step.
//
// Every kernel works in blocks: one workgroup per 128 queries (keys in the key passes), one wave per 32, or, where those leave the
// chip idle, 64 with 16 a wave (forward) or 32 in all (backward), and stages
// of 64 keys (queries) whose rows are staged in LDS exactly as they arrive.  A 16x16 result tile leaves rows
// 4 g + i in a lane; where two such tiles become an operand again with their rows as contraction index (the
// weights in O^T = V^T w^T, dS in d_q^T = K^T dS^T, ..), the matching operand is read from the row-major stage
// through ds_read_b64_tr_b16 with group g taking rows 32 hf + 4 g .. + 3 and 32 hf + 16 + 4 g .. + 3 — the rows
// the two tiles left in that group's lanes — so no stage is ever written transposed or in a permuted order.
// No kernel holds more than one stage of scores: the forward keeps a running maximum (two sweeps where the
// contract wants the normalised weights stored), the query passes accumulate A = sum (w dW) k, B = sum w k and
// D = sum w dW in one sweep and finish with d_q = (A - D B) / sqrt(hd).
//   contract (weights stored / read back):  swa_fwd_blocked_kernel, swa_bwd_q_blocked_kernel, swa_bwd_k_blocked_kernel
//   two statistics per query instead:       swa_fwd_stats_kernel,   swa_bwd_q_stats_kernel,   swa_bwd_k_stats_kernel
#include <hip/hip_runtime.h>
#include <math.h>
#include <stdint.h>

#include <type_traits>

#include "lane_ops.h"
#include "runtime.h"
#include "swa_mfma.h"
#include "swa_pieces.h"

namespace nlh {
namespace {

typedef __bf16 bh8 __attribute__((ext_vector_type(8)));
typedef __bf16 bh2 __attribute__((ext_vector_type(2)));
typedef float f32x4 __attribute__((ext_vector_type(4)));

// The kernels are templates on the head size HDV (64 or 32): NKS = HDV / 32 contraction steps over the dims, NDT = HDV / 16
// output tiles of dims; the LDS stages keep 64-wide rows either way.
constexpr int KS = 64;        // keys per LDS stage
constexpr int LDH = 80;       // LDS row stride in bf16 elements (160 B: both kinds of operand reads fall on different banks)

__device__ __forceinline__ f32x4 mfma32(uint4 a, uint4 b, f32x4 c) {
    return __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(bh8, a), __builtin_bit_cast(bh8, b), c, 0, 0, 0);
}
// two floats -> two bf16 (round to nearest even) in one dword, x in the low half; opaque, because where the compiler sees a half
// widened again it rounds that element a second time
__device__ __forceinline__ unsigned pack2(float x, float y) {
    unsigned p = __builtin_bit_cast(unsigned, bh2{(__bf16)x, (__bf16)y});
    asm("" : "+v"(p));
    return p;
}
__device__ __forceinline__ float bf_lo(unsigned w) { return __uint_as_float(w << 16); }
__device__ __forceinline__ float bf_hi(unsigned w) { return __uint_as_float(w & 0xffff0000u); }
// Largest of the four lanes that share l % 16, without LDS: the row exchanges of lane_ops.h.
__device__ __forceinline__ float groups_max(float x) {
    float a = x, b = x;
    asm volatile("s_nop 1\n\tv_permlane16_swap_b32 %0, %1" : "+v"(a), "+v"(b));
    a = b = fmaxf(a, b);
    asm volatile("s_nop 1\n\tv_permlane32_swap_b32 %0, %1" : "+v"(a), "+v"(b));
    return fmaxf(a, b);
}
// mask of elements e (low half) and e + 1 of those numbered first .. last
__device__ __forceinline__ unsigned own_pair(int e, int first, int last) {
    return (e >= first && e <= last ? 0xffffu : 0u) | (e + 1 >= first && e + 1 <= last ? 0xffff0000u : 0u);
}
// x, y = hi + lo with hi, lo bf16: the pair carries 16 mantissa bits through a bf16 product
__device__ __forceinline__ void split2(float x, float y, unsigned &hi, unsigned &lo) {
    hi = pack2(x, y);
    lo = pack2(x - bf_lo(hi), y - bf_hi(hi));
}
__device__ __forceinline__ void split8(f32x4 a, f32x4 b, uint4 &hi, uint4 &lo) {
    split2(a[0], a[1], hi.x, lo.x);
    split2(a[2], a[3], hi.y, lo.y);
    split2(b[0], b[1], hi.z, lo.z);
    split2(b[2], b[3], hi.w, lo.w);
}
// x = w dw of four elements, the weights w in two bf16 pairs, and x = hi + lo with lo from the product before it is rounded.  Explicit
// fma here and in D's terms: which of these the compiler fuses by itself depends on the code around them, and so would bits.
__device__ __forceinline__ void split_products(unsigned w01, unsigned w23, f32x4 dw, f32x4 &x, uint2 &hi, uint2 &lo) {
    const float w[4] = {bf_lo(w01), bf_hi(w01), bf_lo(w23), bf_hi(w23)};
#pragma unroll
    for (int i = 0; i < 4; i++) x[i] = w[i] * dw[i];
    hi = make_uint2(pack2(x[0], x[1]), pack2(x[2], x[3]));
    lo = make_uint2(pack2(fmaf(w[0], dw[0], -bf_lo(hi.x)), fmaf(w[1], dw[1], -bf_hi(hi.x))),
                    pack2(fmaf(w[2], dw[2], -bf_lo(hi.y)), fmaf(w[3], dw[3], -bf_hi(hi.y))));
}
// their sum; it is there before lo can be used, or factors of every tile would wait in registers for the stage's end
__device__ __forceinline__ float sum_products(unsigned w01, unsigned w23, f32x4 dw, f32x4 x, uint2 &lo) {
    float sum = fmaf(bf_lo(w01), dw[0], x[1]) + fmaf(bf_lo(w23), dw[2], x[3]);
    asm("" : "+v"(sum), "+v"(lo.y));
    return sum;
}
// Workgroup -> (block of the sequence, head * batch) with all blocks of one head on one XCD.
// Workgroups go to the 8 XCDs round robin in linear order, and each XCD has its own L2; blocks
// of one head share K and V rows, so they are given linear ids that are equal modulo 8.
struct BlockCoord { int x, h, b; };
__device__ __forceinline__ BlockCoord xcd_block_coord(int H) {
    const int gx = gridDim.x, heads = gridDim.y * gridDim.z;
    const int lin = blockIdx.x + gx * (blockIdx.y + gridDim.y * blockIdx.z);
    int x = blockIdx.x, bh = blockIdx.y + gridDim.y * blockIdx.z;
    if ((heads & 7) == 0) {
        const int xcd = lin & 7, slot = lin >> 3;
        bh = (slot / gx) * 8 + xcd;
        x = slot % gx;
    }
    return BlockCoord{x, bh % H, bh / H};
}

// Cooperative load of one stage (64 rows of 64 bf16 = 512 chunks of 16 B, two per thread of a
// 256-thread block): chunk = (row, 8 dims), consecutive lanes along a row.
struct StageSrc { const unsigned short *p; size_t row0; int total, hoff, s; };
// OUT16 instantiations of the backward passes: the gradients leave as bf16 into columns of a wider row-major matrix
// (row stride ld elements, the head's dims at the same column offset as in q, k, v), written, not accumulated.
struct Out16 { unsigned short *q, *k, *v; long long ld; };
template <int HDV>
__device__ __forceinline__ void load_rows(const StageSrc &m, int first, uint4 (&regs)[2]) {
    const int tid = threadIdx.x;
#pragma unroll
    for (int c = 0; c < 2; c++) {
        const int chunk = tid + 256 * c, row = first + (chunk >> 3);
        regs[c] = make_uint4(0, 0, 0, 0);
        if (row >= 0 && row < m.s && 8 * (chunk & 7) < HDV)
            regs[c] = *reinterpret_cast<const uint4 *>(m.p + (m.row0 + row) * m.total + m.hoff + 8 * (chunk & 7));
    }
}
// operand of a 32-wide step: row r of the tile at row0, contraction elements 32 ks + 8 g .. + 7
template <int LD>
__device__ __forceinline__ uint4 ld_op(unsigned short (*T)[LD], int row0, int ks) {
    const int l = threadIdx.x & 63;
    return *reinterpret_cast<const uint4 *>(&T[row0 + (l & 15)][32 * ks + 8 * (l >> 4)]);
}

// Forward that keeps statistics instead of weights, in blocks of keys with a running maximum (no score
// outlives its 64-key stage, so a lane holds 32 scores instead of 144 and four workgroups fit a compute unit
// instead of two).  One workgroup per (128 queries, head, batch), one wave per 32 queries; per stage a wave
// forms S^T = K Q^T for its two query tiles (32 matrix-core steps with the products of the second half, against
// 8 per barrier in the kernel above), rescales O^T by exp2(old maximum - new maximum) and adds V^T P^T with the
// unnormalised weights; the division by the sum happens once at the end.  K and V rows are staged as they
// arrive; V^T is read through ds_read_b64_tr_b16: group g of a wave takes keys 32 hf + 4 g .. + 3 and
// 32 hf + 16 + 4 g .. + 3, which are exactly the rows that the two score tiles of that half leave in its lanes.
// Queries per workgroup: 32 a wave, or 16 (NQ = 1) below two workgroups of 128 for a compute unit: a call then takes as long as
// one wave's chain of stages, which is shorter with one query tile.  Every query's sums keep their order.  Workgroups of 128,
// us with 32 and with 16 (weights stored; statistics): 32 30 / 19; 12.9 / 9.1, 256 32 / 25; 17 / 13.5, 376 28 / 21; 16 / 11.6,
// 512 41 / 42; 22.7 / 20.8.
constexpr int FQ = 128;
constexpr int LDV = 80;    // row stride of the V stage (160 B: the transposing reads of a group fall on 32 banks)

template <int LD>
__device__ __forceinline__ uint4 ld_tr2(const unsigned short (*T)[LD], int row_a, int row_b, int col0) {
    typedef short s16x4 __attribute__((ext_vector_type(4)));
    typedef __attribute__((address_space(3))) s16x4 *lds_ptr;
    const int sl = threadIdx.x & 15;
    const s16x4 a = __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_ptr)&T[row_a + (sl >> 2)][col0 + 4 * (sl & 3)]);
    const s16x4 b = __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_ptr)&T[row_b + (sl >> 2)][col0 + 4 * (sl & 3)]);
    const uint2 ua = __builtin_bit_cast(uint2, a), ub = __builtin_bit_cast(uint2, b);
    return make_uint4(ua.x, ua.y, ub.x, ub.y);
}

template <int HDV, int NQ>
__global__ __launch_bounds__(256, 3) void swa_fwd_stats_kernel(const unsigned short *__restrict__ q,
                                                            const unsigned short *__restrict__ k,
                                                            const unsigned short *__restrict__ v,
                                                            unsigned short *__restrict__ out,
                                                            float2 *__restrict__ stats, int s, int H, int ws) {
    __shared__ __align__(16) unsigned short Ks[2][KS][LDH];   // K stage [key][dim]
    __shared__ __align__(16) unsigned short Vs[2][KS][LDV];   // V stage [key][dim]
    const int tid = threadIdx.x, wave = tid >> 6, l = tid & 63, r = l & 15, g = l >> 4;
    constexpr int kRows = 64 * NQ;
    const BlockCoord bc = xcd_block_coord(H);
    const int t0 = bc.x * kRows, h = bc.h, b = bc.b;
    constexpr int NKS = HDV / 32, NDT = HDV / 16;
    constexpr float kInvSqrt = HDV == 64 ? 0.125f : 0.17677669529663687f;   // 1 / sqrt(head size)
    const int total = H * HDV, hoff = h * HDV;
    const size_t row0 = (size_t)b * s;
    const int qlo = t0 + 16 * NQ * wave, qhi = qlo + 16 * NQ - 1;           // this wave's queries
    const int st_lo = max(t0 + 1 - ws, 0) / KS, st_hi = min(t0 + kRows - 1, s - 1) / KS;
    const StageSrc km{k, row0, total, hoff, s}, vm{v, row0, total, hoff, s};

    uint4 qf[NQ][2];   // B operand: query qlo + 16 qt + r, dims 32 ks + 8 g ..
#pragma unroll
    for (int qt = 0; qt < NQ; qt++)
#pragma unroll
        for (int ks = 0; ks < NKS; ks++) {
            const int tq = qlo + 16 * qt + r;
            qf[qt][ks] = make_uint4(0, 0, 0, 0);
            if (tq < s) qf[qt][ks] = *reinterpret_cast<const uint4 *>(q + (row0 + tq) * total + hoff + 32 * ks + 8 * g);
        }
    f32x4 o[NQ][4];
#pragma unroll
    for (int qt = 0; qt < NQ; qt++)
#pragma unroll
        for (int dt = 0; dt < NDT; dt++) o[qt][dt] = f32x4{0.f, 0.f, 0.f, 0.f};
    float mrun[NQ], lsum[NQ];   // running maximum (exp2 units), this lane's share of the sum
#pragma unroll
    for (int qt = 0; qt < NQ; qt++) { mrun[qt] = -INFINITY; lsum[qt] = 0.f; }
    const float c2 = kInvSqrt * 1.44269504088896340736f;   // log2(e) / sqrt(head size)

    uint4 kreg[2], vreg[2];
    load_rows<HDV>(km, KS * st_lo, kreg);
    load_rows<HDV>(vm, KS * st_lo, vreg);
    for (int st = st_lo; st <= st_hi; st++) {
        const int buf = (st - st_lo) & 1, k0 = KS * st;
#pragma unroll
        for (int c = 0; c < 2; c++) {
            const int chunk = tid + 256 * c;
            *reinterpret_cast<uint4 *>(&Ks[buf][chunk >> 3][8 * (chunk & 7)]) = kreg[c];
            *reinterpret_cast<uint4 *>(&Vs[buf][chunk >> 3][8 * (chunk & 7)]) = vreg[c];
        }
        __syncthreads();   // also: every wave is done with the stage before the previous one, whose buffer comes next
        if (st < st_hi) {
            load_rows<HDV>(km, k0 + KS, kreg);
            load_rows<HDV>(vm, k0 + KS, vreg);
        }
        if (k0 > qhi || k0 + KS - 1 < qlo + 1 - ws) continue;   // no key of this stage is seen by this wave's queries
        f32x4 sc[4][NQ];
#pragma unroll
        for (int kt = 0; kt < 4; kt++) {
            const uint4 a0 = ld_op(Ks[buf], 16 * kt, 0), a1 = ld_op(Ks[buf], 16 * kt, 1);
#pragma unroll
            for (int qt = 0; qt < NQ; qt++) {
                sc[kt][qt] = mfma32(a0, qf[qt][0], f32x4{0.f, 0.f, 0.f, 0.f});
                if constexpr (NKS == 2) sc[kt][qt] = mfma32(a1, qf[qt][1], sc[kt][qt]);
            }
        }
        const bool full = k0 + KS - 1 <= qlo && k0 >= qhi + 1 - ws && qhi < s;   // wave-uniform: nothing to mask
        if (!full) {
#pragma unroll
            for (int kt = 0; kt < 4; kt++)
#pragma unroll
                for (int qt = 0; qt < NQ; qt++)
#pragma unroll
                    for (int i = 0; i < 4; i++) {
                        const int key = k0 + 16 * kt + 4 * g + i, tq = qlo + 16 * qt + r;
                        const bool ok = key <= tq && key >= tq + 1 - ws && tq < s;
                        sc[kt][qt][i] = ok ? sc[kt][qt][i] : -INFINITY;
                    }
        }
#pragma unroll
        for (int qt = 0; qt < NQ; qt++) {
            float mx = -INFINITY;
#pragma unroll
            for (int kt = 0; kt < 4; kt++)
#pragma unroll
                for (int i = 0; i < 4; i++) mx = fmaxf(mx, sc[kt][qt][i]);
            mx = groups_max(mx);
            const float mnew = fmaxf(mrun[qt], mx * c2);
            const float mref = mnew == -INFINITY ? 0.f : mnew;
            const float alpha = __builtin_amdgcn_exp2f(mrun[qt] - mref);
            mrun[qt] = mnew;
            float part = 0.f;
#pragma unroll
            for (int kt = 0; kt < 4; kt++)
#pragma unroll
                for (int i = 0; i < 4; i++) {
                    const float e = __builtin_amdgcn_exp2f(fmaf(sc[kt][qt][i], c2, -mref));
                    sc[kt][qt][i] = e;
                    part += e;
                }
            lsum[qt] = fmaf(lsum[qt], alpha, part);
#pragma unroll
            for (int dt = 0; dt < NDT; dt++) o[qt][dt] = o[qt][dt] * alpha;
        }
#pragma unroll
        for (int hf = 0; hf < 2; hf++) {
            uint4 pb[NQ];
#pragma unroll
            for (int qt = 0; qt < NQ; qt++) {
                const f32x4 p0 = sc[2 * hf][qt], p1 = sc[2 * hf + 1][qt];
                pb[qt] = make_uint4(pack2(p0[0], p0[1]), pack2(p0[2], p0[3]), pack2(p1[0], p1[1]), pack2(p1[2], p1[3]));
            }
#pragma unroll
            for (int dt = 0; dt < NDT; dt++) {
                const uint4 av = ld_tr2<LDV>(Vs[buf], 32 * hf + 4 * g, 32 * hf + 16 + 4 * g, 16 * dt);
#pragma unroll
                for (int qt = 0; qt < NQ; qt++) o[qt][dt] = mfma32(av, pb[qt], o[qt][dt]);
            }
        }
    }
#pragma unroll
    for (int qt = 0; qt < NQ; qt++) {
        const int tq = qlo + 16 * qt + r;
        float sum = lsum[qt];
        sum += __shfl_xor(sum, 16, 64);
        sum += __shfl_xor(sum, 32, 64);
        const float inv = sum > 0.f ? 1.0f / sum : 0.f;
        if (tq < s) {
            if (g == 0) stats[(size_t)(b * H + h) * s + tq] = make_float2(mrun[qt] == -INFINITY ? 0.f : mrun[qt], inv);
            unsigned short *ob = out + (row0 + tq) * total + hoff;
#pragma unroll
            for (int dt = 0; dt < NDT; dt++)
                *reinterpret_cast<uint2 *>(ob + 16 * dt + 4 * g) =
                    make_uint2(pack2(o[qt][dt][0] * inv, o[qt][dt][1] * inv), pack2(o[qt][dt][2] * inv, o[qt][dt][3] * inv));
        }
    }
}

// Forward of the contract (normalised weights stored) in the same blocks: the weights need the final maximum
// and sum, so the window is swept twice — scores and running statistics first, then scores again, the weights
// w = bf16(exp2(s c - m) / sum) to their slot rows and O^T += V^T w^T.  Slots behind an early query's own key (t < window - 1)
// are zeroed at the end.
// What bounds it is the weights' way out: a query's row in the tensor starts at its own key, so a lane's four keys are 8 bytes at
// any even address.  Where rows are whole 16-byte pieces (PIECES) a wave passes the stage's weights of 16 queries through LDS,
// behind the eight keys before the stage, and stores the pieces that the stage completes: 128 contiguous aligned bytes a query.
// 8 x 4096 tokens, 8 heads, window 512: 0.21 -> 0.175 ms, 0.14 without any stores; forward and backward 589 -> 556 us.
// A lane's own maximum and sum, joined at the end, gave other bf16 neighbours.
constexpr int LDP = 76;    // row stride of the pieces' LDS (8 keys of the stage before, 64 of this one)
template <int HDV, bool PIECES, int NQ>
__global__ __launch_bounds__(256, 3) void swa_fwd_blocked_kernel(const unsigned short *__restrict__ q,
                                                              const unsigned short *__restrict__ k,
                                                              const unsigned short *__restrict__ v,
                                                              unsigned short *__restrict__ out,
                                                              unsigned short *__restrict__ attn_w, int s, int H,
                                                              int ws) {
    __shared__ __align__(16) unsigned short Ks[2][KS][LDH];   // K stage [key][dim]
    __shared__ __align__(16) unsigned short Vs[2][KS][LDV];   // V stage [key][dim]
    __shared__ __align__(16) unsigned short Ws[PIECES ? 4 : 1][PIECES ? 16 : 1][LDP];   // a wave each: weights on their way out
    const int tid = threadIdx.x, wave = tid >> 6, l = tid & 63, r = l & 15, g = l >> 4;
    constexpr int kRows = 64 * NQ;
    const BlockCoord bc = xcd_block_coord(H);
    const int t0 = bc.x * kRows, h = bc.h, b = bc.b;
    constexpr int NKS = HDV / 32, NDT = HDV / 16;
    constexpr float kInvSqrt = HDV == 64 ? 0.125f : 0.17677669529663687f;   // 1 / sqrt(head size)
    const int total = H * HDV, hoff = h * HDV;
    const size_t row0 = (size_t)b * s;
    const int qlo = t0 + 16 * NQ * wave, qhi = qlo + 16 * NQ - 1;
    const int st_lo = max(t0 + 1 - ws, 0) / KS, st_hi = min(t0 + kRows - 1, s - 1) / KS;
    const StageSrc km{k, row0, total, hoff, s}, vm{v, row0, total, hoff, s};
    const float c2 = kInvSqrt * 1.44269504088896340736f;

    uint4 qf[NQ][2];
#pragma unroll
    for (int qt = 0; qt < NQ; qt++)
#pragma unroll
        for (int ks = 0; ks < NKS; ks++) {
            const int tq = qlo + 16 * qt + r;
            qf[qt][ks] = make_uint4(0, 0, 0, 0);
            if (tq < s) qf[qt][ks] = *reinterpret_cast<const uint4 *>(q + (row0 + tq) * total + hoff + 32 * ks + 8 * g);
        }
    // scores of one stage for this wave's two query tiles, masked keys at -inf
    auto scores = [&](int buf, int k0, f32x4 (&sc)[4][NQ]) {
#pragma unroll
        for (int kt = 0; kt < 4; kt++) {
            const uint4 a0 = ld_op(Ks[buf], 16 * kt, 0), a1 = ld_op(Ks[buf], 16 * kt, 1);
#pragma unroll
            for (int qt = 0; qt < NQ; qt++) {
                sc[kt][qt] = mfma32(a0, qf[qt][0], f32x4{0.f, 0.f, 0.f, 0.f});
                if constexpr (NKS == 2) sc[kt][qt] = mfma32(a1, qf[qt][1], sc[kt][qt]);
            }
        }
        const bool full = k0 + KS - 1 <= qlo && k0 >= qhi + 1 - ws && qhi < s;
        if (!full) {
#pragma unroll
            for (int kt = 0; kt < 4; kt++)
#pragma unroll
                for (int qt = 0; qt < NQ; qt++)
#pragma unroll
                    for (int i = 0; i < 4; i++) {
                        const int key = k0 + 16 * kt + 4 * g + i, tq = qlo + 16 * qt + r;
                        const bool ok = key <= tq && key >= tq + 1 - ws && tq < s;
                        sc[kt][qt][i] = ok ? sc[kt][qt][i] : -INFINITY;
                    }
        }
    };

    // ---- sweep 1: running maximum and sum ----
    float mrun[NQ], lsum[NQ];
#pragma unroll
    for (int qt = 0; qt < NQ; qt++) { mrun[qt] = -INFINITY; lsum[qt] = 0.f; }
    uint4 kreg[2], vreg[2];
    load_rows<HDV>(km, KS * st_lo, kreg);
    for (int st = st_lo; st <= st_hi; st++) {
        const int buf = (st - st_lo) & 1, k0 = KS * st;
#pragma unroll
        for (int c = 0; c < 2; c++) {
            const int chunk = tid + 256 * c;
            *reinterpret_cast<uint4 *>(&Ks[buf][chunk >> 3][8 * (chunk & 7)]) = kreg[c];
        }
        __syncthreads();
        if (st < st_hi) load_rows<HDV>(km, k0 + KS, kreg);
        if (k0 > qhi || k0 + KS - 1 < qlo + 1 - ws) continue;
        f32x4 sc[4][NQ];
        scores(buf, k0, sc);
#pragma unroll
        for (int qt = 0; qt < NQ; qt++) {
            float mx = -INFINITY;
#pragma unroll
            for (int kt = 0; kt < 4; kt++)
#pragma unroll
                for (int i = 0; i < 4; i++) mx = fmaxf(mx, sc[kt][qt][i]);
            mx = fmaxf(mx, __shfl_xor(mx, 16, 64));
            mx = fmaxf(mx, __shfl_xor(mx, 32, 64));
            const float mnew = fmaxf(mrun[qt], mx * c2);
            const float mref = mnew == -INFINITY ? 0.f : mnew;
            const float alpha = __builtin_amdgcn_exp2f(mrun[qt] - mref);
            mrun[qt] = mnew;
            float part = 0.f;
#pragma unroll
            for (int kt = 0; kt < 4; kt++)
#pragma unroll
                for (int i = 0; i < 4; i++) part += __builtin_amdgcn_exp2f(fmaf(sc[kt][qt][i], c2, -mref));
            lsum[qt] = fmaf(lsum[qt], alpha, part);
        }
    }
    float mc[NQ], inv[NQ];
#pragma unroll
    for (int qt = 0; qt < NQ; qt++) {
        float sum = lsum[qt];
        sum += __shfl_xor(sum, 16, 64);
        sum += __shfl_xor(sum, 32, 64);
        inv[qt] = sum > 0.f ? 1.0f / sum : 0.f;
        mc[qt] = mrun[qt] == -INFINITY ? 0.f : mrun[qt];
    }

    // ---- sweep 2: weights out, O^T = V^T w^T ----
    f32x4 o[NQ][4];
#pragma unroll
    for (int qt = 0; qt < NQ; qt++)
#pragma unroll
        for (int dt = 0; dt < NDT; dt++) o[qt][dt] = f32x4{0.f, 0.f, 0.f, 0.f};
    unsigned short *wblk = attn_w + ((size_t)(b * H + h) * s + qlo) * ws;   // row of the wave's first query
    uint2 before[NQ] = {};   // PIECES: the weights of the last tile of the stage before
    __syncthreads();   // every wave is done with the buffers of sweep 1
    load_rows<HDV>(km, KS * st_lo, kreg);
    load_rows<HDV>(vm, KS * st_lo, vreg);
    for (int st = st_lo; st <= st_hi; st++) {
        const int buf = (st - st_lo) & 1, k0 = KS * st;
#pragma unroll
        for (int c = 0; c < 2; c++) {
            const int chunk = tid + 256 * c;
            *reinterpret_cast<uint4 *>(&Ks[buf][chunk >> 3][8 * (chunk & 7)]) = kreg[c];
            *reinterpret_cast<uint4 *>(&Vs[buf][chunk >> 3][8 * (chunk & 7)]) = vreg[c];
        }
        __syncthreads();
        if (st < st_hi) {
            load_rows<HDV>(km, k0 + KS, kreg);
            load_rows<HDV>(vm, k0 + KS, vreg);
        }
        if (k0 > qhi || k0 + KS - 1 < qlo + 1 - ws) continue;
        f32x4 sc[4][NQ];
        scores(buf, k0, sc);
        unsigned wp[NQ][4][2];
#pragma unroll
        for (int qt = 0; qt < NQ; qt++)
#pragma unroll
            for (int kt = 0; kt < 4; kt++) {
                const f32x4 x = sc[kt][qt];
                float w[4];
#pragma unroll
                for (int i = 0; i < 4; i++) w[i] = __builtin_amdgcn_exp2f(fmaf(x[i], c2, -mc[qt])) * inv[qt];
                wp[qt][kt][0] = pack2(w[0], w[1]);
                wp[qt][kt][1] = pack2(w[2], w[3]);
            }
        if constexpr (PIECES) {
            unsigned short(*W)[LDP] = Ws[wave];
            const int pr = l >> 3, pj = l & 7;   // the lane's row (of 8) and piece on the way out
#pragma unroll
            for (int qt = 0; qt < NQ; qt++) {
                wave_lds_order();
                if (g >= 2) *reinterpret_cast<uint2 *>(&W[r][4 * (g - 2)]) = before[qt];
#pragma unroll
                for (int kt = 0; kt < 4; kt++) *reinterpret_cast<uint2 *>(&W[r][8 + 16 * kt + 4 * g]) = make_uint2(wp[qt][kt][0], wp[qt][kt][1]);
                before[qt] = make_uint2(wp[qt][3][0], wp[qt][3][1]);
                wave_lds_order();
#pragma unroll
                for (int half = 0; half < 2; half++) {
                    const int row = 8 * half + pr, tq = qlo + 16 * qt + row, ls = max(tq + 1 - ws, 0);
                    const int first = k0 - ls, piece = (first >> 3) + pj;   // slots 8 piece .. + 7: keys from k0 - first % 8 + 8 pj on
                    // the stage completes eight pieces, less those in front of the row and behind the query's own key
                    const int e = 8 - (first & 7) + 8 * pj, sh = 16 * (e & 1);
                    const unsigned *src = reinterpret_cast<const unsigned *>(W[row]) + (e >> 1);
                    const unsigned d0 = src[0], d1 = src[1], d2 = src[2], d3 = src[3], d4 = src[4];   // d4 may lie in the row's pad: unused then
                    if (tq < s && piece >= 0 && 8 * piece <= tq - ls)
                        *reinterpret_cast<uint4 *>(wblk + (size_t)(16 * qt + row) * ws + 8 * piece) =
                            make_uint4(__builtin_amdgcn_alignbit(d1, d0, sh), __builtin_amdgcn_alignbit(d2, d1, sh),
                                       __builtin_amdgcn_alignbit(d3, d2, sh), __builtin_amdgcn_alignbit(d4, d3, sh));
                }
            }
        } else {
#pragma unroll
            for (int qt = 0; qt < NQ; qt++) {
                const int tq = qlo + 16 * qt + r, ls = max(tq + 1 - ws, 0);
                unsigned short *wrow = wblk + (size_t)(16 * qt + r) * ws;
#pragma unroll
                for (int kt = 0; kt < 4; kt++) {
                    // keys key0 .. key0 + 3 of query tq sit in slots key0 - ls ..; only keys of the window have one
                    const int key0 = k0 + 16 * kt + 4 * g;
                    if (tq < s) {
                        if (key0 >= ls && key0 + 3 <= tq) {
                            const uint2 pr = make_uint2(wp[qt][kt][0], wp[qt][kt][1]);
                            __builtin_memcpy(wrow + (key0 - ls), &pr, 8);
                        } else if (key0 + 3 >= ls && key0 <= tq) {
#pragma unroll
                            for (int i = 0; i < 4; i++)
                                if (key0 + i >= ls && key0 + i <= tq)
                                    wrow[key0 + i - ls] = (unsigned short)(wp[qt][kt][i >> 1] >> (16 * (i & 1)));
                        }
                    }
                }
            }
        }
#pragma unroll
        for (int hf = 0; hf < 2; hf++) {
            uint4 pb[NQ];
#pragma unroll
            for (int qt = 0; qt < NQ; qt++)
                pb[qt] = make_uint4(wp[qt][2 * hf][0], wp[qt][2 * hf][1], wp[qt][2 * hf + 1][0], wp[qt][2 * hf + 1][1]);
#pragma unroll
            for (int dt = 0; dt < NDT; dt++) {
                const uint4 av = ld_tr2<LDV>(Vs[buf], 32 * hf + 4 * g, 32 * hf + 16 + 4 * g, 16 * dt);
#pragma unroll
                for (int qt = 0; qt < NQ; qt++) o[qt][dt] = mfma32(av, pb[qt], o[qt][dt]);
            }
        }
    }
    // early queries: the slots behind the query's own key hold zeros
    if (qlo < ws - 1) {
        unsigned short *awb = attn_w + ((size_t)(b * H + h) * s) * ws;
        for (int qi = 0; qi < 16 * NQ; qi++) {
            const int tt = qlo + qi;
            if (tt >= s || tt >= ws - 1) break;
            for (int slot = tt + 1 + l; slot < ws; slot += 64) awb[(size_t)tt * ws + slot] = 0;
        }
    }
#pragma unroll
    for (int qt = 0; qt < NQ; qt++) {
        const int tq = qlo + 16 * qt + r;
        if (tq < s) {
            unsigned short *ob = out + (row0 + tq) * total + hoff;
#pragma unroll
            for (int dt = 0; dt < NDT; dt++)
                *reinterpret_cast<uint2 *>(ob + 16 * dt + 4 * g) =
                    make_uint2(pack2(o[qt][dt][0], o[qt][dt][1]), pack2(o[qt][dt][2], o[qt][dt][3]));
        }
    }
}

// The backward passes of a call that leaves the chip idle (SPLIT): bound by one wave's chain of stages, so a workgroup has 32
// queries (keys) instead of 128.  Two stages at a time, its four waves form the weights and dS of half a stage each, pass them
// on through LDS (HalfStage), and add the products of both stages up in the order of the keys (queries), each wave for
// a quarter of the result's tiles.  Every sum then has the order that it has in a block of 128, so that a sequence's gradients
// are the same bits alone and in any batch.
// What a workgroup stages serves a quarter of the rows: taken while the four times as many workgroups still fit the chip at
// once, two a compute unit.  Both passes, contract / statistics, us as blocks of 128 and so, head size 64, window 512: 32 blocks of 128
// rows 46 -> 23 / 60 -> 28, 112 blocks 58 -> 38 / 73 -> 43 (21 / 27.5 and 35 / 41 with every wave's sums of its own half stages,
// joined at the end); where they do not fit, with joined sums, 192 blocks 63 -> 62 or 75, 256 blocks (window 256) 46 -> 52, 512 blocks 92 -> 131.
constexpr int SQ = 32;     // queries (keys) per workgroup of these
constexpr int LDQ = 72;  // row stride of the key passes' stages there: two workgroups fit a compute unit
// Operands of the products over half a stage, on their way from the wave that forms them: [tile of rows][operand][lane]
template <int N>
using HalfStage = uint4[2][N][64];
// The tiles of the result that a wave adds up: NT of rows from tile0 on, ND of dims from dt0 on
template <int NDT, bool SPLIT>
struct OwnTiles {
    static constexpr int NT = SPLIT ? 1 : 2, ND = SPLIT ? NDT / 2 : NDT;
    int tile0, dt0;
    __device__ __forceinline__ explicit OwnTiles(int wave) : tile0(SPLIT ? wave >> 1 : 0), dt0(SPLIT ? (wave & 1) * ND : 0) {}
};

// Query pass on statistics, in key blocks like swa_fwd_stats_kernel (one workgroup per 128 queries, one wave per
// 32), in ONE sweep over the window.  dS = w (dW - D) needs D_t = sum_j w dW of the whole window, so the sweep
// accumulates the two sums that do not:  A^T = K^T (w dW)^T and B^T = K^T w^T, and D itself, and ends with
//   d_q = (A - D B) / sqrt(hd)
// (the same numbers as sum_j dS k_j; no sweep that rebuilds O first, and D as exact as before — taking D from
// the forward's bf16 output instead moves it by 2^-9 and, where the window holds few keys, d_q by 5e-3).
// Per stage a wave forms S^T = K Q^T, the weights w = bf16(exp2(s c - m) / sum) as the weight tensor would hold
// them, dW^T = V dO^T; dO and w dW enter as hi + lo pairs, w is exact in bf16.  K^T is read from the K rows
// through ds_read_b64_tr_b16 in the key order that the score tiles leave in the lanes.  D goes to dvec.
template <int HDV, bool OUT16, bool SPLIT>
__global__ __launch_bounds__(256, 2) void swa_bwd_q_stats_kernel(const unsigned short *__restrict__ q,
                                                                 const unsigned short *__restrict__ k,
                                                                 const unsigned short *__restrict__ v,
                                                                 const float2 *__restrict__ stats,
                                                                 const float *__restrict__ d_out,
                                                                 float *__restrict__ d_q, float *__restrict__ dvec,
                                                                 int s, int H, int ws, Out16 o16) {
    __shared__ __align__(16) unsigned short KV[4][KS][LDH];   // two stages [key][dim] of K, then of V
    __shared__ HalfStage<3> Px[SPLIT ? 4 : 1];                // SPLIT: w dW hi and lo and w of a wave's half stage,
    __shared__ float Dx[SPLIT ? 4 : 1][2][2][64];             // and its terms of D
    unsigned short (*const Ks)[KS][LDH] = KV, (*const Vs)[KS][LDH] = KV + 2;
    const int tid = threadIdx.x, wave = tid >> 6, l = tid & 63, r = l & 15, g = l >> 4;
    const BlockCoord bc = xcd_block_coord(H);
    const int t0 = bc.x * (SPLIT ? SQ : FQ), h = bc.h, b = bc.b;
    constexpr int NKS = HDV / 32, NDT = HDV / 16;
    constexpr float kInvSqrt = HDV == 64 ? 0.125f : 0.17677669529663687f;   // 1 / sqrt(head size)
    const int total = H * HDV, hoff = h * HDV;
    const size_t row0 = (size_t)b * s;
    const int qlo = SPLIT ? t0 : t0 + 32 * wave, qhi = qlo + 31;
    const int st_lo = max(t0 + 1 - ws, 0) / KS, st_hi = min(t0 + (SPLIT ? SQ : FQ) - 1, s - 1) / KS;
    const StageSrc km{k, row0, total, hoff, s}, vm{v, row0, total, hoff, s};
    const float c2 = kInvSqrt * 1.44269504088896340736f, scale = kInvSqrt;

    uint4 qf[2][2], doh[2][2], dol[2][2];
    float mc[2], inv[2];
#pragma unroll
    for (int qt = 0; qt < 2; qt++) {
        const int tq = qlo + 16 * qt + r;
        mc[qt] = 0.f; inv[qt] = 0.f;
#pragma unroll
        for (int ks = 0; ks < NKS; ks++) {
            qf[qt][ks] = make_uint4(0, 0, 0, 0);
            f32x4 x0 = f32x4{0.f, 0.f, 0.f, 0.f}, x1 = x0;
            if (tq < s) {
                const size_t o = (row0 + tq) * total + hoff + 32 * ks + 8 * g;
                qf[qt][ks] = *reinterpret_cast<const uint4 *>(q + o);
                x0 = *reinterpret_cast<const f32x4 *>(d_out + o);
                x1 = *reinterpret_cast<const f32x4 *>(d_out + o + 4);
            }
            split8(x0, x1, doh[qt][ks], dol[qt][ks]);
        }
        if (tq < s) {
            const float2 st2 = stats[(size_t)(b * H + h) * s + tq];
            mc[qt] = st2.x;
            inv[qt] = st2.y;
        }
    }
    using Own = OwnTiles<NDT, SPLIT>;
    const Own own(wave);
    f32x4 aq[Own::NT][Own::ND], bq[Own::NT][Own::ND];
    float dpart[Own::NT];
#pragma unroll
    for (int t = 0; t < Own::NT; t++) {
        dpart[t] = 0.f;
#pragma unroll
        for (int dt = 0; dt < Own::ND; dt++) { aq[t][dt] = f32x4{0.f, 0.f, 0.f, 0.f}; bq[t][dt] = f32x4{0.f, 0.f, 0.f, 0.f}; }
    }
    // half hf of a stage added to the sums of this wave's tiles
    auto add = [&](unsigned short(*K)[LDH], int hf, const uint4(&xh)[Own::NT], const uint4(&xl)[Own::NT], const uint4(&wb)[Own::NT])
                   __attribute__((always_inline)) {
#pragma unroll
        for (int dt = 0; dt < Own::ND; dt++) {
            const uint4 a = ld_tr2<LDH>(K, 32 * hf + 4 * g, 32 * hf + 16 + 4 * g, 16 * (own.dt0 + dt));
#pragma unroll
            for (int t = 0; t < Own::NT; t++) {
                aq[t][dt] = mfma32(a, xh[t], aq[t][dt]);
                aq[t][dt] = mfma32(a, xl[t], aq[t][dt]);
                bq[t][dt] = mfma32(a, wb[t], bq[t][dt]);
            }
        }
    };

    uint4 kreg[SPLIT ? 2 : 1][2], vreg[SPLIT ? 2 : 1][2];
    auto fetch_stages = [&](int first) {
#pragma unroll
        for (int p = 0; p < (SPLIT ? 2 : 1); p++) {
            load_rows<HDV>(km, first + KS * p, kreg[p]);
            load_rows<HDV>(vm, first + KS * p, vreg[p]);
        }
    };
    fetch_stages(KS * st_lo);
    for (int st = st_lo; st <= st_hi; st += SPLIT ? 2 : 1) {
        const int buf = SPLIT ? wave >> 1 : (st - st_lo) & 1, k0 = KS * (SPLIT ? st + buf : st);
        if (SPLIT && st > st_lo) __syncthreads();   // the stages and half stages before are read
#pragma unroll
        for (int p = 0; p < (SPLIT ? 2 : 1); p++)
#pragma unroll
            for (int c = 0; c < 2; c++) {
                const int chunk = tid + 256 * c, to = SPLIT ? p : buf;
                *reinterpret_cast<uint4 *>(&Ks[to][chunk >> 3][8 * (chunk & 7)]) = kreg[p][c];
                *reinterpret_cast<uint4 *>(&Vs[to][chunk >> 3][8 * (chunk & 7)]) = vreg[p][c];
            }
        __syncthreads();
        if (st + (SPLIT ? 1 : 0) < st_hi) fetch_stages(KS * (st + (SPLIT ? 2 : 1)));
        if (!SPLIT && (k0 > qhi || k0 + KS - 1 < qlo + 1 - ws)) continue;   // SPLIT: a stage of no key of these queries is not added
        const bool full = k0 + KS - 1 <= qlo && k0 >= qhi + 1 - ws && qhi < s;
#pragma unroll
        for (int half = 0; half < (SPLIT ? 1 : 2); half++) {
            const int hf = SPLIT ? wave & 1 : half;
            uint4 xh[2], xl[2], wb[2];
#pragma unroll
            for (int qt = 0; qt < 2; qt++) {
                unsigned wp[2][2];
                uint2 hi[2], lo[2];
#pragma unroll
                for (int c = 0; c < 2; c++) {
                    const int kt = 2 * hf + c;
                    const uint4 ak0 = ld_op(Ks[buf], 16 * kt, 0), ak1 = ld_op(Ks[buf], 16 * kt, 1);
                    const uint4 av0 = ld_op(Vs[buf], 16 * kt, 0), av1 = ld_op(Vs[buf], 16 * kt, 1);
                    f32x4 sc = mfma32(ak0, qf[qt][0], f32x4{0.f, 0.f, 0.f, 0.f});
                    if constexpr (NKS == 2) sc = mfma32(ak1, qf[qt][1], sc);
                    f32x4 dw = mfma32(av0, doh[qt][0], f32x4{0.f, 0.f, 0.f, 0.f});
                    dw = mfma32(av0, dol[qt][0], dw);
                    if constexpr (NKS == 2) dw = mfma32(av1, doh[qt][1], dw);
                    if constexpr (NKS == 2) dw = mfma32(av1, dol[qt][1], dw);
                    f32x4 w;
#pragma unroll
                    for (int i = 0; i < 4; i++) {
                        const int key = k0 + 16 * kt + 4 * g + i, tq = qlo + 16 * qt + r;
                        const bool ok = full || (key <= tq && key >= tq + 1 - ws && tq < s);
                        w[i] = ok ? __builtin_amdgcn_exp2f(fmaf(sc[i], c2, -mc[qt])) * inv[qt] : 0.f;
                    }
                    wp[c][0] = pack2(w[0], w[1]);   // as the weight tensor holds them
                    wp[c][1] = pack2(w[2], w[3]);
                    f32x4 x;
                    split_products(wp[c][0], wp[c][1], dw, x, hi[c], lo[c]);
                    const float d4 = sum_products(wp[c][0], wp[c][1], dw, x, lo[c]);
                    if constexpr (SPLIT) Dx[wave][qt][c][l] = d4;
                    else dpart[qt] += d4;
                }
                xh[qt] = make_uint4(hi[0].x, hi[0].y, hi[1].x, hi[1].y);
                xl[qt] = make_uint4(lo[0].x, lo[0].y, lo[1].x, lo[1].y);
                wb[qt] = make_uint4(wp[0][0], wp[0][1], wp[1][0], wp[1][1]);
            }
            if constexpr (SPLIT) {
#pragma unroll
                for (int qt = 0; qt < 2; qt++) { Px[wave][qt][0][l] = xh[qt]; Px[wave][qt][1][l] = xl[qt]; Px[wave][qt][2][l] = wb[qt]; }
            } else {
                add(Ks[buf], hf, xh, xl, wb);
            }
        }
        if constexpr (SPLIT) {
            __syncthreads();   // the four half stages are there
#pragma unroll
            for (int p = 0; p < 2; p++) {
                if (st + p > st_hi) break;
#pragma unroll
                for (int hf = 0; hf < 2; hf++) {
                    const int h = 2 * p + hf;
                    const auto &x = Px[h][own.tile0];
                    dpart[0] += Dx[h][own.tile0][0][l];
                    dpart[0] += Dx[h][own.tile0][1][l];
                    add(Ks[p], hf, {x[0][l]}, {x[1][l]}, {x[2][l]});
                }
            }
        }
    }
#pragma unroll
    for (int t = 0; t < Own::NT; t++) {
        const int tq = qlo + 16 * (own.tile0 + t) + r;
        float dsum = dpart[t];
        dsum += __shfl_xor(dsum, 16, 64);
        dsum += __shfl_xor(dsum, 32, 64);
        if (tq < s) {
            if (g == 0 && own.dt0 == 0) dvec[(size_t)(b * H + h) * s + tq] = dsum;
            if (OUT16) {
                unsigned short *ob = o16.q + (row0 + tq) * o16.ld + hoff;
#pragma unroll
                for (int dt = 0; dt < Own::ND; dt++) {
                    const f32x4 x = (aq[t][dt] - dsum * bq[t][dt]) * scale;
                    *reinterpret_cast<uint2 *>(ob + 16 * (own.dt0 + dt) + 4 * g) = make_uint2(pack2(x[0], x[1]), pack2(x[2], x[3]));
                }
            } else {
                float *ob = d_q + (row0 + tq) * total + hoff;
#pragma unroll
                for (int dt = 0; dt < Own::ND; dt++)
                    *reinterpret_cast<f32x4 *>(ob + 16 * (own.dt0 + dt) + 4 * g) = (aq[t][dt] - dsum * bq[t][dt]) * scale;
            }
        }
    }
}

// Where a stage's key (0..63) goes, so that two tiles leave a lane group g eight consecutive keys, 32 hf + 8 g + 4 c + i in row
// 4 g + i of tile 2 hf + c: the weights of a query are then read 16 bytes a lane, 64 side by side.
__device__ __forceinline__ int stage_row(int key) { return (key & 32) + 16 * ((key >> 2) & 1) + 4 * ((key >> 3) & 3) + (key & 3); }

// Query pass of the contract (weights read back from the tensor) in the same blocks and the same single sweep as
// swa_bwd_q_stats_kernel: A = sum_j (w dW) k_j, B = sum_j w k_j and D = sum_j w dW together, d_q = (A - D B)/sqrt(hd).
// A lane's eight keys of two tiles are eight consecutive slots of its query's row: one 16-byte load (2-byte aligned),
// requested a stage ahead.  Bound by the latency of a stage's chain of LDS reads, products and element work on two waves a
// SIMD (matrix cores 0.16, vector units 0.26, LDS 0.11 of their time).  8 x 4096 tokens, 8 heads, window 512: 210 us (247
// with 8-byte loads, slot by slot with a wait in every stage at the window's ends); 192 without any loads of weights.
template <int HDV, bool SPLIT>
__global__ __launch_bounds__(256, 2) void swa_bwd_q_blocked_kernel(const unsigned short *__restrict__ k,
                                                                   const unsigned short *__restrict__ v,
                                                                   const unsigned short *__restrict__ attn_w,
                                                                   const float *__restrict__ d_out,
                                                                   float *__restrict__ d_q, float *__restrict__ dvec,
                                                                   int s, int H, int ws) {
    __shared__ __align__(16) unsigned short KV[4][KS][LDH];   // two stages [key][dim] of K, then of V
    __shared__ HalfStage<3> Px[SPLIT ? 4 : 1];                // SPLIT: w dW hi and lo and w of a wave's half stage,
    __shared__ float Dx[SPLIT ? 4 : 1][2][2][64];             // and its terms of D
    unsigned short (*const Ks)[KS][LDH] = KV, (*const Vs)[KS][LDH] = KV + 2;
    const int tid = threadIdx.x, wave = tid >> 6, l = tid & 63, r = l & 15, g = l >> 4;
    const BlockCoord bc = xcd_block_coord(H);
    const int t0 = bc.x * (SPLIT ? SQ : FQ), h = bc.h, b = bc.b;
    constexpr int NKS = HDV / 32, NDT = HDV / 16;
    constexpr float kInvSqrt = HDV == 64 ? 0.125f : 0.17677669529663687f;   // 1 / sqrt(head size)
    const int total = H * HDV, hoff = h * HDV;
    const size_t row0 = (size_t)b * s;
    const int qlo = SPLIT ? t0 : t0 + 32 * wave, qhi = qlo + 31;
    const int st_lo = max(t0 + 1 - ws, 0) / KS, st_hi = min(t0 + (SPLIT ? SQ : FQ) - 1, s - 1) / KS;
    const StageSrc km{k, row0, total, hoff, s}, vm{v, row0, total, hoff, s};
    const float scale = kInvSqrt;

    uint4 doh[2][2], dol[2][2];
    const unsigned short *wrow[2];
    int lsq[2], tqs[2];
#pragma unroll
    for (int qt = 0; qt < 2; qt++) {
        const int tq = qlo + 16 * qt + r;
        tqs[qt] = tq < s ? tq : -1;   // -1: no key passes "key <= tq"
        lsq[qt] = max(tq + 1 - ws, 0);
        wrow[qt] = attn_w + ((size_t)(b * H + h) * s + min(tq, s - 1)) * ws;
#pragma unroll
        for (int ks = 0; ks < NKS; ks++) {
            f32x4 x0 = f32x4{0.f, 0.f, 0.f, 0.f}, x1 = x0;
            if (tq < s) {
                const size_t o = (row0 + tq) * total + hoff + 32 * ks + 8 * g;
                x0 = *reinterpret_cast<const f32x4 *>(d_out + o);
                x1 = *reinterpret_cast<const f32x4 *>(d_out + o + 4);
            }
            split8(x0, x1, doh[qt][ks], dol[qt][ks]);
        }
    }
    using Own = OwnTiles<NDT, SPLIT>;
    const Own own(wave);
    f32x4 aq[Own::NT][Own::ND], bq[Own::NT][Own::ND];
    float dpart[Own::NT];
#pragma unroll
    for (int t = 0; t < Own::NT; t++) {
        dpart[t] = 0.f;
#pragma unroll
        for (int dt = 0; dt < Own::ND; dt++) { aq[t][dt] = f32x4{0.f, 0.f, 0.f, 0.f}; bq[t][dt] = f32x4{0.f, 0.f, 0.f, 0.f}; }
    }
    // half hf of a stage added to the sums of this wave's tiles
    auto add = [&](unsigned short(*K)[LDH], int hf, const uint4(&xh)[Own::NT], const uint4(&xl)[Own::NT], const uint4(&wb)[Own::NT])
                   __attribute__((always_inline)) {
#pragma unroll
        for (int dt = 0; dt < Own::ND; dt++) {
            const uint4 a = ld_tr2<LDH>(K, 32 * hf + 4 * g, 32 * hf + 16 + 4 * g, 16 * (own.dt0 + dt));
#pragma unroll
            for (int t = 0; t < Own::NT; t++) {
                aq[t][dt] = mfma32(a, xh[t], aq[t][dt]);
                aq[t][dt] = mfma32(a, xl[t], aq[t][dt]);
                bq[t][dt] = mfma32(a, wb[t], bq[t][dt]);
            }
        }
    };

    // Weights of a stage for this lane: wreg[hf][qt] = keys k0 + 32 hf + 8 g .. + 7 of query qt (stage_row).  At the window's ends
    // a piece is read whole as well, out of the rows next to it, and what is not the query's own is taken off where the piece
    // is used: not here, where that would wait for the read.
    constexpr int NH = SPLIT ? 1 : 2;
    uint4 wreg[NH][2];
    const bool at_edge = edge_head(b * H + h, (int)(gridDim.y * gridDim.z), s, ws);
    auto whole = [&](int k0) { return k0 + KS - 1 <= qlo && k0 >= qhi + 1 - ws && qhi < s; };
    auto fetch_weights = [&](int k0) {
        const bool skip = k0 > qhi || k0 + KS - 1 < qlo + 1 - ws, full = whole(k0);
#pragma unroll
        for (int half = 0; half < NH; half++)
#pragma unroll
            for (int qt = 0; qt < 2; qt++) {
                const int key0 = k0 + 32 * (SPLIT ? wave & 1 : half) + 8 * g;
                wreg[half][qt] = make_uint4(0u, 0u, 0u, 0u);
                if (skip) continue;
                const unsigned short *p = wrow[qt] + (key0 - lsq[qt]);
                if (full) {
                    __builtin_memcpy(&wreg[half][qt], p, 16);
                } else if (key0 + 7 >= lsq[qt] && key0 <= tqs[qt]) {
                    if (!at_edge || piece_inside(tqs[qt], s, ws, key0 - lsq[qt])) {
                        __builtin_memcpy(&wreg[half][qt], p, 16);
                    } else {   // at the tensor's own ends
                        unsigned d[4] = {0u, 0u, 0u, 0u};
#pragma unroll
                        for (int e = 0; e < 8; e++) {
                            const int key = key0 + e;
                            unsigned x = 0;
                            if (key >= lsq[qt] && key <= tqs[qt]) x = wrow[qt][key - lsq[qt]];
                            d[e >> 1] |= x << (16 * (e & 1));
                        }
                        wreg[half][qt] = make_uint4(d[0], d[1], d[2], d[3]);
                    }
                }
            }
    };

    const int sub = SPLIT ? wave >> 1 : 0;   // which stage of a pair is this wave's
    uint4 kreg[SPLIT ? 2 : 1][2], vreg[SPLIT ? 2 : 1][2];
    auto fetch_stages = [&](int first) {
#pragma unroll
        for (int p = 0; p < (SPLIT ? 2 : 1); p++) {
            load_rows<HDV>(km, first + KS * p, kreg[p]);
            load_rows<HDV>(vm, first + KS * p, vreg[p]);
        }
        fetch_weights(first + KS * sub);
    };
    fetch_stages(KS * st_lo);
    for (int st = st_lo; st <= st_hi; st += SPLIT ? 2 : 1) {
        const int buf = SPLIT ? sub : (st - st_lo) & 1, k0 = KS * (st + sub);
        if (SPLIT && st > st_lo) __syncthreads();   // the stages and half stages before are read
#pragma unroll
        for (int p = 0; p < (SPLIT ? 2 : 1); p++)
#pragma unroll
            for (int c = 0; c < 2; c++) {
                const int chunk = tid + 256 * c, to = SPLIT ? p : buf;
                *reinterpret_cast<uint4 *>(&Ks[to][stage_row(chunk >> 3)][8 * (chunk & 7)]) = kreg[p][c];
                *reinterpret_cast<uint4 *>(&Vs[to][stage_row(chunk >> 3)][8 * (chunk & 7)]) = vreg[p][c];
            }
        uint4 wcur[NH][2];
        const bool full = whole(k0);
#pragma unroll
        for (int half = 0; half < NH; half++)
#pragma unroll
            for (int qt = 0; qt < 2; qt++) {
                wcur[half][qt] = wreg[half][qt];
                if (!full) {
                    const int key0 = k0 + 32 * (SPLIT ? wave & 1 : half) + 8 * g, first = lsq[qt] - key0, last = tqs[qt] - key0;
                    wcur[half][qt].x &= own_pair(0, first, last);
                    wcur[half][qt].y &= own_pair(2, first, last);
                    wcur[half][qt].z &= own_pair(4, first, last);
                    wcur[half][qt].w &= own_pair(6, first, last);
                }
            }
        __syncthreads();
        if (st + (SPLIT ? 1 : 0) < st_hi) fetch_stages(KS * (st + (SPLIT ? 2 : 1)));
        if (!SPLIT && (k0 > qhi || k0 + KS - 1 < qlo + 1 - ws)) continue;   // SPLIT: a stage of no key of these queries is not added
#pragma unroll
        for (int half = 0; half < NH; half++) {
            const int hf = SPLIT ? wave & 1 : half;
            uint4 xh[2], xl[2], wb[2];
#pragma unroll
            for (int qt = 0; qt < 2; qt++) {
                uint2 hi[2], lo[2];
#pragma unroll
                for (int c = 0; c < 2; c++) {
                    const int kt = 2 * hf + c;
                    const uint4 av0 = ld_op(Vs[buf], 16 * kt, 0), av1 = ld_op(Vs[buf], 16 * kt, 1);
                    f32x4 dw = mfma32(av0, doh[qt][0], f32x4{0.f, 0.f, 0.f, 0.f});
                    dw = mfma32(av0, dol[qt][0], dw);
                    if constexpr (NKS == 2) dw = mfma32(av1, doh[qt][1], dw);
                    if constexpr (NKS == 2) dw = mfma32(av1, dol[qt][1], dw);
                    const uint2 wp = c ? make_uint2(wcur[half][qt].z, wcur[half][qt].w) : make_uint2(wcur[half][qt].x, wcur[half][qt].y);
                    f32x4 x;
                    split_products(wp.x, wp.y, dw, x, hi[c], lo[c]);
                    const float d4 = sum_products(wp.x, wp.y, dw, x, lo[c]);
                    if constexpr (SPLIT) Dx[wave][qt][c][l] = d4;
                    else dpart[qt] += d4;
                }
                xh[qt] = make_uint4(hi[0].x, hi[0].y, hi[1].x, hi[1].y);
                xl[qt] = make_uint4(lo[0].x, lo[0].y, lo[1].x, lo[1].y);
                wb[qt] = wcur[half][qt];
            }
            if constexpr (SPLIT) {
#pragma unroll
                for (int qt = 0; qt < 2; qt++) { Px[wave][qt][0][l] = xh[qt]; Px[wave][qt][1][l] = xl[qt]; Px[wave][qt][2][l] = wb[qt]; }
            } else {
                add(Ks[buf], hf, xh, xl, wb);
            }
        }
        if constexpr (SPLIT) {
            __syncthreads();   // the four half stages are there
#pragma unroll
            for (int p = 0; p < 2; p++) {
                if (st + p > st_hi) break;
#pragma unroll
                for (int hf = 0; hf < 2; hf++) {
                    const int h = 2 * p + hf;
                    const auto &x = Px[h][own.tile0];
                    dpart[0] += Dx[h][own.tile0][0][l];
                    dpart[0] += Dx[h][own.tile0][1][l];
                    add(Ks[p], hf, {x[0][l]}, {x[1][l]}, {x[2][l]});
                }
            }
        }
    }
#pragma unroll
    for (int t = 0; t < Own::NT; t++) {
        const int tq = qlo + 16 * (own.tile0 + t) + r;
        float dsum = dpart[t];
        dsum += __shfl_xor(dsum, 16, 64);
        dsum += __shfl_xor(dsum, 32, 64);
        if (tq < s) {
            if (g == 0 && own.dt0 == 0) dvec[(size_t)(b * H + h) * s + tq] = dsum;
            float *ob = d_q + (row0 + tq) * total + hoff;
#pragma unroll
            for (int dt = 0; dt < Own::ND; dt++)
                *reinterpret_cast<f32x4 *>(ob + 16 * (own.dt0 + dt) + 4 * g) = (aq[t][dt] - dsum * bq[t][dt]) * scale;
        }
    }
}

// Key pass on statistics, in query blocks (one workgroup per 128 keys, one wave per 32): over the stages of 64
// queries that see the block's keys, a wave forms S = Q K^T for its two key tiles (rows = queries, column = the
// lane's key), the weights from the queries' statistics, dW = dO V^T, dS = w (dW - D_t) / sqrt(hd), and
// accumulates d_v^T += dO^T w and d_k^T += Q^T dS.  The Q and dO rows of a stage are staged as they arrive (dO as
// hi + lo); the products that contract over queries read them through ds_read_b64_tr_b16 in the query order
// that the score tiles leave in the lanes.  K and V of the wave's keys sit in registers.
template <int HDV, bool OUT16, bool SPLIT>
__global__ __launch_bounds__(256, 2) void swa_bwd_k_stats_kernel(const unsigned short *__restrict__ q,
                                                                 const unsigned short *__restrict__ k,
                                                                 const unsigned short *__restrict__ v,
                                                                 const float2 *__restrict__ stats,
                                                                 const float *__restrict__ d_out,
                                                                 const float *__restrict__ dvec,
                                                                 float *__restrict__ d_k, float *__restrict__ d_v,
                                                                 int s, int H, int ws, Out16 o16) {
    constexpr int LD = SPLIT ? LDQ : LDH;
    __shared__ __align__(16) unsigned short QD[6][KS][LD];   // two stages [query][dim] of Q, then of dO's hi, then lo
    unsigned short (*const Qs)[KS][LD] = QD, (*const Dh)[KS][LD] = QD + 2, (*const Dl)[KS][LD] = QD + 4;
    __shared__ __align__(16) float Mc[2][KS], Iv[2][KS], Dd[2][KS];   // the stage's queries: maximum, 1 / sum, D
    __shared__ HalfStage<3> Px[SPLIT ? 4 : 1];   // SPLIT: dS hi and lo and w of a wave's half stage
    const int tid = threadIdx.x, wave = tid >> 6, l = tid & 63, r = l & 15, g = l >> 4;
    const BlockCoord bc = xcd_block_coord(H);
    const int j0 = bc.x * (SPLIT ? SQ : FQ), h = bc.h, b = bc.b;
    constexpr int NKS = HDV / 32, NDT = HDV / 16;
    constexpr float kInvSqrt = HDV == 64 ? 0.125f : 0.17677669529663687f;   // 1 / sqrt(head size)
    const int total = H * HDV, hoff = h * HDV;
    const size_t row0 = (size_t)b * s;
    const int jlo = SPLIT ? j0 : j0 + 32 * wave, jhi = jlo + 31;            // this wave's keys
    const int st_lo = j0 / KS, st_hi = min(s - 1, j0 + (SPLIT ? SQ : FQ) - 1 + ws - 1) / KS;
    const float *dvb = dvec + (size_t)(b * H + h) * s;
    const float2 *stb = stats + (size_t)(b * H + h) * s;
    const StageSrc qm{q, row0, total, hoff, s};
    const float c2 = kInvSqrt * 1.44269504088896340736f, scale = kInvSqrt;

    uint4 kf[2][2], vf[2][2];   // B operands: key jlo + 16 jt + r, dims 32 ks + 8 g ..
#pragma unroll
    for (int jt = 0; jt < 2; jt++)
#pragma unroll
        for (int ks = 0; ks < NKS; ks++) {
            const int key = jlo + 16 * jt + r;
            kf[jt][ks] = make_uint4(0, 0, 0, 0);
            vf[jt][ks] = make_uint4(0, 0, 0, 0);
            if (key < s) {
                const size_t o = (row0 + key) * total + hoff + 32 * ks + 8 * g;
                kf[jt][ks] = *reinterpret_cast<const uint4 *>(k + o);
                vf[jt][ks] = *reinterpret_cast<const uint4 *>(v + o);
            }
        }
    using Own = OwnTiles<NDT, SPLIT>;
    const Own own(wave);
    f32x4 dk[Own::NT][Own::ND], dv[Own::NT][Own::ND];   // d_k^T, d_v^T: rows = dims 16 dt + 4 g + i, column = key
#pragma unroll
    for (int t = 0; t < Own::NT; t++)
#pragma unroll
        for (int dt = 0; dt < Own::ND; dt++) { dk[t][dt] = f32x4{0.f, 0.f, 0.f, 0.f}; dv[t][dt] = f32x4{0.f, 0.f, 0.f, 0.f}; }
    // half hq of the stage in buffer `at` added to the sums of this wave's tiles
    auto add = [&](int at, int hq, const uint4(&dsh)[Own::NT], const uint4(&dsl)[Own::NT], const uint4(&wpk)[Own::NT])
                   __attribute__((always_inline)) {
        const int ra = 32 * hq + 4 * g, rb = ra + 16;
#pragma unroll
        for (int dt = 0; dt < Own::ND; dt++) {
            const uint4 aq = ld_tr2<LD>(Qs[at], ra, rb, 16 * (own.dt0 + dt));    // Q^T [dim][query]
            const uint4 ah = ld_tr2<LD>(Dh[at], ra, rb, 16 * (own.dt0 + dt));    // dO^T hi / lo
            const uint4 al = ld_tr2<LD>(Dl[at], ra, rb, 16 * (own.dt0 + dt));
#pragma unroll
            for (int t = 0; t < Own::NT; t++) {
                dk[t][dt] = mfma32(aq, dsh[t], dk[t][dt]);
                dk[t][dt] = mfma32(aq, dsl[t], dk[t][dt]);
                dv[t][dt] = mfma32(ah, wpk[t], dv[t][dt]);
                dv[t][dt] = mfma32(al, wpk[t], dv[t][dt]);
            }
        }
    };

    // one stage ahead in registers: Q rows (two 16-byte pieces per thread), dO rows (thread = quarter row)
    constexpr int NP = SPLIT ? 2 : 1;
    uint4 qreg[NP][2];
    f32x4 dreg[NP][4];
    float2 streg = make_float2(0.f, 0.f);
    float ddreg = 0.f;
    const int drow = tid >> 2, dcol = 16 * (tid & 3);
    auto fetch_stages = [&](int t_lo) {
#pragma unroll
        for (int p = 0; p < NP; p++) {
            load_rows<HDV>(qm, t_lo + KS * p, qreg[p]);
            const int t = t_lo + KS * p + drow;
#pragma unroll
            for (int c = 0; c < 4; c++) {
                dreg[p][c] = f32x4{0.f, 0.f, 0.f, 0.f};
                if (t < s && dcol < HDV) dreg[p][c] = *reinterpret_cast<const f32x4 *>(d_out + (row0 + t) * total + hoff + dcol + 4 * c);
            }
        }
        streg = make_float2(0.f, 0.f);
        ddreg = 0.f;
        if (tid < NP * KS && t_lo + tid < s) { streg = stb[t_lo + tid]; ddreg = dvb[t_lo + tid]; }
    };
    fetch_stages(KS * st_lo);
    for (int st = st_lo; st <= st_hi; st += NP) {
        const int buf = SPLIT ? wave >> 1 : (st - st_lo) & 1, t_lo = KS * (SPLIT ? st + buf : st);
        if (SPLIT && st > st_lo) __syncthreads();   // the stages and half stages before are read
#pragma unroll
        for (int p = 0; p < NP; p++)
#pragma unroll
            for (int c = 0; c < 2; c++) {
                const int chunk = tid + 256 * c, to = SPLIT ? p : buf;
                *reinterpret_cast<uint4 *>(&Qs[to][chunk >> 3][8 * (chunk & 7)]) = qreg[p][c];
                uint4 hi, lo;
                split8(dreg[p][2 * c], dreg[p][2 * c + 1], hi, lo);
                *reinterpret_cast<uint4 *>(&Dh[to][drow][dcol + 8 * c]) = hi;
                *reinterpret_cast<uint4 *>(&Dl[to][drow][dcol + 8 * c]) = lo;
            }
        if (tid < NP * KS) {
            const int to = SPLIT ? tid / KS : buf;
            Mc[to][tid % KS] = streg.x; Iv[to][tid % KS] = streg.y; Dd[to][tid % KS] = ddreg;
        }
        __syncthreads();
        if (st + NP - 1 < st_hi) fetch_stages(KS * (st + NP));
        // no query of this stage sees a key of this wave (SPLIT: such a stage is not added)
        if (!SPLIT && (t_lo + KS - 1 < jlo || t_lo > jhi + ws - 1)) continue;
        const bool full = t_lo >= jhi && t_lo + KS - 1 <= jlo + ws - 1 && t_lo + KS - 1 < s && jhi < s;
#pragma unroll
        for (int half = 0; half < 3 - NP; half++) {
            const int hq = SPLIT ? wave & 1 : half;
            uint4 wpk[2], dsh[2], dsl[2];
            uint2 hi[2][2], lo[2][2];
            unsigned wp[2][2][2];
#pragma unroll
            for (int c = 0; c < 2; c++) {
                const int qt = 2 * hq + c;
                const uint4 aq0 = ld_op(Qs[buf], 16 * qt, 0), aq1 = ld_op(Qs[buf], 16 * qt, 1);
                const uint4 ah0 = ld_op(Dh[buf], 16 * qt, 0), ah1 = ld_op(Dh[buf], 16 * qt, 1);
                const uint4 al0 = ld_op(Dl[buf], 16 * qt, 0), al1 = ld_op(Dl[buf], 16 * qt, 1);
                const f32x4 m4 = *reinterpret_cast<const f32x4 *>(&Mc[buf][16 * qt + 4 * g]);
                const f32x4 i4 = *reinterpret_cast<const f32x4 *>(&Iv[buf][16 * qt + 4 * g]);
                const f32x4 d4 = *reinterpret_cast<const f32x4 *>(&Dd[buf][16 * qt + 4 * g]);
#pragma unroll
                for (int jt = 0; jt < 2; jt++) {
                    f32x4 sc = mfma32(aq0, kf[jt][0], f32x4{0.f, 0.f, 0.f, 0.f});
                    if constexpr (NKS == 2) sc = mfma32(aq1, kf[jt][1], sc);
                    f32x4 dw = mfma32(ah0, vf[jt][0], -d4);   // dW - D
                    dw = mfma32(al0, vf[jt][0], dw);
                    if constexpr (NKS == 2) dw = mfma32(ah1, vf[jt][1], dw);
                    if constexpr (NKS == 2) dw = mfma32(al1, vf[jt][1], dw);
                    f32x4 w;
#pragma unroll
                    for (int i = 0; i < 4; i++) {
                        const int t = t_lo + 16 * qt + 4 * g + i, key = jlo + 16 * jt + r;
                        const bool ok = full || (key <= t && t <= key + ws - 1 && t < s && key < s);
                        w[i] = ok ? __builtin_amdgcn_exp2f(fmaf(sc[i], c2, -m4[i])) * i4[i] : 0.f;
                    }
                    wp[jt][c][0] = pack2(w[0], w[1]);   // as the weight tensor holds them
                    wp[jt][c][1] = pack2(w[2], w[3]);
                    f32x4 ds;
                    split_products(wp[jt][c][0], wp[jt][c][1], dw, ds, hi[jt][c], lo[jt][c]);
                }
            }
#pragma unroll
            for (int jt = 0; jt < 2; jt++) {
                wpk[jt] = make_uint4(wp[jt][0][0], wp[jt][0][1], wp[jt][1][0], wp[jt][1][1]);
                dsh[jt] = make_uint4(hi[jt][0].x, hi[jt][0].y, hi[jt][1].x, hi[jt][1].y);
                dsl[jt] = make_uint4(lo[jt][0].x, lo[jt][0].y, lo[jt][1].x, lo[jt][1].y);
            }
            if constexpr (SPLIT) {
#pragma unroll
                for (int jt = 0; jt < 2; jt++) { Px[wave][jt][0][l] = dsh[jt]; Px[wave][jt][1][l] = dsl[jt]; Px[wave][jt][2][l] = wpk[jt]; }
            } else {
                add(buf, hq, dsh, dsl, wpk);
            }
        }
        if constexpr (SPLIT) {
            __syncthreads();   // the four half stages are there
#pragma unroll
            for (int p = 0; p < 2; p++) {
                if (st + p > st_hi) break;
#pragma unroll
                for (int hq = 0; hq < 2; hq++) {
                    const auto &x = Px[2 * p + hq][own.tile0];
                    add(p, hq, {x[0][l]}, {x[1][l]}, {x[2][l]});
                }
            }
        }
    }
    // accumulate: column = key jlo + 16 jt + r, rows = dims 16 dt + 4 g ..
#pragma unroll
    for (int t = 0; t < Own::NT; t++) {
        const int key = jlo + 16 * (own.tile0 + t) + r;
        if (key >= s) continue;
        if (OUT16) {
            unsigned short *pk = o16.k + (row0 + key) * o16.ld + hoff, *pv = o16.v + (row0 + key) * o16.ld + hoff;
#pragma unroll
            for (int dt = 0; dt < Own::ND; dt++) {
                const int at = 16 * (own.dt0 + dt) + 4 * g;
                const f32x4 a = dk[t][dt] * scale, c = dv[t][dt];
                *reinterpret_cast<uint2 *>(pk + at) = make_uint2(pack2(a[0], a[1]), pack2(a[2], a[3]));
                *reinterpret_cast<uint2 *>(pv + at) = make_uint2(pack2(c[0], c[1]), pack2(c[2], c[3]));
            }
            continue;
        }
        float *pk = d_k + (row0 + key) * total + hoff, *pv = d_v + (row0 + key) * total + hoff;
#pragma unroll
        for (int dt = 0; dt < Own::ND; dt++) {
            const int at = 16 * (own.dt0 + dt) + 4 * g;
            f32x4 *ck = reinterpret_cast<f32x4 *>(pk + at), *cv = reinterpret_cast<f32x4 *>(pv + at);
            *ck = *ck + dk[t][dt] * scale;
            *cv = *cv + dv[t][dt];
        }
    }
}

// Key pass of the contract in query blocks, like swa_bwd_k_stats_kernel, with the weights read back from the tensor:
// the stage's 64 query rows x the block's 128 keys are 256 contiguous bytes per query where the window covers them;
// they are staged in LDS as [query][key] and a lane takes its two tiles (rows = queries, column = its key) with one
// transposing read, which is both the B operand of d_v^T += dO^T w and the w of dS = w (dW - D_t); -D_t is what the sum of
// dW starts from, 1 / sqrt(hd) is applied to the sum.  Same size as above: 232 us (266 with a wait for slots read one by one
// in the stages at the window's ends and two more vector instructions an element).
constexpr int LDW = 144;   // row stride of the weight stage (288 B: the transposing reads of a group fall on 32 banks)

template <int HDV, bool SPLIT>
__global__ __launch_bounds__(256, 2) void swa_bwd_k_blocked_kernel(const unsigned short *__restrict__ q,
                                                                   const unsigned short *__restrict__ v,
                                                                   const unsigned short *__restrict__ attn_w,
                                                                   const float *__restrict__ d_out,
                                                                   const float *__restrict__ dvec,
                                                                   float *__restrict__ d_k, float *__restrict__ d_v,
                                                                   int s, int H, int ws) {
    constexpr int NP = SPLIT ? 2 : 1, LDK = SPLIT ? SQ : LDW, LD = SPLIT ? LDQ : LDH;
    __shared__ __align__(16) unsigned short QD[6][KS][LD];    // two stages [query][dim] of Q, then of dO's hi, then lo
    __shared__ __align__(16) unsigned short Wt[NP * KS][LDK];  // [query][key of the block]
    unsigned short (*const Qs)[KS][LD] = QD, (*const Dh)[KS][LD] = QD + 2, (*const Dl)[KS][LD] = QD + 4;
    __shared__ __align__(16) float Dd[2][KS];
    __shared__ HalfStage<2> Px[SPLIT ? 4 : 1];   // SPLIT: dS hi and lo of a wave's half stage
    const int tid = threadIdx.x, wave = tid >> 6, l = tid & 63, r = l & 15, g = l >> 4;
    const BlockCoord bc = xcd_block_coord(H);
    const int j0 = bc.x * (SPLIT ? SQ : FQ), h = bc.h, b = bc.b;
    constexpr int NKS = HDV / 32, NDT = HDV / 16;
    constexpr float kInvSqrt = HDV == 64 ? 0.125f : 0.17677669529663687f;   // 1 / sqrt(head size)
    const int total = H * HDV, hoff = h * HDV;
    const size_t row0 = (size_t)b * s;
    const int jlo = SPLIT ? j0 : j0 + 32 * wave, jhi = jlo + 31;
    const int st_lo = j0 / KS, st_hi = min(s - 1, j0 + (SPLIT ? SQ : FQ) - 1 + ws - 1) / KS;
    const float *dvb = dvec + (size_t)(b * H + h) * s;
    const float scale = kInvSqrt;
    const unsigned short *awb = attn_w + (size_t)(b * H + h) * s * ws;
    const bool at_edge = edge_head(b * H + h, (int)(gridDim.y * gridDim.z), s, ws);
    const StageSrc qm{q, row0, total, hoff, s};

    uint4 vf[2][2];
#pragma unroll
    for (int jt = 0; jt < 2; jt++)
#pragma unroll
        for (int ks = 0; ks < NKS; ks++) {
            const int key = jlo + 16 * jt + r;
            vf[jt][ks] = make_uint4(0, 0, 0, 0);
            if (key < s) vf[jt][ks] = *reinterpret_cast<const uint4 *>(v + (row0 + key) * total + hoff + 32 * ks + 8 * g);
        }
    using Own = OwnTiles<NDT, SPLIT>;
    const Own own(wave);
    f32x4 dk[Own::NT][Own::ND], dv[Own::NT][Own::ND];   // d_k^T, d_v^T: rows = dims 16 dt + 4 g + i, column = key
#pragma unroll
    for (int t = 0; t < Own::NT; t++)
#pragma unroll
        for (int dt = 0; dt < Own::ND; dt++) { dk[t][dt] = f32x4{0.f, 0.f, 0.f, 0.f}; dv[t][dt] = f32x4{0.f, 0.f, 0.f, 0.f}; }
    // half hq of the stage in buffer `at` added to the sums of this wave's tiles
    auto add = [&](int at, int hq, const uint4(&dsh)[Own::NT], const uint4(&dsl)[Own::NT], const uint4(&wpk)[Own::NT])
                   __attribute__((always_inline)) {
        const int ra = 32 * hq + 4 * g, rb = ra + 16;
#pragma unroll
        for (int dt = 0; dt < Own::ND; dt++) {
            const uint4 aq = ld_tr2<LD>(Qs[at], ra, rb, 16 * (own.dt0 + dt));    // Q^T [dim][query]
            const uint4 ah = ld_tr2<LD>(Dh[at], ra, rb, 16 * (own.dt0 + dt));    // dO^T hi / lo
            const uint4 al = ld_tr2<LD>(Dl[at], ra, rb, 16 * (own.dt0 + dt));
#pragma unroll
            for (int t = 0; t < Own::NT; t++) {
                dk[t][dt] = mfma32(aq, dsh[t], dk[t][dt]);
                dk[t][dt] = mfma32(aq, dsl[t], dk[t][dt]);
                dv[t][dt] = mfma32(ah, wpk[t], dv[t][dt]);
                dv[t][dt] = mfma32(al, wpk[t], dv[t][dt]);
            }
        }
    };

    // Weights: thread (query drow, quarter) reads the quarter's pieces of eight keys of the query's row
    constexpr int NW = SPLIT ? 1 : 4, QK = 8 * NW;
    uint4 qreg[NP][2], wreg[NP][NW];
    f32x4 dreg[NP][4];
    float ddreg = 0.f;
    const int drow = tid >> 2, dcol = 16 * (tid & 3);
    auto fetch_stages = [&](int t_lo) {
        ddreg = (tid < NP * KS && t_lo + tid < s) ? dvb[t_lo + tid] : 0.f;
#pragma unroll
        for (int p = 0; p < NP; p++) {
            load_rows<HDV>(qm, t_lo + KS * p, qreg[p]);
            const int t = t_lo + KS * p + drow;
#pragma unroll
            for (int c = 0; c < 4; c++) {
                dreg[p][c] = f32x4{0.f, 0.f, 0.f, 0.f};
                if (t < s && dcol < HDV) dreg[p][c] = *reinterpret_cast<const f32x4 *>(d_out + (row0 + t) * total + hoff + dcol + 4 * c);
            }
            // pieces are read whole at the window's ends too (out of the rows next to it) and freed of what is not the
            // query's own where they go to LDS
            const int lsq = max(t + 1 - ws, 0), thi = t < s ? t : -1;
            const unsigned short *wrow = awb + (size_t)t * ws;
#pragma unroll
            for (int c = 0; c < NW; c++) {
                const int key0 = j0 + QK * (tid & 3) + 8 * c;
                wreg[p][c] = make_uint4(0, 0, 0, 0);
                if (key0 + 7 >= lsq && key0 <= thi) {
                    if (!at_edge || piece_inside(t, s, ws, key0 - lsq)) {
                        __builtin_memcpy(&wreg[p][c], wrow + (key0 - lsq), 16);
                    } else {   // at the tensor's own ends
                        unsigned d[4] = {0u, 0u, 0u, 0u};
#pragma unroll
                        for (int e = 0; e < 8; e++) {
                            const int key = key0 + e;
                            unsigned x = 0;
                            if (key >= lsq && key <= thi) x = wrow[key - lsq];
                            d[e >> 1] |= x << (16 * (e & 1));
                        }
                        wreg[p][c] = make_uint4(d[0], d[1], d[2], d[3]);
                    }
                }
            }
        }
    };
    // weights of half hq of the stage in buffer `at` for key tile jt
    auto weights = [&](int at, int hq, int jt) __attribute__((always_inline)) {
        const int ra = 32 * hq + 4 * g;
        return ld_tr2<LDK>(Wt + (SPLIT ? KS * at : 0), ra, ra + 16, (SPLIT ? 0 : 32 * wave) + 16 * jt);
    };
    fetch_stages(KS * st_lo);
    for (int st = st_lo; st <= st_hi; st += NP) {
        const int buf = SPLIT ? wave >> 1 : (st - st_lo) & 1, t_lo = KS * (SPLIT ? st + buf : st);
#pragma unroll
        for (int p = 0; p < NP; p++) {
            const int to = SPLIT ? p : buf, t_p = KS * (st + p);
            const bool inner = t_p >= j0 + (SPLIT ? SQ : FQ) - 1 && t_p + KS - 1 <= j0 + ws - 1 && t_p + KS - 1 < s;   // every query sees every key
#pragma unroll
            for (int c = 0; c < 2; c++) {
                const int chunk = tid + 256 * c;
                *reinterpret_cast<uint4 *>(&Qs[to][chunk >> 3][8 * (chunk & 7)]) = qreg[p][c];
                uint4 hi, lo;
                split8(dreg[p][2 * c], dreg[p][2 * c + 1], hi, lo);
                *reinterpret_cast<uint4 *>(&Dh[to][drow][dcol + 8 * c]) = hi;
                *reinterpret_cast<uint4 *>(&Dl[to][drow][dcol + 8 * c]) = lo;
            }
#pragma unroll
            for (int c = 0; c < NW; c++) {
                uint4 &w = wreg[p][c];
                if (!inner) {
                    const int t = t_p + drow, key0 = j0 + QK * (tid & 3) + 8 * c;
                    const int first = max(t + 1 - ws, 0) - key0, last = (t < s ? t : -1) - key0;
                    if (__any(first > 0 || last < 7)) {
                        w.x &= own_pair(0, first, last);
                        w.y &= own_pair(2, first, last);
                        w.z &= own_pair(4, first, last);
                        w.w &= own_pair(6, first, last);
                    }
                }
                *reinterpret_cast<uint4 *>(&Wt[KS * (SPLIT ? p : 0) + drow][QK * (tid & 3) + 8 * c]) = w;
            }
        }
        if (tid < NP * KS) Dd[SPLIT ? tid / KS : buf][tid % KS] = ddreg;
        __syncthreads();
        if (st + NP - 1 < st_hi) fetch_stages(KS * (st + NP));
        // a query of this stage sees a key of this wave (SPLIT: a stage without one is not added)
        if (SPLIT || !(t_lo + KS - 1 < jlo || t_lo > jhi + ws - 1)) {
#pragma unroll
            for (int half = 0; half < 3 - NP; half++) {
                const int hq = SPLIT ? wave & 1 : half;
                uint4 wpk[2], dsh[2], dsl[2];
                uint2 hi[2][2], lo[2][2];
#pragma unroll
                for (int jt = 0; jt < 2; jt++) wpk[jt] = weights(buf, hq, jt);
#pragma unroll
                for (int c = 0; c < 2; c++) {
                    const int qt = 2 * hq + c;
                    const uint4 ah0 = ld_op(Dh[buf], 16 * qt, 0), ah1 = ld_op(Dh[buf], 16 * qt, 1);
                    const uint4 al0 = ld_op(Dl[buf], 16 * qt, 0), al1 = ld_op(Dl[buf], 16 * qt, 1);
                    const f32x4 d4 = *reinterpret_cast<const f32x4 *>(&Dd[buf][16 * qt + 4 * g]);
#pragma unroll
                    for (int jt = 0; jt < 2; jt++) {
                        f32x4 dw = mfma32(ah0, vf[jt][0], -d4);   // dW - D
                        dw = mfma32(al0, vf[jt][0], dw);
                        if constexpr (NKS == 2) dw = mfma32(ah1, vf[jt][1], dw);
                        if constexpr (NKS == 2) dw = mfma32(al1, vf[jt][1], dw);
                        const unsigned w01 = c ? wpk[jt].z : wpk[jt].x, w23 = c ? wpk[jt].w : wpk[jt].y;
                        f32x4 ds;
                        split_products(w01, w23, dw, ds, hi[jt][c], lo[jt][c]);
                    }
                }
#pragma unroll
                for (int jt = 0; jt < 2; jt++) {
                    dsh[jt] = make_uint4(hi[jt][0].x, hi[jt][0].y, hi[jt][1].x, hi[jt][1].y);
                    dsl[jt] = make_uint4(lo[jt][0].x, lo[jt][0].y, lo[jt][1].x, lo[jt][1].y);
                }
                if constexpr (SPLIT) {
#pragma unroll
                    for (int jt = 0; jt < 2; jt++) { Px[wave][jt][0][l] = dsh[jt]; Px[wave][jt][1][l] = dsl[jt]; }
                } else {
                    add(buf, hq, dsh, dsl, wpk);
                }
            }
        }
        if constexpr (SPLIT) {
            __syncthreads();   // the four half stages are there
#pragma unroll
            for (int p = 0; p < 2; p++) {
                if (st + p > st_hi) break;
#pragma unroll
                for (int hq = 0; hq < 2; hq++) {
                    const auto &x = Px[2 * p + hq][own.tile0];
                    add(p, hq, {x[0][l]}, {x[1][l]}, {weights(p, hq, own.tile0)});
                }
            }
        }
        __syncthreads();   // the weight stage has one buffer: every wave is done with it before the next one lands
    }
#pragma unroll
    for (int t = 0; t < Own::NT; t++) {
        const int key = jlo + 16 * (own.tile0 + t) + r;
        if (key >= s) continue;
        float *pk = d_k + (row0 + key) * total + hoff, *pv = d_v + (row0 + key) * total + hoff;
#pragma unroll
        for (int dt = 0; dt < Own::ND; dt++) {
            const int at = 16 * (own.dt0 + dt) + 4 * g;
            f32x4 *ck = reinterpret_cast<f32x4 *>(pk + at), *cv = reinterpret_cast<f32x4 *>(pv + at);
            *ck = *ck + dk[t][dt] * scale;
            *cv = *cv + dv[t][dt];
        }
    }
}

}  // namespace

bool swa_forward_mfma(const uint16_t *q, const uint16_t *k, const uint16_t *v, uint16_t *out, uint16_t *attn_weights,
                      int seq_len, int num_heads, int head_dim, int window, int batch, int n_persistent, float *stats) {
    if ((head_dim != 64 && head_dim != 32) || n_persistent != 0 || window > 512 || window < 1) return false;
    const bool few = (long long)ceil_div(seq_len, FQ) * num_heads * batch < 2LL * compute_units();
    const dim3 grid(ceil_div(seq_len, few ? FQ / 2 : FQ), num_heads, batch);
    const bool wide = head_dim == 64;
    if (stats) {
        KernelTimer kt("swa_fwd_stats_kernel");
        auto kernel = wide ? (few ? swa_fwd_stats_kernel<64, 1> : swa_fwd_stats_kernel<64, 2>)
                           : (few ? swa_fwd_stats_kernel<32, 1> : swa_fwd_stats_kernel<32, 2>);
        hipLaunchKernelGGL(kernel, grid, dim3(256), 0, stream(), q, k, v, out, reinterpret_cast<float2 *>(stats), seq_len, num_heads, window);
        check_launch("swa_fwd_stats_kernel");
        return true;
    }
    KernelTimer kt("swa_fwd_blocked_kernel");
    const bool pieces = window % 8 == 0 && ((uintptr_t)attn_weights & 15) == 0;   // rows of whole 16-byte pieces
    auto kernel = few ? (wide ? (pieces ? swa_fwd_blocked_kernel<64, true, 1> : swa_fwd_blocked_kernel<64, false, 1>)
                              : (pieces ? swa_fwd_blocked_kernel<32, true, 1> : swa_fwd_blocked_kernel<32, false, 1>))
                      : (wide ? (pieces ? swa_fwd_blocked_kernel<64, true, 2> : swa_fwd_blocked_kernel<64, false, 2>)
                              : (pieces ? swa_fwd_blocked_kernel<32, true, 2> : swa_fwd_blocked_kernel<32, false, 2>));
    hipLaunchKernelGGL(kernel, grid, dim3(256), 0, stream(), q, k, v, out, attn_weights, seq_len, num_heads, window);
    check_launch("swa_fwd_blocked_kernel");
    return true;
}

// f with the head size, the kind of output and SPLIT as types
template <class F>
static void choose(bool wide, bool out16, bool split, F f) {
    auto third = [&](auto hd, auto o) { if (split) f(hd, o, std::true_type{}); else f(hd, o, std::false_type{}); };
    auto second = [&](auto hd) { if (out16) third(hd, std::true_type{}); else third(hd, std::false_type{}); };
    if (wide) second(std::integral_constant<int, 64>{}); else second(std::integral_constant<int, 32>{});
}

bool swa_backward_mfma(const uint16_t *q, const uint16_t *k, const uint16_t *v, const uint16_t *attn_weights,
                       const float *d_attn_out, float *d_q, float *d_k, float *d_v, int seq_len, int num_heads,
                       int head_dim, int window, int batch, int n_persistent, const float *stats, const SwaGradCols *cols) {
    const ErrorScope es;
    if ((head_dim != 64 && head_dim != 32) || n_persistent != 0 || window > 512 || window < 1) return false;
    float *dvec = scratch(1, (size_t)batch * num_heads * seq_len * sizeof(float));
    if (es.failed()) return true;
    // 32 rows a workgroup while those fit the chip at once, two to a compute unit (both sides at SQ)
    const bool split = 2ll * ceil_div(seq_len, FQ) * num_heads * batch <= compute_units();
    const dim3 grid(ceil_div(seq_len, split ? SQ : FQ), num_heads, batch);
    const bool wide = head_dim == 64;
    if (stats) {
        const float2 *st2 = reinterpret_cast<const float2 *>(stats);
        const Out16 o16 = cols ? Out16{cols->q, cols->k, cols->v, cols->ld} : Out16{nullptr, nullptr, nullptr, 0};
        auto both = [&](auto hd, auto out16, auto halves) {
            constexpr int HDV = decltype(hd)::value;
            constexpr bool O16 = decltype(out16)::value, SPLIT = decltype(halves)::value;
            {
                KernelTimer kt("swa_bwd_q_stats_kernel");
                hipLaunchKernelGGL((swa_bwd_q_stats_kernel<HDV, O16, SPLIT>), grid, dim3(256), 0, stream(), q, k, v, st2, d_attn_out,
                                   d_q, dvec, seq_len, num_heads, window, o16);
                check_launch("swa_bwd_q_stats_kernel");
            }
            KernelTimer kt("swa_bwd_k_stats_kernel");
            hipLaunchKernelGGL((swa_bwd_k_stats_kernel<HDV, O16, SPLIT>), grid, dim3(256), 0, stream(), q, k, v, st2, d_attn_out,
                               dvec, d_k, d_v, seq_len, num_heads, window, o16);
            check_launch("swa_bwd_k_stats_kernel");
        };
        choose(wide, cols != nullptr, split, both);
        return true;
    }
    if (cols) return false;   // bf16 column output exists for the statistics pair only
    choose(wide, false, split, [&](auto hd, auto, auto halves) {
        constexpr int HDV = decltype(hd)::value;
        constexpr bool SPLIT = decltype(halves)::value;
        {
            KernelTimer kt("swa_bwd_q_blocked_kernel");
            hipLaunchKernelGGL((swa_bwd_q_blocked_kernel<HDV, SPLIT>), grid, dim3(256), 0, stream(), k, v, attn_weights, d_attn_out,
                               d_q, dvec, seq_len, num_heads, window);
            check_launch("swa_bwd_q_blocked_kernel");
        }
        KernelTimer kt("swa_bwd_k_blocked_kernel");
        hipLaunchKernelGGL((swa_bwd_k_blocked_kernel<HDV, SPLIT>), grid, dim3(256), 0, stream(), q, v, attn_weights, d_attn_out, dvec,
                           d_k, d_v, seq_len, num_heads, window);
        check_launch("swa_bwd_k_blocked_kernel");
    });
    return true;
}

}  // namespace nlh
