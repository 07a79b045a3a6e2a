// One decode step of cached generation, token id in and logits out (core/src/gpu_forward.rs:3377-3492,
// gpu_single_token_forward), as four dependent launches.
//
// A token is a chain of matrix-vector products over weights that are each read once, so the step is bound by the
// weights' bytes and by the length of the chain, not by arithmetic.  Written as one launch per operation (embedding
// row, one product per projection, casts, cache copies, row norms, gates, head splits, the rule, attention, combine,
// two more products) a step of four levels is 44 launches of 2 to 50 us each behind 0.5 ms of host work; here it is
//   1. decode_project_kernel   every product with the embedded token: attention q, k, v (k and v rounded straight into
//                              their cache row) and the levels' k, v, q, one wave per four rows
//   2. decode_heads_kernel     per (level, head): row norms, gates, memory update, read; per (head, slice of the
//                              window): attention scores and the slice's share of the output.  All independent.
//   3. decode_output_kernel    attention slices merged, levels combined, sigmoid gate, output projection
//   4. decode_logits_kernel    the unembedding, written to the workspace and to host-visible memory
// Measured on one MI355X at d = 512, four levels of which one is active, window 512, vocabulary 32 000: 0.50 -> 0.048 ms
// a token with the host side, of which 4.1 + 4.4 + 4.9 + 12.2 us in the four kernels (the last one moves 65 MB at
// 5.4 TB/s) and about 11 us before the first one starts and after the last one has ended.
#include <float.h>
#include <hip/hip_runtime.h>
#include <stdint.h>

#include "../../include/nl_hecate_ffi.h"
#include "rule_common.h"
#include "runtime.h"

namespace nlh {
namespace {

constexpr int kDecThr = 256;
constexpr int kMaxLevels = 8;
constexpr int kSliceKeys = 128;   // keys of the window per attention workgroup: 4 passes of 32 (head size 64)

struct DecLevel {
    const float *w_alpha, *b_alpha, *w_theta, *b_theta;
    float *memory;               // [heads, hd*hd]
    float *k, *v, *q, *y;        // [d] each, in the work buffer
    float alpha_floor, alpha_ceil, theta_floor, theta_ceil, clip, m_norm;
    int rule;                    // -1 frozen (read only), 0 Hebbian, 1 Delta / Titans, 2 DGD, 3 read with the normalised q
};
struct DecArgs {
    const float *x;              // the token's embedding row
    const float *w_o;
    uint16_t *q_bf16;
    const uint16_t *k_cache, *v_cache;
    float *part_o, *part_ml;     // attention slices: [slice][d], [slice][heads][2]
    float *embedded, *attn_out, *y_combined, *gate, *gated, *projected;
    uint16_t *attn_bf16;
    int d, nh, hd_log2, levels, pos, window, n_persistent, slices;
    DecLevel lv[kMaxLevels];
    // the products with the embedded token: d rows each, outputs q, k, v of the attention (rounded) or floats
    const float *seg_w[3 + 3 * kMaxLevels];
    void *seg_out[3 + 3 * kMaxLevels];
};

__device__ __forceinline__ float bf2f(uint16_t u) { return __uint_as_float((uint32_t)u << 16); }
__device__ __forceinline__ float dot4(const float4 &a, const float4 &b) { return a.x * b.x + a.y * b.y + a.z * b.z + a.w * b.w; }

__host__ __device__ inline bool reads_only(int rule) { return rule < 0 || rule == 3; }

// Segments of d rows in the order: attention q, k, v, then per active level k, v, q, per frozen level q; their addresses come
// by number (a search over the levels' rules, one scalar load after the other, stood ahead of every other load: 4.85 -> 4.05 us
// at d = 512, four levels of which one is active).
__global__ __launch_bounds__(kDecThr) void decode_project_kernel(DecArgs a) {
    const int lane = threadIdx.x & 63, seg = blockIdx.y, n4 = a.d >> 2;   // d is a multiple of 32: whole workgroups of 16 rows
    const int r = 16 * blockIdx.x + 4 * __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const float *w = a.seg_w[seg];
    float *out = seg < 3 ? nullptr : (float *)a.seg_out[seg];
    uint16_t *out16 = (uint16_t *)a.seg_out[seg];
    const float4 *x = reinterpret_cast<const float4 *>(a.x);
    const float4 *w0 = reinterpret_cast<const float4 *>(w + (size_t)r * a.d);
    float acc[4] = {0.f, 0.f, 0.f, 0.f};
    for (int i0 = lane; i0 < n4; i0 += 128) {   // 512 columns of four rows in flight
        float4 xv[2], wv[2][4];
#pragma unroll
        for (int q = 0; q < 2; q++) {
            const int i = min(i0 + 64 * q, n4 - 1);
            xv[q] = i0 + 64 * q < n4 ? x[i] : f4_zero();
#pragma unroll
            for (int j = 0; j < 4; j++) wv[q][j] = w0[(size_t)j * n4 + i];
        }
#pragma unroll
        for (int q = 0; q < 2; q++)
#pragma unroll
            for (int j = 0; j < 4; j++) acc[j] += dot4(wv[q][j], xv[q]);
    }
#pragma unroll
    for (int j = 0; j < 4; j++) acc[j] = wave_allreduce(acc[j]);
    if (lane < 4) {
        const float y = lane == 0 ? acc[0] : lane == 1 ? acc[1] : lane == 2 ? acc[2] : acc[3];
        if (out) out[r + lane] = y;
        else out16[r + lane] = f32_to_bf16_rne(y);
    }
    if (blockIdx.x == 0 && seg == 0)
        for (int i = threadIdx.x; i < n4; i += kDecThr) reinterpret_cast<float4 *>(a.embedded)[i] = x[i];
}

template <int N>
__device__ __forceinline__ void block_sums(float (&v)[N], float *red) {
    const int lane = threadIdx.x & 63, w = threadIdx.x >> 6;
#pragma unroll
    for (int i = 0; i < N; i++) v[i] = wave_allreduce(v[i]);
    __syncthreads();   // red may still be read from the sums before
    if (lane == 0) {
#pragma unroll
        for (int i = 0; i < N; i++) red[w * N + i] = v[i];
    }
    __syncthreads();
#pragma unroll
    for (int i = 0; i < N; i++) v[i] = (red[i] + red[N + i]) + (red[2 * N + i] + red[3 * N + i]);
}

// One (level, head): the memory matrix in registers, kDecThr / HD lanes per row, lane c of a row holding the 16-byte
// pieces at columns 4 (c + LPR i).
template <int HD>
__device__ __forceinline__ void level_head(const DecArgs &a, int l, int h, float *red) {
    constexpr int LPR = kDecThr / HD, NP = HD / (4 * LPR);
    const DecLevel &lv = a.lv[l];
    const int tid = threadIdx.x, row = tid / LPR, c = tid % LPR, d = a.d, hoff = h * HD;
    float4 *Mg = reinterpret_cast<float4 *>(lv.memory + (size_t)h * HD * HD) + row * (HD / 4) + c;
    float4 m[NP], qv[NP];
#pragma unroll
    for (int i = 0; i < NP; i++) m[i] = Mg[LPR * i];
    const float4 *qh = reinterpret_cast<const float4 *>(lv.q + hoff) + c;
#pragma unroll
    for (int i = 0; i < NP; i++) qv[i] = qh[LPR * i];
    float y = 0.f;
    if (reads_only(lv.rule)) {   // y = M q, with the raw projection for a frozen level
        float n2[1] = {0.f};
        if (lv.rule == 3) {
            for (int i = tid; i < d; i += kDecThr) n2[0] += lv.q[i] * lv.q[i];
            block_sums(n2, red);
        }
#pragma unroll
        for (int i = 0; i < NP; i++) y += dot4(m[i], qv[i]);
        y = group_allreduce<LPR>(y) * (lv.rule == 3 ? 1.f / fmaxf(sqrtf(n2[0]), 1e-8f) : 1.f);
        if (c == 0) lv.y[hoff + row] = y;
        return;
    }
    float4 kv[NP];
    const float4 *kh = reinterpret_cast<const float4 *>(lv.k + hoff) + c;
#pragma unroll
    for (int i = 0; i < NP; i++) kv[i] = kh[LPR * i];
    const float vr = lv.v[hoff + row];
    // norms of k and q over the model width, and the gate products (k enters normalised: scaled afterwards)
    float s[6] = {0.f, 0.f, 0.f, 0.f, 0.f, 0.f};
    for (int i = tid; i < d; i += kDecThr) {
        const float kk = lv.k[i], qq = lv.q[i], vv = lv.v[i];
        s[0] += kk * kk;
        s[1] += qq * qq;
        s[2] += kk * lv.w_alpha[i];
        s[3] += vv * lv.w_alpha[d + i];
        s[4] += kk * lv.w_theta[i];
        s[5] += vv * lv.w_theta[d + i];
    }
    block_sums(s, red);
    const float ki = 1.f / fmaxf(sqrtf(s[0]), 1e-8f), qi = 1.f / fmaxf(sqrtf(s[1]), 1e-8f);
    float alpha = 1.f / (1.f + expf(-(s[2] * ki + s[3] + lv.b_alpha[0])));
    const float zt = s[4] * ki + s[5] + lv.b_theta[0];
    float theta = zt > 20.f ? zt : log1pf(expf(zt));
    alpha = clamp_gate(alpha, lv.alpha_floor, lv.alpha_ceil, 1.f);
    theta = clamp_gate(theta, lv.theta_floor, lv.theta_ceil, FLT_MAX);
    float u = 0.f;
#pragma unroll
    for (int i = 0; i < NP; i++) { kv[i] = f4_scale(ki, kv[i]); qv[i] = f4_scale(qi, qv[i]); u += dot4(m[i], kv[i]); }
    float coef;   // M' = (1 - alpha) M + coef k^T
    if (lv.rule == 0) coef = vr;
    else {
        float e = group_allreduce<LPR>(u) - vr;
        if (lv.clip > 0.f) {
            float n2[1] = {c == 0 ? e * e : 0.f};
            block_sums(n2, red);
            const float n = sqrtf(n2[0]);
            if (n > lv.clip) e *= lv.clip / n;
        }
        coef = -theta * e;
    }
    float sq = 0.f;
#pragma unroll
    for (int i = 0; i < NP; i++) { m[i] = f4_axpby(1.f - alpha, m[i], coef, kv[i]); sq += dot4(m[i], m[i]); }
    float scale = 1.f;
    if (mnorm_active(lv.m_norm)) {
        float n2[1] = {sq};
        block_sums(n2, red);
        const float n = sqrtf(n2[0]);
        if (n > lv.m_norm) scale = lv.m_norm / n;
    }
    // Delta and Titans project inside the token, before the read; the others' carried memory is clamped after it
    const float read = lv.rule == 1 ? scale : 1.f;
#pragma unroll
    for (int i = 0; i < NP; i++) { y += dot4(m[i], qv[i]); Mg[LPR * i] = f4_scale(scale, m[i]); }
    y = group_allreduce<LPR>(y) * read;
    if (c == 0) lv.y[hoff + row] = y;
}

// One (head, slice of the visible keys): HD / 8 lanes per key, each eight dims; every K and V load of the slice is
// issued before the first is used.
template <int HD>
__device__ __forceinline__ void attention_slice(const DecArgs &a, int h, int slice, float *red) {
    constexpr int LPK = HD / 8, KPP = kDecThr / LPK, NP = kSliceKeys / KPP;   // keys per pass, passes
    const int tid = threadIdx.x, lane = tid & 63, w = tid >> 6, c = tid % LPK, g = tid / LPK;
    const int n_pre = min(a.pos + 1, a.n_persistent), ls = max(a.pos + 1 - a.window, a.n_persistent);
    const int n_keys = n_pre + max(0, a.pos + 1 - ls);
    const float sc = rsqrtf((float)HD);
    float qf[8];
    {
        const uint4 q = *reinterpret_cast<const uint4 *>(a.q_bf16 + h * HD + 8 * c);
        const uint32_t u[4] = {q.x, q.y, q.z, q.w};
#pragma unroll
        for (int i = 0; i < 4; i++) { qf[2 * i] = __uint_as_float(u[i] << 16); qf[2 * i + 1] = __uint_as_float(u[i] & 0xffff0000u); }
    }
    uint4 kk[NP], vv[NP];
    bool ok[NP];
#pragma unroll
    for (int p = 0; p < NP; p++) {
        const int slot = slice * kSliceKeys + p * KPP + g;
        ok[p] = slot < n_keys;
        const int key = !ok[p] ? a.pos : slot < n_pre ? slot : ls + slot - n_pre;
        const size_t at = (size_t)key * a.d + h * HD + 8 * c;
        kk[p] = *reinterpret_cast<const uint4 *>(a.k_cache + at);
        vv[p] = *reinterpret_cast<const uint4 *>(a.v_cache + at);
    }
    float s[NP], mx = -FLT_MAX;
#pragma unroll
    for (int p = 0; p < NP; p++) {
        const uint32_t u[4] = {kk[p].x, kk[p].y, kk[p].z, kk[p].w};
        float acc = 0.f;
#pragma unroll
        for (int i = 0; i < 4; i++)
            acc = fmaf(qf[2 * i + 1], __uint_as_float(u[i] & 0xffff0000u), fmaf(qf[2 * i], __uint_as_float(u[i] << 16), acc));
        s[p] = ok[p] ? group_allreduce<LPK>(acc) * sc : -FLT_MAX;
        mx = fmaxf(mx, s[p]);
    }
#pragma unroll
    for (int o = 32; o > 0; o >>= 1) mx = fmaxf(mx, __shfl_xor(mx, o, 64));
    if (lane == 0) red[w] = mx;
    __syncthreads();
    mx = fmaxf(fmaxf(red[0], red[1]), fmaxf(red[2], red[3]));
    float sum = 0.f, o[8] = {0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int p = 0; p < NP; p++) {
        const float e = ok[p] ? expf(s[p] - mx) : 0.f;
        sum += e;
        const uint32_t u[4] = {vv[p].x, vv[p].y, vv[p].z, vv[p].w};
#pragma unroll
        for (int i = 0; i < 4; i++) {
            o[2 * i] = fmaf(e, __uint_as_float(u[i] << 16), o[2 * i]);
            o[2 * i + 1] = fmaf(e, __uint_as_float(u[i] & 0xffff0000u), o[2 * i + 1]);
        }
    }
    // over the key groups of a wave (lanes with the same c), then over the waves
    sum = stride_allreduce<LPK>(sum);
#pragma unroll
    for (int i = 0; i < 8; i++) o[i] = stride_allreduce<LPK>(o[i]);
    float *ro = red + 16;   // [4][HD], then the sums
    if (lane < LPK) {
#pragma unroll
        for (int i = 0; i < 8; i++) ro[w * HD + 8 * lane + i] = o[i];
        if (lane == 0) red[4 + w] = sum;
    }
    __syncthreads();
    if (tid < HD) a.part_o[(size_t)slice * a.d + h * HD + tid] = (ro[tid] + ro[HD + tid]) + (ro[2 * HD + tid] + ro[3 * HD + tid]);
    if (tid == 0) {
        float *ml = a.part_ml + ((size_t)slice * a.nh + h) * 2;
        ml[0] = mx;
        ml[1] = (red[4] + red[5]) + (red[6] + red[7]);
    }
}

template <int HD>
__global__ __launch_bounds__(kDecThr) void decode_heads_kernel(DecArgs a) {
    __shared__ float red[16 + 4 * HD];
    const int h = blockIdx.x, part = blockIdx.y;
    if (part < a.slices) attention_slice<HD>(a, h, part, red);
    else level_head<HD>(a, part - a.slices, h, red);
}

// Eight rows of the output projection per workgroup; every workgroup forms the whole gated vector for itself.  The
// chain of loads is what takes the time, so nothing is loaded behind a value it does not need: the weights of the first
// 1024 columns, the slices' statistics (one thread each, then shared in LDS) and the levels and slices of a thread's first
// two columns are all requested at the top (10.0 -> 7.0 -> 4.9 us at d = 512, 5 slices, 4 levels).
__global__ __launch_bounds__(kDecThr) void decode_output_kernel(DecArgs a) {
    extern __shared__ float smem[];
    float *gated = smem, *wgt = smem + a.d;   // [d], [slices][heads]: a slice's weight in the merged softmax
    const int tid = threadIdx.x, lane = tid & 63, w = tid >> 6, d = a.d, n4 = d >> 2;
    const int r = blockIdx.x * 8 + 2 * w;
    const float4 *w0 = reinterpret_cast<const float4 *>(a.w_o + (size_t)r * d), *w1 = w0 + n4;
    constexpr int NW = 4;
    float4 p0[NW], p1[NW];
#pragma unroll
    for (int j = 0; j < NW; j++) {
        const int i = min(lane + 64 * j, n4 - 1);
        p0[j] = w0[i];
        p1[j] = w1[i];
    }
    constexpr int NL = 4, NS = 8;
    float ty[2][NL], to[2][NS];
#pragma unroll
    for (int c = 0; c < 2; c++) {
        const int i = min(tid + c * kDecThr, d - 1);
#pragma unroll
        for (int j = 0; j < NL; j++) ty[c][j] = a.lv[min(j, a.levels - 1)].y[i];
#pragma unroll
        for (int j = 0; j < NS; j++) to[c][j] = a.part_o[(size_t)min(j, a.slices - 1) * d + i];
    }
    const float scale = a.levels > 2 ? 1.f / sqrtf((float)a.levels) : 1.f;
    const int stats = a.slices * a.nh;
    if (stats <= min(kDecThr, d)) {   // one of them a thread; their sums wait where gated will stand
        float2 ml = make_float2(0.f, 0.f);
        if (tid < stats) {
            ml = *reinterpret_cast<const float2 *>(a.part_ml + (size_t)tid * 2);
            wgt[tid] = ml.x;
            gated[tid] = ml.y;
        }
        __syncthreads();
        float weight = 0.f;
        if (tid < stats) {
            float mx = -FLT_MAX, sum = 0.f;
            for (int i = tid % a.nh; i < stats; i += a.nh) mx = fmaxf(mx, wgt[i]);
            for (int i = tid % a.nh; i < stats; i += a.nh) sum += expf(wgt[i] - mx) * gated[i];
            weight = expf(ml.x - mx) * (1.f / sum);
        }
        __syncthreads();
        if (tid < stats) wgt[tid] = weight;
    } else for (int h = tid; h < a.nh; h += kDecThr) {
        float mx = -FLT_MAX, sum = 0.f;
        for (int s = 0; s < a.slices; s++) mx = fmaxf(mx, a.part_ml[((size_t)s * a.nh + h) * 2]);
        for (int s = 0; s < a.slices; s++) {
            const float2 ml = *reinterpret_cast<const float2 *>(a.part_ml + ((size_t)s * a.nh + h) * 2);
            const float e = expf(ml.x - mx);
            sum += e * ml.y;
            wgt[s * a.nh + h] = e;
        }
        const float inv = 1.f / sum;
        for (int s = 0; s < a.slices; s++) wgt[s * a.nh + h] *= inv;
    }
    __syncthreads();
    auto column = [&](int i, const float(&t0)[NL], const float(&o0)[NS]) {
        const int h = i >> a.hd_log2;
        float o = 0.f, y = 0.f;
        for (int l = 0; l < a.levels; l += NL) {
            float t[NL];
#pragma unroll
            for (int j = 0; j < NL; j++) t[j] = l + j < a.levels ? l ? a.lv[l + j].y[i] : t0[j] : 0.f;
            y += (t[0] + t[1]) + (t[2] + t[3]);
        }
        for (int s = 0; s < a.slices; s += NS) {
            float t[NS];
#pragma unroll
            for (int j = 0; j < NS; j++) t[j] = s ? a.part_o[(size_t)min(s + j, a.slices - 1) * d + i] : o0[j];
#pragma unroll
            for (int j = 0; j < NS; j++) o += s + j < a.slices ? wgt[(s + j) * a.nh + h] * t[j] : 0.f;
        }
        const uint16_t o16 = f32_to_bf16_rne(o);
        y *= scale;
        const float g = 1.f / (1.f + expf(-y)), at = bf2f(o16);
        gated[i] = at * g;
        if (blockIdx.x == 0) {
            a.attn_bf16[i] = o16;
            a.attn_out[i] = at;
            a.y_combined[i] = y;
            a.gate[i] = g;
            a.gated[i] = at * g;
        }
    };
#pragma unroll
    for (int c = 0; c < 2; c++)
        if (tid + c * kDecThr < d) column(tid + c * kDecThr, ty[c], to[c]);
    for (int i = tid + 2 * kDecThr; i < d; i += kDecThr) {
        float t[NL], o[NS];
#pragma unroll
        for (int j = 0; j < NL; j++) t[j] = a.lv[min(j, a.levels - 1)].y[i];
#pragma unroll
        for (int j = 0; j < NS; j++) o[j] = a.part_o[(size_t)min(j, a.slices - 1) * d + i];
        column(i, t, o);
    }
    __syncthreads();
    float acc0 = 0.f, acc1 = 0.f;
#pragma unroll
    for (int j = 0; j < NW; j++) {
        const int i = lane + 64 * j;
        if (i < n4) {
            const float4 g = reinterpret_cast<const float4 *>(gated)[i];
            acc0 += dot4(p0[j], g);
            acc1 += dot4(p1[j], g);
        }
    }
    for (int i = lane + 64 * NW; i < n4; i += 64) {
        const float4 g = reinterpret_cast<const float4 *>(gated)[i];
        acc0 += dot4(w0[i], g);
        acc1 += dot4(w1[i], g);
    }
    acc0 = wave_allreduce(acc0);
    acc1 = wave_allreduce(acc1);
    if (lane < 2) a.projected[r + lane] = lane ? acc1 : acc0;
}

// 64 columns of the unembedding per workgroup of eight waves: 16 lanes x 4 columns wide (256 consecutive bytes of a
// row), 32 groups of lanes over the rows, so that a vocabulary of a few thousand still fills the chip and every
// thread has its d / 32 loads in flight.
constexpr int kLogThr = 512;
template <int VEC>
__global__ __launch_bounds__(kLogThr) void decode_logits_kernel(const float *__restrict__ x, const float *__restrict__ w,
                                                                float *__restrict__ out, float *__restrict__ host, int d, int v) {
    constexpr int NB = 8;   // rows per group of lanes in flight
    __shared__ float xs[4096 + 32 * NB], part[8][16 * VEC];
    const int tid = threadIdx.x, lane = tid & 63, wv = tid >> 6, c = lane & 15, g = tid >> 4;
    const int col = min((blockIdx.x * 16 + c) * VEC, v - VEC);   // columns past the end repeat the last ones, unused
    for (int i = tid; i < d + 32 * NB; i += kLogThr) xs[i] = i < d ? x[i] : 0.f;
    __syncthreads();
    float acc[VEC];
#pragma unroll
    for (int i = 0; i < VEC; i++) acc[i] = 0.f;
    for (int r = g; r < d; r += 32 * NB) {
        float y[NB][VEC];
#pragma unroll
        for (int j = 0; j < NB; j++) {   // rows past the end meet a zero of xs
            const float *p = w + (size_t)min(r + 32 * j, d - 1) * v + col;
            if constexpr (VEC == 4) {
                const float4 q = *reinterpret_cast<const float4 *>(p);
                y[j][0] = q.x; y[j][1] = q.y; y[j][2] = q.z; y[j][3] = q.w;
            } else y[j][0] = *p;
        }
#pragma unroll
        for (int j = 0; j < NB; j++)
#pragma unroll
            for (int i = 0; i < VEC; i++) acc[i] = fmaf(xs[r + 32 * j], y[j][i], acc[i]);
    }
#pragma unroll
    for (int i = 0; i < VEC; i++) {
        acc[i] = xor_add<16>(acc[i]);
        acc[i] = xor_add<32>(acc[i]);
        if (lane < 16) part[wv][c * VEC + i] = acc[i];
    }
    __syncthreads();
    const int o = blockIdx.x * 16 * VEC + tid;
    if (tid < 16 * VEC && o < v) {
        float y = 0.f;
#pragma unroll
        for (int i = 0; i < 8; i++) y += part[i][tid];
        out[o] = y;
        host[o] = y;
    }
}

}  // namespace
}  // namespace nlh

extern "C" {

int decode_work_floats_rocm(int d, int heads, int levels, int window, int n_persistent) {
    const long long slices = nlh::ceil_div((long long)window + n_persistent, nlh::kSliceKeys);
    return (int)(4LL * levels * d + slices * d + slices * heads * 2 + d);
}

int decode_token_rocm(const float *embedding_row, const float *w_q, const float *w_k, const float *w_v, const float *w_o,
                      const float *w_unembed, const void *const *level_ptrs, const int *level_rule, const float *level_bounds,
                      int levels, int d, int heads, int vocab, int window, int n_persistent, int pos, uint16_t *k_cache,
                      uint16_t *v_cache, float *work, void *const *workspace, float *logits, float *logits_host) {
    using namespace nlh;
    const char *fn = "decode_token_rocm";
    const ErrorScope es;
    const int hd = heads > 0 ? d / heads : 0;
    if (levels < 1 || levels > kMaxLevels || heads < 1 || hd * heads != d || (hd != 32 && hd != 64 && hd != 128) || d > 4096 ||
        vocab < 1 || window < 1 || n_persistent < 0 || pos < 0) {
        fail("%s: levels=%d (1..8), d=%d (<= 4096), heads=%d (head size 32, 64 or 128), vocab=%d, window=%d, n_persistent=%d, pos=%d.",
             fn, levels, d, heads, vocab, window, n_persistent, pos);
        return 1;
    }
    DecArgs a;
    a.x = embedding_row;
    a.w_o = w_o;
    a.k_cache = k_cache; a.v_cache = v_cache;
    a.embedded = (float *)workspace[0];
    a.q_bf16 = (uint16_t *)workspace[1];
    a.attn_bf16 = (uint16_t *)workspace[2];
    a.attn_out = (float *)workspace[3];
    a.y_combined = (float *)workspace[4];
    a.gate = (float *)workspace[5];
    a.gated = (float *)workspace[6];
    a.d = d; a.nh = heads; a.hd_log2 = hd == 32 ? 5 : hd == 64 ? 6 : 7; a.levels = levels; a.pos = pos; a.window = window; a.n_persistent = n_persistent;
    const int n_pre = pos + 1 < n_persistent ? pos + 1 : n_persistent;
    const int ls = pos + 1 - window > n_persistent ? pos + 1 - window : n_persistent;
    const int n_keys = n_pre + (pos + 1 > ls ? pos + 1 - ls : 0);
    a.slices = ceil_div(n_keys, kSliceKeys);
    if ((size_t)(d + a.slices * heads) * sizeof(float) > 64 * 1024) {
        fail("%s: %d visible keys of %d heads exceed the merge's LDS.", fn, n_keys, heads);
        return 1;
    }
    float *p = work;
    int segs = 0;
    a.seg_w[segs] = w_q; a.seg_out[segs++] = a.q_bf16;
    a.seg_w[segs] = w_k; a.seg_out[segs++] = k_cache + (size_t)pos * d;
    a.seg_w[segs] = w_v; a.seg_out[segs++] = v_cache + (size_t)pos * d;
    for (int l = 0; l < levels; l++) {
        const void *const *lp = level_ptrs + 8 * l;
        const float *b = level_bounds + 6 * l;
        DecLevel &lv = a.lv[l];
        lv.w_alpha = (const float *)lp[3]; lv.b_alpha = (const float *)lp[4];
        lv.w_theta = (const float *)lp[5]; lv.b_theta = (const float *)lp[6];
        lv.memory = (float *)const_cast<void *>(lp[7]);
        lv.k = p; lv.v = p + d; lv.q = p + 2 * d; lv.y = p + 3 * d;
        p += 4 * d;
        lv.alpha_floor = b[0]; lv.alpha_ceil = b[1]; lv.theta_floor = b[2]; lv.theta_ceil = b[3]; lv.clip = b[4]; lv.m_norm = b[5];
        lv.rule = level_rule[l];
        if (!reads_only(lv.rule)) {
            a.seg_w[segs] = (const float *)lp[0]; a.seg_out[segs++] = lv.k;
            a.seg_w[segs] = (const float *)lp[1]; a.seg_out[segs++] = lv.v;
        }
        a.seg_w[segs] = (const float *)lp[2]; a.seg_out[segs++] = lv.q;
    }
    a.part_o = p; p += (size_t)a.slices * d;
    a.part_ml = p; p += (size_t)a.slices * heads * 2;
    a.projected = p;
    const hipStream_t st = stream();
    {
        KernelTimer kt("decode_project_kernel");
        hipLaunchKernelGGL(decode_project_kernel, dim3(d / 16, segs), dim3(kDecThr), 0, st, a);
        check_launch("decode_project_kernel");
    }
    {
        KernelTimer kt("decode_heads_kernel");
        const dim3 grid(heads, a.slices + levels);
        if (hd == 32) hipLaunchKernelGGL(decode_heads_kernel<32>, grid, dim3(kDecThr), 0, st, a);
        else if (hd == 64) hipLaunchKernelGGL(decode_heads_kernel<64>, grid, dim3(kDecThr), 0, st, a);
        else hipLaunchKernelGGL(decode_heads_kernel<128>, grid, dim3(kDecThr), 0, st, a);
        check_launch("decode_heads_kernel");
    }
    {
        KernelTimer kt("decode_output_kernel");
        hipLaunchKernelGGL(decode_output_kernel, dim3(d / 8), dim3(kDecThr), (size_t)(d + a.slices * heads) * sizeof(float),
                           st, a);
        check_launch("decode_output_kernel");
    }
    {
        KernelTimer kt("decode_logits_kernel");
        if (vocab % 4 == 0 && ((uintptr_t)w_unembed & 15) == 0)
            hipLaunchKernelGGL(decode_logits_kernel<4>, dim3(ceil_div(vocab, 64)), dim3(kLogThr), 0, st, a.projected, w_unembed,
                               logits, logits_host, d, vocab);
        else
            hipLaunchKernelGGL(decode_logits_kernel<1>, dim3(ceil_div(vocab, 16)), dim3(kLogThr), 0, st, a.projected, w_unembed,
                               logits, logits_host, d, vocab);
        check_launch("decode_logits_kernel");
    }
    if (es.failed()) return 2;
    check_hip(hipStreamSynchronize(st), fn);   // the logits are on the host when the call returns, as the caller expects
    return es.failed() ? 3 : 0;
}

}  // extern "C"
