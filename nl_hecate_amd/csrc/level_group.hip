// The glue either side of the memory rules for a group of levels that run the same rule on the same tokens
// (gpu_memory_forward / gpu_memory_backward, core/src/gpu_forward.rs:1197-1540, core/src/gpu_backward.rs:459-1200,
// 2047-2117): one launch per step for all levels instead of eleven per level forward and fifteen backward.  Each pass
// reads and writes every [tokens, d] tensor once; one wave per token where a row is reduced.
#include <float.h>
#include <hip/hip_runtime.h>
#include <stdint.h>

#include "../../include/nl_hecate_ffi.h"
#include "rule_common.h"
#include "runtime.h"

namespace nlh {
namespace {

constexpr int kMaxLevels = 8, kThr = 256;

struct InLevel {
    float *k, *v, *q;            // [n, d] projections; k and q leave normalised
    const float *wa, *ba, *wt, *bt, *we, *be;
    float *k_norms, *q_norms, *alpha, *theta, *eta;
    float a_lo, a_hi, t_lo, t_hi;
};
struct InArgs {
    InLevel lv[kMaxLevels];
    float *kh, *vh, *qh, *ah, *th, *eh;   // [levels * bs * nh, s, hd], [levels * bs * nh, s]
    int bs, s, nh, hd;
    float eps;
};

__device__ __forceinline__ float sigmoidf_(float x) { return 1.f / (1.f + expf(-x)); }
__device__ __forceinline__ float softplusf_(float x) { return x > 20.f ? x : logf(1.f + expf(x)); }
__device__ __forceinline__ float dot4f(const float4 &a, const float4 &b) { return a.x * b.x + a.y * b.y + a.z * b.z + a.w * b.w; }
__device__ __forceinline__ float4 ld4(const float *p, int i4) { return reinterpret_cast<const float4 *>(p)[i4]; }
__device__ __forceinline__ void st4(float *p, int i4, const float4 &x) { reinterpret_cast<float4 *>(p)[i4] = x; }

// Row norms, gates (clamped where a bound is set), head split of k, v, q and the per-head copies of the gates.  The gate products take the raw
// k and are divided by its norm afterwards, so one sweep over a token's rows serves all eight sums.
template <int NP, bool HAS_Q, bool HAS_ETA>
__global__ __launch_bounds__(kThr) void level_inputs_kernel(InArgs a) {
    const InLevel &lv = a.lv[blockIdx.y];
    const int lane = threadIdx.x & 63, d = a.nh * a.hd, d4 = d >> 2, hd4 = a.hd >> 2, n = a.bs * a.s;
    const size_t chain0 = (size_t)blockIdx.y * a.bs * a.nh;
    const float ba = lv.ba[0], bt = lv.bt[0], be = HAS_ETA ? lv.be[0] : 0.f;
    for (int tok = (blockIdx.x * kThr + threadIdx.x) >> 6; tok < n; tok += gridDim.x * (kThr / 64)) {
        float *kr = lv.k + (size_t)tok * d, *qr = HAS_Q ? lv.q + (size_t)tok * d : nullptr;
        const float *vr = lv.v + (size_t)tok * d;
        float4 k[NP], v[NP], q[HAS_Q ? NP : 1];
        float s[8] = {0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f};
#pragma unroll
        for (int j = 0; j < NP; j++) {
            const int i = lane + 64 * j;
            const bool in = i < d4;
            k[j] = in ? ld4(kr, i) : f4_zero();
            v[j] = in ? ld4(vr, i) : f4_zero();
            if (HAS_Q) q[j] = in ? ld4(qr, i) : f4_zero();
        }
#pragma unroll
        for (int j = 0; j < NP; j++) {
            const int i = min(lane + 64 * j, d4 - 1);   // past the end the rows are zero
            s[0] += dot4f(k[j], k[j]);
            if (HAS_Q) s[1] += dot4f(q[j], q[j]);
            s[2] += dot4f(k[j], ld4(lv.wa, i));
            s[3] += dot4f(v[j], ld4(lv.wa + d, i));
            s[4] += dot4f(k[j], ld4(lv.wt, i));
            s[5] += dot4f(v[j], ld4(lv.wt + d, i));
            if (HAS_ETA) { s[6] += dot4f(k[j], ld4(lv.we, i)); s[7] += dot4f(v[j], ld4(lv.we + d, i)); }
        }
#pragma unroll
        for (int i = 0; i < 8; i++) s[i] = wave_allreduce(s[i]);
        const float kn = sqrtf(s[0]), qn = sqrtf(s[1]), ki = 1.f / fmaxf(kn, a.eps), qi = 1.f / fmaxf(qn, a.eps);
        const float al = clamp_gate(sigmoidf_(s[2] * ki + s[3] + ba), lv.a_lo, lv.a_hi, 1.f);
        const float th = clamp_gate(softplusf_(s[4] * ki + s[5] + bt), lv.t_lo, lv.t_hi, FLT_MAX);
        const float et = HAS_ETA ? sigmoidf_(s[6] * ki + s[7] + be) : 0.f;
        const int b = tok / a.s, t = tok - b * a.s;
        const size_t c0 = chain0 + (size_t)b * a.nh;
#pragma unroll
        for (int j = 0; j < NP; j++) {
            const int i = lane + 64 * j;
            if (i >= d4) continue;
            const int h = i / hd4;
            const size_t o = ((c0 + h) * a.s + t) * hd4 + (i - h * hd4);
            const float4 kk = f4_scale(ki, k[j]);
            st4(kr, i, kk);
            reinterpret_cast<float4 *>(a.kh)[o] = kk;
            reinterpret_cast<float4 *>(a.vh)[o] = v[j];
            if (HAS_Q) {
                const float4 qq = f4_scale(qi, q[j]);
                st4(qr, i, qq);
                reinterpret_cast<float4 *>(a.qh)[o] = qq;
            }
        }
        if (lane == 0) {
            lv.k_norms[tok] = kn;
            if (HAS_Q) lv.q_norms[tok] = qn;
            lv.alpha[tok] = al;
            lv.theta[tok] = th;
            if (HAS_ETA) lv.eta[tok] = et;
        }
        for (int h = lane; h < a.nh; h += 64) {
            const size_t o = (c0 + h) * a.s + t;
            a.ah[o] = al;
            a.th[o] = th;
            if (HAS_ETA) a.eh[o] = et;
        }
    }
}

struct OutLevel {
    const float *k, *q, *k_norms, *q_norms, *alpha, *theta, *eta;
    float *dk, *dv, *dq;   // [n, d] gradients of the raw projections
    float a_lo, a_hi, t_lo, t_hi;
    int clamp_a, clamp_t;
};
struct OutArgs {
    OutLevel lv[kMaxLevels];
    const float *dkh, *dvh, *dqh, *dah, *dth, *deh;
    float *pre;            // [levels][3][n]: gradients of the gates' pre-activations
    int bs, s, nh, hd;
    float eps;
};

// Head merge of d_k, d_v, d_q with the backward of the two row normalisations, head sums of the gate gradients with the
// straight-through clamp masks and the activations' derivatives (from the cached outputs).
template <int NP, bool HAS_ETA>
__global__ __launch_bounds__(kThr) void level_grads_kernel(OutArgs a) {
    const OutLevel &lv = a.lv[blockIdx.y];
    const int lane = threadIdx.x & 63, d = a.nh * a.hd, d4 = d >> 2, hd4 = a.hd >> 2, n = a.bs * a.s;
    const size_t chain0 = (size_t)blockIdx.y * a.bs * a.nh;
    float *pre = a.pre + (size_t)blockIdx.y * 3 * n;
    for (int tok = (blockIdx.x * kThr + threadIdx.x) >> 6; tok < n; tok += gridDim.x * (kThr / 64)) {
        const int b = tok / a.s, t = tok - b * a.s;
        const size_t c0 = chain0 + (size_t)b * a.nh;
        float4 gk[NP], gq[NP], gv[NP], xk[NP], xq[NP];
#pragma unroll
        for (int j = 0; j < NP; j++) {
            const int i = lane + 64 * j, h = min(i, d4 - 1) / hd4;
            const size_t o = ((c0 + h) * a.s + t) * hd4 + (min(i, d4 - 1) - h * hd4);
            const bool in = i < d4;
            gk[j] = in ? reinterpret_cast<const float4 *>(a.dkh)[o] : f4_zero();
            gq[j] = in ? reinterpret_cast<const float4 *>(a.dqh)[o] : f4_zero();
            gv[j] = in ? reinterpret_cast<const float4 *>(a.dvh)[o] : f4_zero();
            xk[j] = in ? ld4(lv.k + (size_t)tok * d, i) : f4_zero();
            xq[j] = in ? ld4(lv.q + (size_t)tok * d, i) : f4_zero();
        }
        float ga = 0.f, gt = 0.f, ge = 0.f;
        for (int h = lane; h < a.nh; h += 64) {
            const size_t o = (c0 + h) * a.s + t;
            ga += a.dah[o];
            gt += a.dth[o];
            if (HAS_ETA) ge += a.deh[o];
        }
        float sk = 0.f, sq = 0.f;
#pragma unroll
        for (int j = 0; j < NP; j++) { sk += dot4f(gk[j], xk[j]); sq += dot4f(gq[j], xq[j]); }
        sk = wave_allreduce(sk); sq = wave_allreduce(sq);
        ga = wave_allreduce(ga); gt = wave_allreduce(gt);
        if (HAS_ETA) ge = wave_allreduce(ge);
        const float kn = lv.k_norms[tok], qn = lv.q_norms[tok];
        // below the norm floor the row was divided by it: no projection term
        const float ki = kn >= a.eps ? 1.f / kn : 1.f / a.eps, qi = qn >= a.eps ? 1.f / qn : 1.f / a.eps;
        sk = kn >= a.eps ? sk : 0.f;
        sq = qn >= a.eps ? sq : 0.f;
#pragma unroll
        for (int j = 0; j < NP; j++) {
            const int i = lane + 64 * j;
            if (i >= d4) continue;
            st4(lv.dk + (size_t)tok * d, i, f4_axpby(ki, gk[j], -ki * sk, xk[j]));
            st4(lv.dq + (size_t)tok * d, i, f4_axpby(qi, gq[j], -qi * sq, xq[j]));
            st4(lv.dv + (size_t)tok * d, i, gv[j]);
        }
        if (lane == 0) {
            const float al = lv.alpha[tok], th = lv.theta[tok];
            if (lv.clamp_a && (al <= lv.a_lo || al >= lv.a_hi)) ga = 0.f;
            if (lv.clamp_t && (th <= lv.t_lo || th >= lv.t_hi)) gt = 0.f;
            pre[tok] = ga * al * (1.f - al);
            pre[n + tok] = gt * (1.f - expf(-th));
            if (HAS_ETA) { const float et = lv.eta[tok]; pre[2 * n + tok] = ge * et * (1.f - et); }
        }
    }
}

// Gate weights: d_w = sum_t pre_t [k_t | v_t], d_b = sum_t pre_t.  Stage 1: 64 tokens x 256 columns per workgroup; stage 2
// adds the token blocks in a fixed order.
struct GateLevel { const float *k, *v; float *dw[3], *db[3]; };
struct GateArgs {
    GateLevel lv[kMaxLevels];
    const float *pre;
    float *part;   // [levels][blocks][3][2d + 1]
    int n, d, blocks, gates;
};
constexpr int kGateTok = 64;
__global__ __launch_bounds__(kThr) void level_gate_part_kernel(GateArgs a) {
    __shared__ float g[3][kGateTok];
    const GateLevel &lv = a.lv[blockIdx.z];
    const int t0 = blockIdx.x * kGateTok, tn = min(kGateTok, a.n - t0), d = a.d;
    const float *pre = a.pre + (size_t)blockIdx.z * 3 * a.n;
    for (int j = threadIdx.x; j < 3 * kGateTok; j += kThr) {
        const int w = j / kGateTok, t = j % kGateTok;
        g[w][t] = (w < a.gates && t < tn) ? pre[w * a.n + t0 + t] : 0.f;
    }
    __syncthreads();
    const int c = blockIdx.y * kThr + threadIdx.x, ld = 2 * d + 1;
    float *out = a.part + ((size_t)blockIdx.z * a.blocks + blockIdx.x) * 3 * ld;
    if (c < 2 * d) {
        const float *x = (c < d ? lv.k + c : lv.v + (c - d)) + (size_t)t0 * d;
        float s0 = 0.f, s1 = 0.f, s2 = 0.f;
#pragma unroll 8
        for (int t = 0; t < tn; t++) {
            const float y = x[(size_t)t * d];
            s0 += g[0][t] * y;
            s1 += g[1][t] * y;
            s2 += g[2][t] * y;
        }
        out[c] = s0;
        out[ld + c] = s1;
        out[2 * ld + c] = s2;
    }
    if (blockIdx.y == 0 && threadIdx.x < 3) {
        float s = 0.f;
        for (int t = 0; t < tn; t++) s += g[threadIdx.x][t];
        out[threadIdx.x * ld + 2 * d] = s;
    }
}
__global__ __launch_bounds__(kThr) void level_gate_sum_kernel(GateArgs a) {
    const int c = blockIdx.x * kThr + threadIdx.x, w = blockIdx.y, ld = 2 * a.d + 1;
    if (c >= ld) return;
    const float *p = a.part + ((size_t)blockIdx.z * a.blocks * 3 + w) * ld + c;
    float s = 0.f;
#pragma unroll 4
    for (int b = 0; b < a.blocks; b++) s += p[(size_t)b * 3 * ld];
    const GateLevel &lv = a.lv[blockIdx.z];
    if (c < 2 * a.d) lv.dw[w][c] = s;
    else lv.db[w][0] = s;
}

// Carried memories of a group of levels: gathered as the initial states of one batch of chains, and written back from
// the states at the end with the reference's clamp of the carried state (m_norm_clamp_batch, elementwise.cu:251).
struct StateArgs { float *ctx[kMaxLevels]; float bound[kMaxLevels]; };
__global__ __launch_bounds__(kThr) void level_states_gather_kernel(StateArgs a, float *__restrict__ dst, int n4) {
    const float4 *src = reinterpret_cast<const float4 *>(a.ctx[blockIdx.y]);
    for (int i = blockIdx.x * kThr + threadIdx.x; i < n4; i += gridDim.x * kThr)
        reinterpret_cast<float4 *>(dst)[(size_t)blockIdx.y * n4 + i] = src[i];
}
__global__ __launch_bounds__(kThr) void level_states_final_kernel(StateArgs a, const float *__restrict__ states, long long stride,
                                                                  int chains, int dd) {
    __shared__ float red[kThr / 64];
    const int lv = blockIdx.x / chains, c = blockIdx.x % chains;
    const float4 *src = reinterpret_cast<const float4 *>(states + (size_t)blockIdx.x * stride);
    float4 *dst = reinterpret_cast<float4 *>(a.ctx[lv] + (size_t)c * dd);
    const float bound = a.bound[lv];
    float scale = 1.f;
    if (mnorm_active(bound)) {
        float s = 0.f;
        for (int i = threadIdx.x; i < dd / 4; i += kThr) s += dot4f(src[i], src[i]);
        s = wave_allreduce(s);
        if ((threadIdx.x & 63) == 0) red[threadIdx.x >> 6] = s;
        __syncthreads();
        const float norm = sqrtf((red[0] + red[1]) + (red[2] + red[3]));
        if (norm > bound) scale = bound / norm;
    }
    for (int i = threadIdx.x; i < dd / 4; i += kThr) dst[i] = f4_scale(scale, src[i]);
}

// One token-major gradient as the head-major gradient of every level.
__global__ __launch_bounds__(kThr) void level_heads_repeat_kernel(const float4 *__restrict__ x, float4 *__restrict__ out, int bs, int s,
                                                                  int nh, int hd4, int levels) {
    const size_t n4 = (size_t)bs * s * nh * hd4;
    for (size_t o = (size_t)blockIdx.x * kThr + threadIdx.x; o < n4; o += (size_t)gridDim.x * kThr) {
        const int c = o % hd4;
        size_t r = o / hd4;
        const int t = r % s;
        r /= s;
        const int h = r % nh, b = r / nh;
        const float4 y = x[(((size_t)b * s + t) * nh + h) * hd4 + c];
        for (int l = 0; l < levels; l++) out[(size_t)l * n4 + o] = y;
    }
}

constexpr int kMaxSaxpy = 64, kSaxpyPer = 4096;   // elements per workgroup
struct SaxpyArgs { const float *x[kMaxSaxpy]; float *y[kMaxSaxpy]; int n[kMaxSaxpy], first[kMaxSaxpy + 1]; int count; float alpha; };
__global__ __launch_bounds__(kThr) void saxpy_multi_kernel(SaxpyArgs a) {
    const int t = batch_entry(a.first, a.count, blockIdx.x);
    const float *x = a.x[t];
    float *y = a.y[t];
    const int i0 = ((int)blockIdx.x - a.first[t]) * kSaxpyPer, i1 = min(a.n[t], i0 + kSaxpyPer);
    if ((((uintptr_t)x | (uintptr_t)y) & 15) == 0) {
        for (int i = i0 + 4 * (int)threadIdx.x; i + 3 < i1; i += 4 * kThr) {
            float4 p = *reinterpret_cast<float4 *>(y + i);
            f4_fma(p, a.alpha, *reinterpret_cast<const float4 *>(x + i));
            *reinterpret_cast<float4 *>(y + i) = p;
        }
        for (int i = i0 + ((i1 - i0) & ~3) + threadIdx.x; i < i1; i += kThr) y[i] += a.alpha * x[i];
    } else {
        for (int i = i0 + threadIdx.x; i < i1; i += kThr) y[i] += a.alpha * x[i];
    }
}

bool check_group(const char *fn, int levels, int bs, int s, int nh, int hd) {
    if (levels < 1 || levels > kMaxLevels || bs < 1 || s < 1 || nh < 1 || hd < 4 || hd % 4 || nh * hd > 1024) {
        fail("%s: levels=%d (1..%d), bs=%d, s=%d, heads=%d x %d (head size a multiple of 4, width at most 1024).", fn, levels,
             kMaxLevels, bs, s, nh, hd);
        return false;
    }
    return true;
}
int token_blocks(long long n) { const long long b = (n + kThr / 64 - 1) / (kThr / 64); return (int)(b > 1024 ? 1024 : b); }

}  // namespace
}  // namespace nlh

using namespace nlh;

extern "C" {

void level_group_inputs_f32_rocm(const void *const *ptrs, const float *bounds, int levels, float *k_heads, float *v_heads,
                                 float *q_heads, float *alpha_heads, float *theta_heads, float *eta_heads, int bs, int s, int nh,
                                 int hd, float eps) {
    if (!check_group("level_group_inputs_f32_rocm", levels, bs, s, nh, hd)) return;
    InArgs a;
    for (int l = 0; l < levels; l++) {
        float *const *p = (float *const *)(ptrs + 14 * l);
        a.lv[l] = InLevel{p[0], p[1], p[2], p[3], p[4], p[5], p[6], p[7], p[8], p[9], p[10], p[11], p[12], p[13],
                          bounds[4 * l], bounds[4 * l + 1], bounds[4 * l + 2], bounds[4 * l + 3]};
    }
    a.kh = k_heads; a.vh = v_heads; a.qh = q_heads; a.ah = alpha_heads; a.th = theta_heads; a.eh = eta_heads;
    a.bs = bs; a.s = s; a.nh = nh; a.hd = hd; a.eps = eps;
    const dim3 grid(token_blocks((long long)bs * s), levels);
    const bool wide = nh * hd > 512, q = q_heads != nullptr, eta = eta_heads != nullptr;
    KernelTimer kt("level_inputs_kernel");
#define NLH_IN(NP)                                                                                             \
    do {                                                                                                       \
        if (q && eta) hipLaunchKernelGGL((level_inputs_kernel<NP, true, true>), grid, dim3(kThr), 0, stream(), a);        \
        else if (q) hipLaunchKernelGGL((level_inputs_kernel<NP, true, false>), grid, dim3(kThr), 0, stream(), a);         \
        else if (eta) hipLaunchKernelGGL((level_inputs_kernel<NP, false, true>), grid, dim3(kThr), 0, stream(), a);       \
        else hipLaunchKernelGGL((level_inputs_kernel<NP, false, false>), grid, dim3(kThr), 0, stream(), a);               \
    } while (0)
    if (wide) NLH_IN(4);
    else NLH_IN(2);
#undef NLH_IN
    check_launch("level_inputs_kernel");
}

void level_group_grads_f32_rocm(const void *const *ptrs, const float *bounds, int levels, const float *d_k_heads,
                                const float *d_v_heads, const float *d_q_heads, const float *d_alpha_heads,
                                const float *d_theta_heads, const float *d_eta_heads, int bs, int s, int nh, int hd, float eps) {
    const ErrorScope es;
    if (!check_group("level_group_grads_f32_rocm", levels, bs, s, nh, hd)) return;
    const int n = bs * s, d = nh * hd, blocks = ceil_div(n, kGateTok);
    float *pre = scratch(38, (size_t)levels * 3 * n * sizeof(float));
    float *part = scratch(39, (size_t)levels * blocks * 3 * (2 * d + 1) * sizeof(float));
    if (es.failed()) return;
    OutArgs a;
    GateArgs g;
    for (int l = 0; l < levels; l++) {
        float *const *p = (float *const *)(ptrs + 17 * l);
        const float *b = bounds + 4 * l;
        a.lv[l] = OutLevel{p[0], p[2], p[3], p[4], p[5], p[6], p[7], p[8], p[9], p[10], b[0], b[1], b[2], b[3],
                           b[0] > 0.f || b[1] < 1.f, b[2] > 0.f || b[3] < FLT_MAX};
        g.lv[l] = GateLevel{p[0], p[1], {p[11], p[13], p[15]}, {p[12], p[14], p[16]}};
    }
    a.dkh = d_k_heads; a.dvh = d_v_heads; a.dqh = d_q_heads; a.dah = d_alpha_heads; a.dth = d_theta_heads; a.deh = d_eta_heads;
    a.pre = pre; a.bs = bs; a.s = s; a.nh = nh; a.hd = hd; a.eps = eps;
    const dim3 grid(token_blocks(n), levels);
    {
        KernelTimer kt("level_grads_kernel");
        const bool wide = d > 512, eta = d_eta_heads != nullptr;
        if (wide && eta) hipLaunchKernelGGL((level_grads_kernel<4, true>), grid, dim3(kThr), 0, stream(), a);
        else if (wide) hipLaunchKernelGGL((level_grads_kernel<4, false>), grid, dim3(kThr), 0, stream(), a);
        else if (eta) hipLaunchKernelGGL((level_grads_kernel<2, true>), grid, dim3(kThr), 0, stream(), a);
        else hipLaunchKernelGGL((level_grads_kernel<2, false>), grid, dim3(kThr), 0, stream(), a);
        check_launch("level_grads_kernel");
    }
    g.pre = pre; g.part = part; g.n = n; g.d = d; g.blocks = blocks; g.gates = d_eta_heads ? 3 : 2;
    KernelTimer kt("level_gate_kernels");
    hipLaunchKernelGGL(level_gate_part_kernel, dim3(blocks, ceil_div(2 * d, kThr), levels), dim3(kThr), 0, stream(), g);
    check_launch("level_gate_part_kernel");
    hipLaunchKernelGGL(level_gate_sum_kernel, dim3(ceil_div(2 * d + 1, kThr), g.gates, levels), dim3(kThr), 0, stream(), g);
    check_launch("level_gate_sum_kernel");
}

void level_group_states_gather_rocm(const float *const *contexts, int levels, float *initial, int chains, int dd) {
    if (levels < 1 || levels > kMaxLevels || chains < 1 || dd < 4 || dd % 4) {
        fail("level_group_states_gather_rocm: levels=%d chains=%d dd=%d.", levels, chains, dd);
        return;
    }
    StateArgs a;
    for (int l = 0; l < levels; l++) a.ctx[l] = const_cast<float *>(contexts[l]);
    const int n4 = chains * dd / 4, blocks = ceil_div(n4, kThr);
    hipLaunchKernelGGL(level_states_gather_kernel, dim3(blocks > 512 ? 512 : blocks, levels), dim3(kThr), 0, stream(), a, initial, n4);
    check_launch("level_states_gather_kernel");
}

void level_group_states_final_rocm(const float *states, long long stride, float *const *contexts, const float *m_norm_max,
                                   int levels, int chains, int dd) {
    if (levels < 1 || levels > kMaxLevels || chains < 1 || dd < 4 || dd % 4 || stride % 4) {
        fail("level_group_states_final_rocm: levels=%d chains=%d dd=%d stride=%lld.", levels, chains, dd, stride);
        return;
    }
    StateArgs a;
    for (int l = 0; l < levels; l++) { a.ctx[l] = contexts[l]; a.bound[l] = m_norm_max[l]; }
    hipLaunchKernelGGL(level_states_final_kernel, dim3(levels * chains), dim3(kThr), 0, stream(), a, states, stride, chains, dd);
    check_launch("level_states_final_kernel");
}

void level_group_heads_repeat_rocm(const float *x, float *out, int bs, int s, int nh, int hd, int levels) {
    if (!check_group("level_group_heads_repeat_rocm", levels, bs, s, nh, hd)) return;
    const int blocks = ceil_div((long long)bs * s * nh * hd / 4, kThr);
    hipLaunchKernelGGL(level_heads_repeat_kernel, dim3(blocks > 2048 ? 2048 : blocks), dim3(kThr), 0, stream(),
                       reinterpret_cast<const float4 *>(x), reinterpret_cast<float4 *>(out), bs, s, nh, hd / 4, levels);
    check_launch("level_heads_repeat_kernel");
}

void saxpy_multi_rocm(float alpha, const float *const *x, float *const *y, const int *n, int count) {
    SaxpyArgs a;
    a.alpha = alpha;
    a.count = 0;
    int blocks = 0;
    auto flush = [&] {
        if (!blocks) return;
        a.first[a.count] = blocks;
        hipLaunchKernelGGL(saxpy_multi_kernel, dim3(blocks), dim3(kThr), 0, stream(), a);
        check_launch("saxpy_multi_kernel");
        a.count = blocks = 0;
    };
    auto meet = [](const float *p, int np, const float *q, int nq) { return p < q + nq && q < p + np; };
    for (int i = 0; i < count; i++) {
        if (n[i] <= 0) continue;
        // pairs in one launch run beside each other: one that writes or reads what another writes (levels that share their
        // parameters) comes after it
        bool apart = a.count == kMaxSaxpy;
        for (int j = 0; j < a.count && !apart; j++)
            apart = meet(y[i], n[i], a.y[j], a.n[j]) || meet(x[i], n[i], a.y[j], a.n[j]) || meet(y[i], n[i], a.x[j], a.n[j]);
        if (apart) flush();
        a.x[a.count] = x[i];
        a.y[a.count] = y[i];
        a.n[a.count] = n[i];
        a.first[a.count++] = blocks;
        blocks += ceil_div(n[i], kSaxpyPer);
    }
    flush();
}

}  // extern "C"
