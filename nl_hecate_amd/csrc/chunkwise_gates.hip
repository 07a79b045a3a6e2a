// Backward of the frozen-M0 chunkwise Titans / Delta rule: the gate gradients d_alpha, d_eta.
//
//   d_alpha_s = -<M_(s-1), A_s>,   d_eta_s = <S_(s-1), B_s>
// with A_s, B_s the adjoints of M_s, S_s inside the chunk (core/kernels/titans_chunkwise_backward.cu:
// 118-358 accumulates the same inner products token by token on full d x d matrices):
//   A_s = sum_(t >= s) r[s][t] dy_t q_t^T + r[s][L-1] dMo
//   B_s = sum_(t >= s) c[t][s] dy_t q_t^T + c[L-1][s] dMo + bb[s][L-1] dSo
// Every inner product of a state with a rank-1 term is a scalar that obeys the rule's own recurrence:
// with u_s(t) = <M_s, dy_t q_t^T>, v_s(t) = <S_s, dy_t q_t^T>,
//   v_s(t) = eta_s v_(s-1)(t) + xs[s][t],   u_s(t) = keep_s u_(s-1)(t) + v_s(t),   u_(-1) = p0[t], v_(-1) = ps[t]
// where xs[s][t] = -theta_s (dy_t . e_s)(q_t . k_s) and p0, ps come from the gradient pass; the same holds
// for <M_s, dMo>, <S_s, dMo>, <S_s, dSo> with -theta_s e_s^T dMo k_s and -theta_s e_s^T dSo k_s as the
// per-token terms.  The weights r, c, bb obey forward recurrences in t.  So a chunk costs two sweeps of
// 64 steps on ONE wave and no matrix product, no coefficient table and no division:
//   sweep 1 (lane = t): u, v for s = 0..63, parked in LDS as rows s + 1
//   sweep 2 (lane = s): the weighted sums over t >= s with the weights advanced step by step.
// Row s is only ever read at t >= s, so the rows are packed as a triangle: half the LDS of a square, which is what
// decides how many chunks a compute unit works on at once.  Row s holds t = s .. 63 and starts at (63 - s)(64 - s) / 2, behind
// the rows that follow it: what the lanes t < s store lies in the places of later rows, which overwrite it, and needs no mask; a wave's LDS stores
// take effect in the order of its instructions, which the sweep keeps.
// Sweep 1 writes a row at consecutive addresses; in sweep 2 lane s reads address t plus a triangular number less one and 63:
// the triangular numbers of 32 consecutive s fall on 32 different banks.
// The sweeps are bound by the vector instructions they issue, four fifths of them in their steps, so gates and the per-token
// terms of the chunk's end come from LDS, four tokens a load, no store is masked, and weights and sums start by one comparison a
// step; the next chunk's terms are requested meanwhile.  16384 chunks 94 -> 63 us (71 with a workgroup per four chunks), 8192
// with the sums of 128 chains 62 -> 42, 2048 17.6 -> 12.5, 64 10.1 -> 7.7; their terms alone take 30, 15 and 4 at HBM's rate.
// Tokens beyond a short chunk carry keep = 1, eta = 0 and zero terms in sweep 1; sweep 2 ends before them.
#include <hip/hip_runtime.h>
#include <stdint.h>

#include <algorithm>

#include "chunkwise_grads.h"
#include "lane_ops.h"
#include "runtime.h"

namespace nlh {
namespace {

constexpr int GW = 64;            // tokens per chunk tile
constexpr int GTRI = GW * (GW + 1) / 2 + GW;   // floats of one packed triangle, and what the last rows store in front of it
constexpr int kGateWaves = 4;     // chunks per workgroup, one wave each
// where token 0 of row r would be: token t = r comes first
__host__ __device__ constexpr int tri_row(int r) { return GW + (GW - 1 - r) * (GW - r) / 2 - r; }
// gates of a chunk and the per-token terms of <M_s, dMo> and <S_s, dSo>
template <class T>
struct GateRows {
    T keep[GW];
    float eta[GW], g1[GW], g2[GW];
};
template <class T>
struct alignas(16) Four { T x[4]; };
template <class T>
__device__ __forceinline__ Four<T> four_at(const T *p) { return *reinterpret_cast<const Four<T> *>(p); }
template <class T>
constexpr size_t gate_lds(bool has_s) { return kGateWaves * (sizeof(GateRows<T>) + (has_s ? 2 : 1) * GTRI * sizeof(float)); }

// The launch carries a second, unrelated piece of the same backward, spread over its workgroups from the last one on: the first stage of
// the sum over the batch of the gradient of the initial state (it depends on the adjoint scan only, is far too
// small for a launch of its own, and runs beside the sweeps): piece (e, y, z) adds `per` chains' matrices
// z (0: M, 1: S), elements 256 e .. 256 e + 255, into tmp[z][y]; a second launch adds the rows of tmp in a fixed order.
struct FirstSum {
    const float *src[2];   // [batch][chain_stride]: gradient of the initial M / S per chain
    float *tmp;            // [nsum][rows][d*d]
    size_t chain_stride;
    int batch, per, rows, nsum, elems;   // elems = d*d, a multiple of 256
};

// T: type of the running values and sums (the rows in between are kept in float either way).
template <bool HAS_S, class T>
__global__ __launch_bounds__(64 * kGateWaves, 2) void cw_gates_sweep_kernel(
    const float *__restrict__ alpha, const float *__restrict__ eta, const float *__restrict__ pvec,
    const float *__restrict__ xs, const float *__restrict__ scal, float *__restrict__ d_alpha,
    float *__restrict__ d_eta, int s, int C, int nc, int ntask, FirstSum fs) {
    extern __shared__ __align__(16) float smem[];
    const int lane = threadIdx.x & 63, wv = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int nb = fs.elems / 256;
    for (int bid = gridDim.x - 1 - blockIdx.x; bid < nb * fs.rows * fs.nsum; bid += gridDim.x) {
        const int eb = bid % nb, y = (bid / nb) % fs.rows, z = bid / (nb * fs.rows);
        const int e = eb * 256 + threadIdx.x, b0 = y * fs.per, b1 = min(fs.batch, b0 + fs.per);
        const float *st = fs.src[z] + e;
        float x = 0.f;
        for (int b = b0; b < b1; b += 8) {   // eight loads in flight
            float r[8];
#pragma unroll
            for (int i = 0; i < 8; i++) r[i] = b + i < b1 ? st[(size_t)(b + i) * fs.chain_stride] : 0.f;
#pragma unroll
            for (int i = 0; i < 8; i++) x += r[i];
        }
        fs.tmp[((size_t)z * fs.rows + y) * fs.elems + e] = x;
    }
    const int step_tasks = gridDim.x * kGateWaves;
    int task = blockIdx.x * kGateWaves + wv;
    if (task >= ntask) return;   // no barrier below: waves are independent
    GateRows<T> &gr = reinterpret_cast<GateRows<T> *>(smem)[wv];
    float *U = smem + kGateWaves * sizeof(GateRows<T>) / sizeof(float) + (size_t)wv * (HAS_S ? 2 : 1) * GTRI, *V = U + GTRI;
    struct Chunk {
        size_t tok;
        int L;
        float alpha, eta, m0dm, s0dm, s0ds;
        float4 pv;
    };
    auto chunk_of = [&](int tk) __attribute__((always_inline)) {
        const int chain = tk / nc, t0 = tk % nc * C;
        Chunk c;
        c.L = min(C, s - t0);
        c.tok = (size_t)chain * s + t0;
        const bool in = lane < c.L;
        c.alpha = in ? alpha[c.tok + lane] : 0.f;
        c.eta = (HAS_S && in) ? eta[c.tok + lane] : 0.f;
        c.pv = in ? *reinterpret_cast<const float4 *>(pvec + (c.tok + lane) * 4) : make_float4(0.f, 0.f, 0.f, 0.f);
        c.m0dm = scal[(size_t)tk * 4 + 0];
        c.s0dm = scal[(size_t)tk * 4 + 1];
        c.s0ds = scal[(size_t)tk * 4 + 2];
        return c;
    };
    // The whole column of per-token terms is in registers; 16 rows of the next chunk are requested as soon as the sweep has
    // used those of this one.  Row s is used at t >= s only, and the
    // producer leaves out the 16 x 16 tiles that lie entirely below that: those are neither read nor used.
    float xr[GW];
#pragma unroll
    for (int i = 0; i < GW; i++) xr[i] = 0.f;
    auto request = [&](int tk, int b) __attribute__((always_inline)) {
        const float *x = xs + (size_t)tk * GW * GW + lane;
        if ((lane >> 4) >= b) {
#pragma unroll
            for (int i = 16 * b; i < 16 * b + 16; i++) xr[i] = x[i * GW];
        }
    };
    Chunk coming = chunk_of(task);
#pragma unroll
    for (int b = 0; b < GW / 16; b++) request(task, b);
    for (; task < ntask; task += step_tasks) {
        const Chunk c = coming;
        const int L = c.L, after = task + step_tasks;
        const bool in = lane < L;
        int own = lane;
        asm volatile("" : "+v"(own));   // as if new for each chunk: 64 comparisons kept for all of them would not fit the scalar registers
        if (after < ntask) coming = chunk_of(after);
        wave_lds_order();   // the chunk before has been read
        gr.keep[lane] = in ? T(1) - T(c.alpha) : T(1);
        gr.eta[lane] = c.eta;
        gr.g1[lane] = c.pv.z;
        gr.g2[lane] = c.pv.w;

        // ── sweep 1: lane = t ──
        T u = c.pv.x, v = c.pv.y;                    // <M_s, dy_t q_t^T>, <S_s, dy_t q_t^T>
        T um = c.m0dm, vm = c.s0dm, vs = c.s0ds;     // <M_s, dMo>, <S_s, dMo>, <S_s, dSo> (wave-uniform)
        T pum = um, pvm = vm, pvs = vs;              // their values at s = lane - 1
        U[tri_row(0) + lane] = (float)u;
        if (HAS_S) V[tri_row(0) + lane] = (float)v;
        wave_lds_order();   // the gates for the sweep; and row 0 before the others
        Four<T> kpn = four_at(gr.keep);
        Four<float> etn = four_at(gr.eta), g1n = four_at(gr.g1), g2n = four_at(gr.g2);
#pragma unroll
        for (int s0 = 0; s0 < GW; s0 += 4) {
            const Four<T> kp4 = kpn;
            const Four<float> et4 = etn, g14 = g1n, g24 = g2n;
            const int next = s0 + 4 < GW ? s0 + 4 : s0;   // requested four steps ahead of their use
            kpn = four_at(gr.keep + next);
            etn = four_at(gr.eta + next);
            g1n = four_at(gr.g1 + next);
            g2n = four_at(gr.g2 + next);
#pragma unroll
            for (int i = 0; i < 4; i++) {
                const int sx = s0 + i;
                const T xv = xr[sx], kp = kp4.x[i], g1 = g14.x[i];
                if (HAS_S) {
                    const T et = et4.x[i], g2 = g24.x[i];
                    v = fma(et, v, xv);
                    vm = fma(et, vm, g1);
                    vs = fma(et, vs, g2);
                } else {
                    v = xv;
                    vm = g1;
                }
                u = fma(kp, u, v);
                um = fma(kp, um, vm);
                if (sx + 1 < GW) {
                    U[tri_row(sx + 1) + lane] = (float)u;
                    if (HAS_S) V[tri_row(sx + 1) + lane] = (float)v;
                    asm volatile("" ::: "memory");   // the next row's stores stay behind these and apart from them
                    if (own == sx + 1) { pum = um; pvm = vm; pvs = vs; }
                }
            }
            // the choices are made here: put off behind the sweep they would keep 192 values in registers
            asm volatile("" : "+v"(pum), "+v"(pvm), "+v"(pvs));
            if (s0 % 16 == 12 && after < ntask) request(after, s0 / 16);
            __builtin_amdgcn_sched_barrier(0);
        }
        wave_lds_order();

        // ── sweep 2: lane = s; weights r[s][t], c[t][s], bb[s][t] advance with t and start, with the sums, at t = s: what the lane
        // reads before, other rows' values, leaves nothing behind ──
        T rho = 0, cc = 0, bb = 0, accA = 0, accE = 0;
        const float *Ur = U + tri_row(lane), *Vr = V + tri_row(lane);
        auto step = [&](int t, T kp, float eta_t) __attribute__((always_inline)) {
            const T x = Ur[t];
            const bool first = t == own;
            rho = first ? T(1) : rho * kp;
            accA = first ? x : fma(rho, x, accA);
            if (HAS_S) {
                const T et = eta_t, y = Vr[t];
                bb = first ? T(1) : bb * et;
                cc = first ? T(1) : fma(kp, cc, bb);
                accE = first ? y : fma(cc, y, accE);
            }
        };
        int tb = 0;
#pragma unroll 2
        for (; tb + 4 <= L; tb += 4) {
            const Four<T> kp4 = four_at(gr.keep + tb);
            const Four<float> et4 = four_at(gr.eta + tb);
#pragma unroll
            for (int i = 0; i < 4; i++) step(tb + i, kp4.x[i], et4.x[i]);
        }
        for (; tb < L; tb++) step(tb, gr.keep[tb], gr.eta[tb]);
        if (in) {
            d_alpha[c.tok + lane] = -(float)fma(rho, pum, accA);
            if (HAS_S) d_eta[c.tok + lane] = (float)(accE + cc * pvm + bb * pvs);
        }
    }
}

}  // namespace

void chunkwise_gate_gradients(const float *alpha, const float *eta, const float *pvec, const float *xs,
                              const float *scal, float *d_alpha, float *d_eta, int seq_len, int batch,
                              int chunk_size, bool has_s, const float *dm_first, const float *ds_first,
                              size_t chain_stride, int per, int nsum, float *tmp, int elems, bool wide) {
    const ErrorScope es;
    const int nc = ceil_div(seq_len, chunk_size), ntask = batch * nc;
    const size_t lds = wide ? gate_lds<double>(has_s) : gate_lds<float>(has_s);
    static bool attr_set = false;
    if (!attr_set) {
        auto lds_of = [](const void *kernel, size_t bytes) {
            check_hip(hipFuncSetAttribute(kernel, hipFuncAttributeMaxDynamicSharedMemorySize, (int)bytes), "dynamic LDS size");
        };
        lds_of(reinterpret_cast<const void *>(cw_gates_sweep_kernel<true, float>), gate_lds<float>(true));
        lds_of(reinterpret_cast<const void *>(cw_gates_sweep_kernel<false, float>), gate_lds<float>(false));
        lds_of(reinterpret_cast<const void *>(cw_gates_sweep_kernel<true, double>), gate_lds<double>(true));
        lds_of(reinterpret_cast<const void *>(cw_gates_sweep_kernel<false, double>), gate_lds<double>(false));
        attr_set = true;
    }
    if (es.failed()) return;
    static_assert(64 * kGateWaves == 256, "the sum workgroups take 256 elements each");
    // Workgroups for the places that LDS leaves, each wave walking over its chunks with the next one's terms in flight: a wave per
    // chunk waited for its 10 KB before every sweep.
    const int rows = ceil_div(batch, per), places = compute_units() * std::max(1, (int)(160 * 1024 / lds));
    const FirstSum fs{{dm_first, ds_first}, tmp, chain_stride, batch, per, rows, nsum, elems};
    const dim3 grid(std::min(ceil_div(ntask, kGateWaves) + (elems / 256) * rows * nsum, places)), block(64 * kGateWaves);
    KernelTimer kt("cw_gates_sweep_kernel");
    auto kernel = has_s ? (wide ? cw_gates_sweep_kernel<true, double> : cw_gates_sweep_kernel<true, float>)
                        : (wide ? cw_gates_sweep_kernel<false, double> : cw_gates_sweep_kernel<false, float>);
    hipLaunchKernelGGL(kernel, grid, block, lds, stream(), alpha, has_s ? eta : nullptr, pvec, xs, scal, d_alpha,
                       has_s ? d_eta : nullptr, seq_len, chunk_size, nc, ntask, fs);
    check_launch("cw_gates_sweep_kernel");
}

}  // namespace nlh
