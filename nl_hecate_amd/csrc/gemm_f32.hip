// Groups of fp32 products that share their shape, in one launch each, on the fp32 matrix cores
// (v_mfma_f32_16x16x4_f32, fp32 accumulation): the dense projections around the memory levels, which the reference issues
// as one cublasSgemm per matrix (core/src/gpu_forward.rs:1205 ff., core/src/gpu_backward.rs:2047 ff.).  At the model
// sizes of a training step (512 tokens x 512 x 512) one product fills a quarter of the chip for 10 us behind 15 us of host
// work; 3 + 3 * levels of them side by side fill it.
//   op 0  y_j = x_j W_j^T      a_j [m, k], b_j [n, k], c_j [m, n]      forward
//   op 1  dx = sum_j g_j W_j   a_j [m, k], b_j [k, n], c_0 [m, n]      input gradient, the sum over j inside the product
//   op 2  dW_j = g_j^T x_j     a_j [k, m], b_j [k, n], c_j [m, n]      weight gradient
// Block tile 128 x 128 (eight waves, 32 x 64 each) or 64 x 64 (four waves, 32 x 32), 32-wide contraction steps, two LDS
// buffers, the next step's tiles in registers while this one's products run.  An operand that is contiguous along the
// contraction sits in LDS as [row][36] and a lane takes its eight contraction indices of a step with two 16-byte reads
// (16 rows fall on 64 different banks); one that is contiguous along its rows sits as [k][rows + 2], read one element at a
// time (the four lane groups, eight k apart, 16 banks apart).  So every operand is staged the way it arrives.
#include <hip/hip_runtime.h>
#include <stdint.h>

#include "../../include/nl_hecate_ffi.h"
#include "lane_ops.h"
#include "runtime.h"

namespace nlh {
namespace {

using f32x4 = __attribute__((ext_vector_type(4))) float;
constexpr int kMaxGroup = 32, BK = 32;

struct GroupArgs {
    const float *a[kMaxGroup], *b[kMaxGroup];
    void *c[kMaxGroup];
    uint32_t bf16_mask;     // op 0: outputs that leave rounded to bf16
    int count, m, n, k, tiles_n, steps, splits;
    float *part;            // splits > 1: [split][m][n]
};

// A [ROWS x BK] tile of a row-major operand, contraction contiguous (KC) or rows contiguous.
template <bool KC, int ROWS, int NTHR>
struct Operand {
    static constexpr int LD = KC ? BK + 4 : ROWS + 2, PER = ROWS * BK / 4 / NTHR, FLOATS = KC ? ROWS * LD : BK * LD;
    float4 x[PER];
    // rows / ks: how many rows and contraction indices of the tile exist; ld: the operand's row stride
    __device__ __forceinline__ void load(const float *p, int ld, int rows, int ks) {
#pragma unroll
        for (int i = 0; i < PER; i++) {
            const int e = i * NTHR + threadIdx.x;
            if constexpr (KC) {
                const int r = e / (BK / 4), c = 4 * (e % (BK / 4));
                x[i] = (r < rows && c < ks) ? *reinterpret_cast<const float4 *>(p + (size_t)r * ld + c) : make_float4(0, 0, 0, 0);
            } else {
                const int r = e / (ROWS / 4), c = 4 * (e % (ROWS / 4));
                x[i] = (r < ks && c < rows) ? *reinterpret_cast<const float4 *>(p + (size_t)r * ld + c) : make_float4(0, 0, 0, 0);
            }
        }
    }
    __device__ __forceinline__ void store(float *s) const {
#pragma unroll
        for (int i = 0; i < PER; i++) {
            const int e = i * NTHR + threadIdx.x;
            if constexpr (KC) {
                *reinterpret_cast<float4 *>(s + (e / (BK / 4)) * LD + 4 * (e % (BK / 4))) = x[i];
            } else {
                float *q = s + (e / (ROWS / 4)) * LD + 4 * (e % (ROWS / 4));
                *reinterpret_cast<float2 *>(q) = make_float2(x[i].x, x[i].y);
                *reinterpret_cast<float2 *>(q + 2) = make_float2(x[i].z, x[i].w);
            }
        }
    }
    // half h (four) of this lane's contraction indices, 8 (l / 16) + 4 h + 0..3, of row r
    static __device__ __forceinline__ f32x4 read(const float *s, int r, int h, int l) {
        const int kb = 8 * (l >> 4) + 4 * h;
        if constexpr (KC) return *reinterpret_cast<const f32x4 *>(s + r * LD + kb);
        else return f32x4{s[kb * LD + r], s[(kb + 1) * LD + r], s[(kb + 2) * LD + r], s[(kb + 3) * LD + r]};
    }
};

template <int OP, int BT, int WM, int WN>
__global__ __launch_bounds__(64 * WM * WN) void group_gemm_kernel(GroupArgs g) {
    constexpr int NTHR = 64 * WM * WN, TM = BT / WM / 16, TN = BT / WN / 16;
    using OA = Operand<OP != 2, BT, NTHR>;
    using OB = Operand<OP == 0, BT, NTHR>;
    __shared__ __align__(16) float sa[2][OA::FLOATS], sb[2][OB::FLOATS];
    const int tile_m = blockIdx.x / g.tiles_n, tile_n = blockIdx.x % g.tiles_n, m0 = tile_m * BT, n0 = tile_n * BT;
    const int l = threadIdx.x & 63, w = threadIdx.x >> 6, wm = (w / WN) * (BT / WM), wn = (w % WN) * (BT / WN);
    const int lda = OP == 2 ? g.m : g.k, ldb = OP == 0 ? g.k : g.n;
    const int per_seg = (g.k + BK - 1) / BK;                     // steps of one product
    const int total = OP == 1 ? per_seg * g.count : per_seg;
    const int per = (total + g.splits - 1) / g.splits, s0 = blockIdx.z * per, s1 = min(total, s0 + per);
    OA ra;
    OB rb;
    auto load = [&](int step) {
        const int j = OP == 1 ? step / per_seg : blockIdx.y, k0 = (OP == 1 ? step % per_seg : step) * BK;
        const int ks = g.k - k0;
        ra.load(g.a[j] + (OP == 2 ? (size_t)k0 * lda + m0 : (size_t)m0 * lda + k0), lda, g.m - m0, ks);
        rb.load(g.b[j] + (OP == 0 ? (size_t)n0 * ldb + k0 : (size_t)k0 * ldb + n0), ldb, g.n - n0, ks);
    };
    // A sum over products adds whole products: one running sum over all of their terms rounds like a contraction of that
    // length (seven of 1024: 7.6e-7 of the result instead of 5.7e-7).
    f32x4 acc[TM][TN], sum[OP == 1 ? TM : 1][OP == 1 ? TN : 1];
#pragma unroll
    for (int i = 0; i < TM; i++)
#pragma unroll
        for (int j = 0; j < TN; j++) {
            acc[i][j] = f32x4{0.f, 0.f, 0.f, 0.f};
            if constexpr (OP == 1) sum[i][j] = acc[i][j];
        }
    if (s0 < s1) load(s0);
    for (int s = s0; s < s1; s++) {
        const int buf = (s - s0) & 1;
        ra.store(sa[buf]);
        rb.store(sb[buf]);
        __syncthreads();   // the buffer is complete; the other one's readers are past their products
        if (s + 1 < s1) load(s + 1);
        f32x4 av[2][TM], bv[2][TN];
#pragma unroll
        for (int h = 0; h < 2; h++) {   // the second half is read while the first one's products run
#pragma unroll
            for (int i = 0; i < TM; i++) av[h][i] = OA::read(sa[buf], wm + 16 * i + (l & 15), h, l);
#pragma unroll
            for (int j = 0; j < TN; j++) bv[h][j] = OB::read(sb[buf], wn + 16 * j + (l & 15), h, l);
        }
#pragma unroll
        for (int h = 0; h < 2; h++)
#pragma unroll
            for (int e = 0; e < 4; e++)
#pragma unroll
                for (int i = 0; i < TM; i++)
#pragma unroll
                    for (int j = 0; j < TN; j++)
                        acc[i][j] = __builtin_amdgcn_mfma_f32_16x16x4f32(av[h][i][e], bv[h][j][e], acc[i][j], 0, 0, 0);
        if constexpr (OP == 1) {
            if ((s + 1) % per_seg == 0 || s + 1 == s1) {
#pragma unroll
                for (int i = 0; i < TM; i++)
#pragma unroll
                    for (int j = 0; j < TN; j++) { sum[i][j] += acc[i][j]; acc[i][j] = f32x4{0.f, 0.f, 0.f, 0.f}; }
            }
        }
    }
    if constexpr (OP == 1) {
#pragma unroll
        for (int i = 0; i < TM; i++)
#pragma unroll
            for (int j = 0; j < TN; j++) acc[i][j] = sum[i][j];
    }
    const bool part = g.splits > 1, b16 = OP == 0 && ((g.bf16_mask >> blockIdx.y) & 1);
    float *c = part ? g.part + (size_t)blockIdx.z * g.m * g.n : reinterpret_cast<float *>(g.c[OP == 1 ? 0 : blockIdx.y]);
#pragma unroll
    for (int i = 0; i < TM; i++)
#pragma unroll
        for (int j = 0; j < TN; j++) {
            const int col = n0 + wn + 16 * j + (l & 15);
#pragma unroll
            for (int e = 0; e < 4; e++) {
                const int row = m0 + wm + 16 * i + 4 * (l >> 4) + e;
                if (row < g.m && col < g.n) {
                    if (b16) reinterpret_cast<uint16_t *>(c)[(size_t)row * g.n + col] = f32_to_bf16_rne(acc[i][j][e]);
                    else c[(size_t)row * g.n + col] = acc[i][j][e];
                }
            }
        }
}

__global__ __launch_bounds__(256) void group_sum_kernel(const float *__restrict__ part, float *__restrict__ c, long long n4, int splits) {
    const long long i = (long long)blockIdx.x * 256 + threadIdx.x;
    if (i >= n4) return;
    f32x4 s = {0.f, 0.f, 0.f, 0.f};
    for (int z = 0; z < splits; z++) s += reinterpret_cast<const f32x4 *>(part)[(size_t)z * n4 + i];
    reinterpret_cast<f32x4 *>(c)[i] = s;
}

template <int OP>
void launch(const GroupArgs &g, bool big, int tiles, int ny) {
    const dim3 grid((unsigned)tiles, (unsigned)ny, (unsigned)g.splits);
    if (big) hipLaunchKernelGGL((group_gemm_kernel<OP, 128, 4, 2>), grid, dim3(512), 0, stream(), g);
    else hipLaunchKernelGGL((group_gemm_kernel<OP, 64, 2, 2>), grid, dim3(256), 0, stream(), g);
    check_launch("group_gemm_kernel");
}

}  // namespace
}  // namespace nlh

extern "C" void linear_group_f32_rocm(int op, int count, const float *const *a, const float *const *b, void *const *c,
                                      unsigned bf16_mask, int m, int n, int k) {
    using namespace nlh;
    const char *fn = "linear_group_f32_rocm";
    const ErrorScope es;
    if (op < 0 || op > 2 || count < 1 || count > kMaxGroup || m < 0 || n < 1 || k < 1) {
        fail("%s: op=%d (0..2), count=%d (1..%d), m=%d, n=%d, k=%d.", fn, op, count, kMaxGroup, m, n, k);
        return;
    }
    if (n % 4 || (op == 2 ? m : k) % 4) {
        fail("%s: rows are read in 16-byte pieces: n=%d and %s=%d must be multiples of 4.", fn, n, op == 2 ? "m" : "k", op == 2 ? m : k);
        return;
    }
    if (m == 0) return;
    GroupArgs g{};
    for (int j = 0; j < count; j++) {
        g.a[j] = a[j];
        g.b[j] = b[j];
        if (op != 1 || j == 0) g.c[j] = c[j];
    }
    g.bf16_mask = op == 0 ? bf16_mask : 0;
    g.count = count; g.m = m; g.n = n; g.k = k; g.splits = 1;
    // Tile and split: the large tile keeps the matrix cores of a compute unit at about 0.9 of their rate, three or four
    // workgroups of the small one at about 0.82 (4096^3: 128 and 114 of 140 TFLOP/s); what decides is how much work the
    // fullest compute unit gets.  A sum over products (op 1) and a single product with a long contraction have few output tiles: their
    // contraction is split until one (large tile) or two workgroups per compute unit are there.
    const int cus = compute_units(), ny = op == 1 ? 1 : count;
    const int big_tiles = ceil_div(m, 128) * ceil_div(n, 128), small_tiles = ceil_div(m, 64) * ceil_div(n, 64);
    const int total = op == 1 ? ceil_div(k, BK) * count : ceil_div(k, BK);
    auto splits_of = [&](int tiles, int per_cu) {
        int s = ny == 1 && !bf16_mask ? per_cu * cus / tiles : 1;
        if (s > total / 4) s = total / 4;
        return s < 1 ? 1 : (s > 16 ? 16 : s);
    };
    const int sb = splits_of(big_tiles, 1), ss = splits_of(small_tiles, 2);
    const double t_big = (double)ceil_div((long long)big_tiles * ny * sb, cus) * ceil_div(total, sb) * 4096 / 0.90;
    const double t_small = (double)ceil_div((long long)small_tiles * ny * ss, cus) * ceil_div(total, ss) * 1024 / 0.82;
    const bool big = t_big < t_small;
    g.splits = big ? sb : ss;
    g.tiles_n = ceil_div(n, big ? 128 : 64);
    if (g.splits > 1) {
        g.part = scratch(37, (size_t)g.splits * m * n * sizeof(float));
        if (es.failed()) return;
    }
    KernelTimer kt("group_gemm_kernel");
    const int tiles = big ? big_tiles : small_tiles;
    if (op == 0) launch<0>(g, big, tiles, ny);
    else if (op == 1) launch<1>(g, big, tiles, ny);
    else launch<2>(g, big, tiles, ny);
    if (g.splits > 1) {
        const long long n4 = (long long)m * n / 4;
        hipLaunchKernelGGL(group_sum_kernel, dim3((unsigned)((n4 + 255) / 256)), dim3(256), 0, stream(), g.part,
                           reinterpret_cast<float *>(g.c[0]), n4, g.splits);
        check_launch("group_sum_kernel");
    }
}
