// One product on the bf16 matrix cores with fp32 sums and an fp32 result, for sizes that leave a library kernel's large tiles
// mostly idle: the projections' gradients and the output projection of a layer step over a few hundred to a few thousand
// tokens.  Operands are bf16, or fp32 that is rounded to bf16 (nearest, even) on the way to LDS, which saves a conversion
// launch and its pass over memory.
//   op 0  c [m, n] = a [m, k] b [n, k]^T     op 1  c = a [m, k] b [k, n]     op 2  c = a [k, m]^T b [k, n]
// Block tile 64 x 64, four waves of 32 x 32, 64-wide steps.  An operand that is contiguous along the contraction sits in LDS as
// [row][72] and is read 16 bytes a lane, one that is contiguous along its rows as [k][80] and is read through
// ds_read_b64_tr_b16: both are staged the way they arrive.  Two LDS buffers, and two steps on their way in registers: a step's
// eight matrix instructions are far shorter than a memory latency, which is what bounds these sizes (about 0.6 us a step).
// Where the tiles leave compute units idle the contraction is split into runs of at least six steps, up to four workgroups a
// compute unit, and the parts are added in their order.
#include "gemm_bf16.h"

#include <hip/hip_runtime.h>
#include <stdint.h>

#include <algorithm>

#include "bf16_tiles.h"
#include "runtime.h"

namespace nlh {
namespace {

constexpr int TB = 64, kThr = 256, kColLd = 80;   // tile and step; threads; row stride of a [k][row] buffer

struct Args {
    ProductBf16 p;
    float *part;   // splits > 1: [split][m][n]
    int tiles_m, splits;
};

// A [64 rows x 64 contraction indices] tile, contraction contiguous (KC) or rows contiguous, of T = u16 (bf16) or float.
template <bool KC, class T>
struct Operand {
    static constexpr int ELEMS = KC ? TB * LDB : TB * kColLd;
    bf16x8 x[2];
    // p: the tile's first element; rows, ks: how many rows and contraction indices of it exist.  Rows behind the last repeat it
    // (their results are not stored), contraction indices behind the last are zero; along the contiguous dimension the counts
    // are multiples of eight.
    __device__ __forceinline__ void load(const T *p, long long ld, int rows, int ks) {
#pragma unroll
        for (int i = 0; i < 2; i++) {
            const int e = i * kThr + threadIdx.x, far = e >> 3, near = 8 * (e & 7);
            const int r = KC ? min(far, rows - 1) : min(near, rows - 8), c = KC ? near : far;
            const bool in = c < ks;
            const T *q = p + (KC ? r * ld + (in ? c : 0) : (in ? c : 0) * ld + r);
            if constexpr (sizeof(T) == 2) {
                x[i] = *reinterpret_cast<const bf16x8 *>(q);
            } else {
                const float4 a = *reinterpret_cast<const float4 *>(q), b = *reinterpret_cast<const float4 *>(q + 4);
                x[i] = bf16x8{(__bf16)a.x, (__bf16)a.y, (__bf16)a.z, (__bf16)a.w, (__bf16)b.x, (__bf16)b.y, (__bf16)b.z, (__bf16)b.w};
            }
            if (!in) x[i] = __builtin_bit_cast(bf16x8, uint4{0, 0, 0, 0});
        }
    }
    __device__ __forceinline__ void store(u16 *s) const {
#pragma unroll
        for (int i = 0; i < 2; i++) {
            const int e = i * kThr + threadIdx.x;
            *reinterpret_cast<bf16x8 *>(s + (e >> 3) * (KC ? LDB : kColLd) + 8 * (e & 7)) = x[i];
        }
    }
    static __device__ __forceinline__ bf16x8 read(const u16 *s, int row0, int ks) {
        if constexpr (KC) return ld_op(s, row0, ks);
        else return ld_op_tr<kColLd>(s, row0, ks);
    }
};

template <int OP, class TA, class TBe>
constexpr int kBufElems = 2 * (Operand<OP != 2, TA>::ELEMS + Operand<OP == 0, TBe>::ELEMS);

// Block tile `tile`, run `split` of the contraction; lds: kBufElems.
template <int OP, class TA, class TBe>
__device__ __forceinline__ void product(const Args &g, int tile, int split, u16 *lds) {
    using OA = Operand<OP != 2, TA>;
    using OB = Operand<OP == 0, TBe>;
    u16 *sa[2] = {lds, lds + OA::ELEMS}, *sb[2] = {lds + 2 * OA::ELEMS, lds + 2 * OA::ELEMS + OB::ELEMS};
    const ProductBf16 &p = g.p;
    const int m0 = tile % g.tiles_m * TB, n0 = tile / g.tiles_m * TB;
    const int l = threadIdx.x & 63, w = threadIdx.x >> 6, wm = (w >> 1) * 32, wn = (w & 1) * 32;
    const int total = (p.k + TB - 1) / TB, per = (total + g.splits - 1) / g.splits;
    const int s0 = min(total, split * per), s1 = min(total, s0 + per);
    OA ra[2];
    OB rb[2];
    auto load = [&](int s, int set) __attribute__((always_inline)) {
        const long long k0 = (long long)s * TB;
        const TA *a = reinterpret_cast<const TA *>(p.a) + (OP == 2 ? k0 * p.lda + m0 : m0 * p.lda + k0);
        const bool second = p.b2 && k0 >= p.k_first;
        const long long kb = second ? k0 - p.k_first : k0;
        const TBe *b = reinterpret_cast<const TBe *>(second ? p.b2 : p.b) + (OP == 0 ? n0 * p.ldb + kb : kb * p.ldb + n0);
        ra[set].load(a, p.lda, p.m - m0, (int)(p.k - k0));
        rb[set].load(b, p.ldb, p.n - n0, (int)(p.k - k0));
    };
    f32x4 acc[2][2] = {{zero4(), zero4()}, {zero4(), zero4()}};
    auto step = [&](int s, int set) __attribute__((always_inline)) {   // set = (s - s0) % 2 = its buffer
        ra[set].store(sa[set]);
        rb[set].store(sb[set]);
        if (s + 2 < s1) load(s + 2, set);
        __syncthreads();   // the buffer's earlier readers are two steps behind
#pragma unroll
        for (int ks = 0; ks < TB / 32; ks++) {
            bf16x8 av[2], bv[2];
#pragma unroll
            for (int i = 0; i < 2; i++) { av[i] = OA::read(sa[set], wm + 16 * i, ks); bv[i] = OB::read(sb[set], wn + 16 * i, ks); }
#pragma unroll
            for (int i = 0; i < 2; i++)
#pragma unroll
                for (int j = 0; j < 2; j++) acc[i][j] = mfma32(av[i], bv[j], acc[i][j]);
        }
    };
    if (s0 < s1) load(s0, 0);
    if (s0 + 1 < s1) load(s0 + 1, 1);
    for (int s = s0; s < s1; s += 2) {
        step(s, 0);
        if (s + 1 < s1) step(s + 1, 1);
    }
    float *c = g.splits > 1 ? g.part + (size_t)split * p.m * p.n : p.c;
#pragma unroll
    for (int i = 0; i < 2; i++)
#pragma unroll
        for (int j = 0; j < 2; j++)
#pragma unroll
            for (int e = 0; e < 4; e++) {
                const int row = m0 + wm + 16 * i + 4 * (l >> 4) + e, col = n0 + wn + 16 * j + (l & 15);
                if (row < p.m && col < p.n) c[(size_t)row * p.n + col] = acc[i][j][e];
            }
}

template <int OP, class TA, class TBe>
__global__ __launch_bounds__(kThr) void product_bf16_kernel(Args g) {
    __shared__ __align__(16) u16 lds[kBufElems<OP, TA, TBe>];
    product<OP, TA, TBe>(g, blockIdx.x, blockIdx.y, lds);
}
// The gradients of a projection: dW (op 2, the longer ones, first) and dx (op 1) are no larger at a few hundred tokens than
// the launch between them.  Layer step of 500 tokens, d = 256: 6 + 10 and 9 + 10 us one after the other, 11 and 12 together.
template <class TG, class TW, class TX>
__global__ __launch_bounds__(kThr) void product_bf16_pair_kernel(Args dw, Args dx, int dw_blocks, int dw_tiles, int dx_tiles) {
    constexpr int A = kBufElems<2, TG, TX>, B = kBufElems<1, TG, TW>;
    __shared__ __align__(16) u16 lds[A > B ? A : B];
    const int i = blockIdx.x;
    if (i < dw_blocks) product<2, TG, TX>(dw, i % dw_tiles, i / dw_tiles, lds);
    else product<1, TG, TW>(dx, (i - dw_blocks) % dx_tiles, (i - dw_blocks) / dx_tiles, lds);
}

__global__ __launch_bounds__(256) void product_sum_kernel(const float *__restrict__ part, float *__restrict__ c, long long n4, int splits) {
    const long long i = (long long)blockIdx.x * 256 + threadIdx.x;
    if (i >= n4) return;
    f32x4 s = reinterpret_cast<const f32x4 *>(part)[i];
    for (int z = 1; z < splits; z++) s += reinterpret_cast<const f32x4 *>(part)[z * n4 + i];
    reinterpret_cast<f32x4 *>(c)[i] = s;
}

template <int OP>
void launch(const Args &g, dim3 grid) {
    const ProductBf16 &p = g.p;
    if (p.a_bf16 && p.b_bf16) hipLaunchKernelGGL((product_bf16_kernel<OP, u16, u16>), grid, dim3(kThr), 0, stream(), g);
    else if (p.a_bf16) hipLaunchKernelGGL((product_bf16_kernel<OP, u16, float>), grid, dim3(kThr), 0, stream(), g);
    else if (p.b_bf16) hipLaunchKernelGGL((product_bf16_kernel<OP, float, u16>), grid, dim3(kThr), 0, stream(), g);
    else hipLaunchKernelGGL((product_bf16_kernel<OP, float, float>), grid, dim3(kThr), 0, stream(), g);
}

}  // namespace

bool product_bf16_serves(const ProductBf16 &p, int op) {
    const auto al16 = [](const void *x) { return ((uintptr_t)x & 15) == 0; };
    // rows along the contiguous dimension and contraction indices along it come eight at a time
    if (p.n % 8 || (op == 2 ? p.m : p.k) % 8 || p.lda % 8 || p.ldb % 8 || (p.b2 && p.k_first % TB)) return false;
    if (!al16(p.a) || !al16(p.b) || !al16(p.b2) || !al16(p.c)) return false;
    // A result in the place of an operand: the operands are read while the first tiles are stored.  The callers' other path
    // has its fp32 operands converted into scratch before anything is written.
    const auto meets = [&](const void *x, long long rows, long long cols, long long ld, bool bf16) {
        const uintptr_t x0 = (uintptr_t)x, x1 = x0 + ((rows - 1) * ld + cols) * (bf16 ? 2 : 4);
        const uintptr_t c0 = (uintptr_t)p.c, c1 = c0 + (size_t)p.m * p.n * sizeof(float);
        return x && x0 < c1 && c0 < x1;
    };
    const int kb = p.b2 ? p.k_first : p.k;
    if (meets(p.a, op == 2 ? p.k : p.m, op == 2 ? p.m : p.k, p.lda, p.a_bf16) ||
        meets(p.b, op == 0 ? p.n : kb, op == 0 ? p.k : p.n, p.ldb, p.b_bf16) || meets(p.b2, p.k - kb, p.n, p.ldb, p.b_bf16))
        return false;
    // In a captured graph, us here / library kernel with its conversions (and the library's slabs for op 2):
    //   op 0  d 512 x 512: 2000 rows 8.7 / 10.0, 4000 12.8 / 11.5; 256 x 2304: 1000 8.5 / 12.3, 2000 13 / 13
    //   op 1  256 x 2304: 500 rows 11 / 17, 2000 17 / 24, 4000 35 / 28; 512 x 7680: 500 32 / 39
    //   op 2  256 x 2304: 500 rows 7.9 / 15, 4000 24 / 50; 512 x 3072: 2000 27 / 37, 8192 79 / 66
    constexpr double kLargest[3] = {2.2e9, 3e9, 8e9};
    return 2.0 * p.m * p.n * p.k <= kLargest[op];
}

namespace {
Args product_args(const ProductBf16 &p) {
    Args g{};
    g.p = p;
    g.tiles_m = ceil_div(p.m, TB);
    g.splits = std::max(1, std::min({4 * compute_units() / (g.tiles_m * ceil_div(p.n, TB)), ceil_div(p.k, TB) / 6, 16}));
    return g;
}
size_t part_floats(const Args &g) { return g.splits > 1 ? (size_t)g.splits * g.p.m * g.p.n : 0; }
void sum_parts(const Args &g) {
    if (g.splits == 1) return;
    const long long n4 = (long long)g.p.m * g.p.n / 4;
    hipLaunchKernelGGL(product_sum_kernel, dim3((unsigned)((n4 + 255) / 256)), dim3(256), 0, stream(), g.part, g.p.c, n4, g.splits);
    check_launch("product_sum_kernel");
}
}  // namespace

void product_bf16(const ProductBf16 &p, int op) {
    const ErrorScope es;
    Args g = product_args(p);
    if (g.splits > 1) {
        g.part = scratch(30, part_floats(g) * sizeof(float));
        if (es.failed()) return;
    }
    const dim3 grid((unsigned)(g.tiles_m * ceil_div(p.n, TB)), (unsigned)g.splits);
    if (op == 0) launch<0>(g, grid);
    else if (op == 1) launch<1>(g, grid);
    else launch<2>(g, grid);
    check_launch("product_bf16_kernel");
    sum_parts(g);
}

void product_bf16_pair(const ProductBf16 &a, const ProductBf16 &b) {
    const ErrorScope es;
    const auto result_meets = [](const ProductBf16 &p, const void *x, long long rows, long long cols, long long ld, int bytes) {
        const uintptr_t x0 = (uintptr_t)x, x1 = x0 + ((rows - 1) * ld + cols) * bytes, c0 = (uintptr_t)p.c;
        return x && x0 < c0 + (size_t)p.m * p.n * sizeof(float) && c0 < x1;
    };
    const int kb = a.b2 ? a.k_first : a.k, ab = a.b_bf16 ? 2 : 4, bb = b.b_bf16 ? 2 : 4;
    const bool apart = !result_meets(b, a.a, a.m, a.k, a.lda, a.a_bf16 ? 2 : 4) && !result_meets(b, a.b, kb, a.n, a.ldb, ab) &&
                       !result_meets(b, a.b2, a.k - kb, a.n, a.ldb, ab) && !result_meets(a, b.a, b.k, b.m, b.lda, b.a_bf16 ? 2 : 4) &&
                       !result_meets(a, b.b, b.k, b.n, b.ldb, bb) && !result_meets(a, b.c, b.m, b.n, b.n, 4);
    if (!apart || a.a_bf16 != b.a_bf16 || a.b_bf16 || !b.b_bf16) {
        product_bf16(a, 1);
        if (!es.failed()) product_bf16(b, 2);
        return;
    }
    Args dx = product_args(a), dw = product_args(b);
    if (dx.splits > 1 || dw.splits > 1) {
        float *part = scratch(30, (part_floats(dx) + part_floats(dw)) * sizeof(float));
        if (es.failed()) return;
        dx.part = part;
        dw.part = part + part_floats(dx);
    }
    const int dx_tiles = dx.tiles_m * ceil_div(a.n, TB), dw_tiles = dw.tiles_m * ceil_div(b.n, TB), dw_blocks = dw_tiles * dw.splits;
    const dim3 grid((unsigned)(dw_blocks + dx_tiles * dx.splits));
    if (a.a_bf16)
        hipLaunchKernelGGL((product_bf16_pair_kernel<u16, float, u16>), grid, dim3(kThr), 0, stream(), dw, dx, dw_blocks, dw_tiles, dx_tiles);
    else
        hipLaunchKernelGGL((product_bf16_pair_kernel<float, float, u16>), grid, dim3(kThr), 0, stream(), dw, dx, dw_blocks, dw_tiles, dx_tiles);
    check_launch("product_bf16_pair_kernel");
    sum_parts(dx);
    sum_parts(dw);
}

}  // namespace nlh
