// Groups of fp32 products that share their shape, in one launch each: the dense projections around the memory levels and the
// products with the unembedding, which the reference issues as one cublasSgemm per matrix (core/src/gpu_forward.rs:1205 ff.,
// core/src/gpu_backward.rs:2047 ff.).  At the model sizes of a training step (512 tokens x 512 x 512) one product fills a
// quarter of the chip for 10 us behind 15 us of host work; 3 + 3 * levels of them side by side fill it.
//   op 0  y_j = x_j W_j^T      a_j [m, k], b_j [n, k], c_j [m, n]      forward
//   op 1  dx = sum_j g_j W_j   a_j [m, k], b_j [k, n], c_0 [m, n]      input gradient, the sum over j inside the product
//   op 2  dW_j = g_j^T x_j     a_j [k, m], b_j [k, n], c_j [m, n]      weight gradient
//
// On the bf16 matrix cores (v_mfma_f32_16x16x32_bf16), without rounding the operands: a float is the sum of three bf16
// (hi, mid, lo: 24 bits), a product of two floats the six products of pieces that reach 2^-24 of it, summed in fp32.  Six
// products at 2.5 PFLOP/s are 416 TFLOP/s where the fp32 matrix cores have 157, and one instruction adds 32 terms before it
// rounds, the fp32 one rounds term by term.  Unit normals, 2-norm of the error over that of the result, in 1e-7, largest tile /
// others / fp32 matrix cores: k = 64: - / 0.50 / 1.45, 128: 1.9 / 0.65 / 2.0, 512: 3.5 / 1.3 / 4.1, 4096: 10 / 4.0 / 11.5;
// 32000 in parts 2.8 (8.0), the sum of fifteen products of 512 1.3 (4.1).
//
// Block tile 256 x 128 or 128 x 128 (eight waves) or 64 x 64 (four), 32-wide contraction steps, two LDS buffers.  The pieces
// are made on the way to LDS by the vector units, a few instructions behind every matrix instruction, out of registers that
// take the tile after the next at once.  What bounds it: LDS (43 % busy at 256 x 128) and the wait at a step's barrier hold
// the matrix cores at 0.62 of their clocks, and those clocks at 1.6 to 1.9 GHz under it.  4096^3: 600 us, 229 TFLOP/s; with
// products on the fp32 matrix cores 128 TFLOP/s here and 150 in the library.
#include <hip/hip_runtime.h>
#include <stdint.h>

#include <algorithm>

#include "../../include/nl_hecate_ffi.h"
#include "lane_ops.h"
#include "runtime.h"

namespace nlh {
namespace {

using f32x4 = __attribute__((ext_vector_type(4))) float;
using u32x4 = __attribute__((ext_vector_type(4))) uint32_t;
using bf16x2 = __attribute__((ext_vector_type(2))) __bf16;
using bf16x8 = __attribute__((ext_vector_type(8))) __bf16;
constexpr int kMaxGroup = 32, BK = 32;

struct GroupArgs {
    const float *a[kMaxGroup], *b[kMaxGroup];
    void *c[kMaxGroup];
    uint32_t bf16_mask;     // op 0: outputs that leave rounded to bf16
    int count, m, n, k, tiles, tiles_m, splits;
    float *part;            // splits > 1: [split][m][n]
};

// x = hi + mid + lo, three bf16 whose 24 bits hold all of x's.  Two elements at a time, packed as the matrix cores read them;
// opaque, because where the compiler sees a piece taken off it rounds that element a second time.
__device__ __forceinline__ uint32_t bf16_pair(float x, float y) {
    uint32_t p = __builtin_bit_cast(uint32_t, bf16x2{(__bf16)x, (__bf16)y});
    asm("" : "+v"(p));
    return p;
}
__device__ __forceinline__ void take_off(float &x, float &y, uint32_t p) {
    x -= __uint_as_float(p << 16);
    y -= __uint_as_float(p & 0xffff0000u);
}

// A [ROWS x BK] tile of a row-major operand, contraction contiguous (KC) or rows contiguous.  A slot is eight contraction
// indices of one row; in LDS a row is 64 bytes a piece, its four slots permuted by the row's bits 2 and 3, so that sixteen
// rows of one slot fall on different banks, and so do the two halves of rows that a 16-byte read takes together (rows 0..3,
// 12..15 of one slot with rows 4..11 of the next).
template <bool KC, int ROWS, int NTHR>
struct Operand {
    static constexpr int PER = ROWS * (BK / 8) / NTHR, PIECE = ROWS * BK;   // PIECE in elements
    static_assert(PER * NTHR == ROWS * (BK / 8), "whole slots per thread");
    float x[PER][8];
    // Slot i.  rows: how many rows of the tile exist (others repeat the last one: their results are not stored); ks:
    // contraction indices that exist (TAIL: others are zero).
    template <bool TAIL>
    __device__ __forceinline__ void load(int i, const float *p, int ld, int rows, int ks) {
        typedef float f32x4u __attribute__((ext_vector_type(4), aligned(4)));
        const int e = i * NTHR + threadIdx.x;
        const int r = min(KC ? e / (BK / 8) : e % ROWS, rows - 1);
        // rows contiguous: the contraction index is the same for a whole wave, and so are the addresses of its rows
        const int c = 8 * (KC ? e % (BK / 8) : __builtin_amdgcn_readfirstlane(e / ROWS));
        if constexpr (TAIL) {
#pragma unroll
            for (int j = 0; j < 8; j++) {
                const int k = min(c + j, ks - 1);
                const float v = KC ? p[(size_t)r * ld + k] : p[(size_t)k * ld + r];
                x[i][j] = c + j < ks ? v : 0.f;
            }
        } else if constexpr (KC) {
            const f32x4u *q = reinterpret_cast<const f32x4u *>(p + (size_t)r * ld + c);
            const f32x4u a = q[0], b = q[1];
#pragma unroll
            for (int j = 0; j < 4; j++) { x[i][j] = a[j]; x[i][4 + j] = b[j]; }
        } else {
            const float *row = p + (size_t)c * ld;
#pragma unroll
            for (int j = 0; j < 8; j++, row += ld) x[i][j] = row[(unsigned)r];
        }
    }
    static __device__ __forceinline__ int at(int r, int slot) {
        return r * BK + 8 * (slot ^ ((r >> 1) & 2) ^ ((r >> 3) & 1) * 3);
    }
    // Step q < STEPS of taking the slots to LDS: a third of a pair's pieces, or a slot's 16-byte writes behind its pairs.
    static constexpr int STEPS = PER * 13;
    u32x4 hi, mid, lo;
    __device__ __forceinline__ void store_step(uint16_t *s, int q) {
        const int i = q / 13, part = q % 13 % 3, j = q % 13 / 3;
        if (q % 13 == 12) {
            const int e = i * NTHR + threadIdx.x;
            uint16_t *to = s + at(KC ? e / (BK / 8) : e % ROWS, KC ? e % (BK / 8) : e / ROWS);
            *reinterpret_cast<u32x4 *>(to) = hi;
            *reinterpret_cast<u32x4 *>(to + PIECE) = mid;
            *reinterpret_cast<u32x4 *>(to + 2 * PIECE) = lo;
            return;
        }
        float &a = x[i][2 * j], &b = x[i][2 * j + 1];
        if (part == 0) {
            hi[j] = bf16_pair(a, b);
            take_off(a, b, hi[j]);
        } else if (part == 1) {
            mid[j] = bf16_pair(a, b);
            take_off(a, b, mid[j]);
        } else {
            lo[j] = bf16_pair(a, b);
        }
    }
    // this lane's operand of one step: row r, contraction indices 8 (l / 16) .. + 8
    static __device__ __forceinline__ bf16x8 read(const uint16_t *s, int piece, int r, int l) {
        return *reinterpret_cast<const bf16x8 *>(s + piece * PIECE + at(r, l >> 4));
    }
};

template <int OP, bool SUM, int BM, int BN, int WM, int WN>
__global__ __launch_bounds__(64 * WM * WN) void group_gemm_kernel(GroupArgs g) {
    constexpr int NTHR = 64 * WM * WN, TM = BM / WM / 16, TN = BN / WN / 16;
    using OA = Operand<OP != 2, BM, NTHR>;
    using OB = Operand<OP == 0, BN, NTHR>;
    __shared__ __align__(16) uint16_t sa[2][3 * OA::PIECE], sb[2][3 * OB::PIECE];
    // workgroups go to the eight XCDs in turn: each takes a run of tiles, the tiles of one column block of b next to
    // each other
    const int per_xcd = gridDim.x >> 3, tile = (blockIdx.x & 7) * per_xcd + (blockIdx.x >> 3);
    if (tile >= g.tiles) return;
    const int m0 = tile % g.tiles_m * BM, n0 = tile / g.tiles_m * BN;
    const int l = threadIdx.x & 63, w = threadIdx.x >> 6, wm = (w / WN) * (BM / WM), wn = (w % WN) * (BN / WN);
    const int lda = OP == 2 ? g.m : g.k, ldb = OP == 0 ? g.k : g.n;
    const int per_seg = g.k / BK;                                // whole steps of one product
    const int total = SUM ? per_seg * g.count : per_seg;
    const int per = (total + g.splits - 1) / g.splits, s0 = min(total, (int)blockIdx.z * per), s1 = min(total, s0 + per);
    OA ra;
    OB rb;
    struct Source { const float *a, *b; };
    auto source = [&](int j, int k0) -> Source {
        return {g.a[j] + (OP == 2 ? (size_t)k0 * lda + m0 : (size_t)m0 * lda + k0),
                g.b[j] + (OP == 0 ? (size_t)n0 * ldb + k0 : (size_t)k0 * ldb + n0)};
    };
    auto step_source = [&](int step) -> Source {
        const int j = SUM ? step / per_seg : blockIdx.y;
        return source(j, (SUM ? step - j * per_seg : step) * BK);
    };
    auto load = [&](const Source &p, int i) __attribute__((always_inline)) {
        if (i < OA::PER) ra.template load<false>(i, p.a, lda, g.m - m0, BK);
        else rb.template load<false>(i - OA::PER, p.b, ldb, g.n - n0, BK);
    };
    // A sum over products adds whole products: one running sum over all of their terms rounds like a contraction of that
    // length.
    // The five smaller products have a sum of their own where the registers hold one, so that the first piece's sum rounds
    // once a step.
    constexpr bool APART = TM * TN <= 8;
    f32x4 acc[TM][TN], small[APART ? TM : 1][APART ? TN : 1], sum[SUM ? TM : 1][SUM ? TN : 1];
#pragma unroll
    for (int i = 0; i < TM; i++)
#pragma unroll
        for (int j = 0; j < TN; j++) {
            acc[i][j] = f32x4{0.f, 0.f, 0.f, 0.f};
            if constexpr (APART) small[i][j] = acc[i][j];
            if constexpr (SUM) sum[i][j] = acc[i][j];
        }
    // Step s: the first pieces of its operands are in registers, the next step's tile as well.  While the products of a's
    // first piece run, the other pieces are read and the next tile is taken apart, a few instructions behind each matrix
    // instruction; then the wave meets the others and requests the next first pieces under the rest.
    bf16x8 av[3][TM], bv[3][TN];
    auto read_a = [&](int buf, int p) __attribute__((always_inline)) {
#pragma unroll
        for (int i = 0; i < TM; i++) av[p][i] = OA::read(sa[buf], p, wm + 16 * i + (l & 15), l);
    };
    auto read_b = [&](int buf, int p) __attribute__((always_inline)) {
#pragma unroll
        for (int j = 0; j < TN; j++) bv[p][j] = OB::read(sb[buf], p, wn + 16 * j + (l & 15), l);
    };
    auto multiply_tile = [&](int pa, int pb, int i, int j) __attribute__((always_inline)) {
        f32x4 &c = APART && pa + pb > 0 ? small[APART ? i : 0][APART ? j : 0] : acc[i][j];
        c = __builtin_amdgcn_mfma_f32_16x16x32_bf16(av[pa][i], bv[pb][j], c, 0, 0, 0);
    };
    auto multiply = [&](int pa, int pb) __attribute__((always_inline)) {
#pragma unroll
        for (int i = 0; i < TM; i++)
#pragma unroll
            for (int j = 0; j < TN; j++) multiply_tile(pa, pb, i, j);
    };
    auto join = [&]() __attribute__((always_inline)) {
        if constexpr (APART) {
#pragma unroll
            for (int i = 0; i < TM; i++)
#pragma unroll
                for (int j = 0; j < TN; j++) { acc[i][j] += small[i][j]; small[i][j] = f32x4{0.f, 0.f, 0.f, 0.f}; }
        }
    };
    constexpr int STEPS = OA::STEPS + OB::STEPS;
    auto store_step = [&](int buf, int q) __attribute__((always_inline)) {
        if (q < OA::STEPS) ra.store_step(sa[buf], q);
        else rb.store_step(sb[buf], q - OA::STEPS);
    };
    constexpr int SLOTS = OA::PER + OB::PER;
    if (s0 < s1) {
        const Source p = step_source(s0), p1 = step_source(min(s0 + 1, s1 - 1));
#pragma unroll
        for (int i = 0; i < SLOTS; i++) load(p, i);
#pragma unroll
        for (int q = 0; q < STEPS; q++) {
            store_step(0, q);
            if (q % 13 == 12) load(p1, q / 13);
        }
    }
    __syncthreads();
    read_a(0, 0);
    read_b(0, 0);
    for (int s = s0; s < s1; s++) {
        const int buf = (s - s0) & 1;
        const Source next = step_source(min(s + 2, s1 - 1));   // behind the last step: the last tile again, not used
        __builtin_amdgcn_sched_barrier(0);
        read_b(buf, 1);
        read_b(buf, 2);
        read_a(buf, 1);
#pragma unroll
        for (int p = 0; p < 3; p++) {
            if (p == 2) read_a(buf, 2);
#pragma unroll
            for (int t = 0; t < TM * TN; t++) {
                constexpr int ALL = 3 * TM * TN;
                const int n = p * TM * TN + t, i = t / TN, j = t % TN;
                __builtin_amdgcn_sched_barrier(0);
                multiply_tile(0, p, i, j);
                __builtin_amdgcn_sched_barrier(0);
#pragma unroll
                for (int q = n * STEPS / ALL; q < (n + 1) * STEPS / ALL; q++) {
                    store_step(buf ^ 1, q);
                    if (q % 13 == 12) load(next, q / 13);   // a slot's registers take the tile after the next at once
                }
            }
        }
        __builtin_amdgcn_sched_barrier(0);
        __syncthreads();
        read_a(buf ^ 1, 0);
        __builtin_amdgcn_sched_barrier(0);
        multiply(1, 0);
        multiply(2, 0);
        __builtin_amdgcn_sched_barrier(0);
        read_b(buf ^ 1, 0);
        __builtin_amdgcn_sched_barrier(0);
        multiply(1, 1);
        if constexpr (SUM) {
            if ((s + 1) % per_seg == 0) {
                join();
#pragma unroll
                for (int i = 0; i < TM; i++)
#pragma unroll
                    for (int j = 0; j < TN; j++) { sum[i][j] += acc[i][j]; acc[i][j] = f32x4{0.f, 0.f, 0.f, 0.f}; }
            }
        }
    }
    // contraction indices behind the last whole step
    if (g.k % BK && blockIdx.z == gridDim.z - 1) {
        for (int j = SUM ? 0 : blockIdx.y; j < (SUM ? g.count : (int)blockIdx.y + 1); j++) {
            const Source p = source(j, per_seg * BK);
#pragma unroll
            for (int i = 0; i < OA::PER; i++) ra.template load<true>(i, p.a, lda, g.m - m0, g.k % BK);
#pragma unroll
            for (int i = 0; i < OB::PER; i++) rb.template load<true>(i, p.b, ldb, g.n - n0, g.k % BK);
            __syncthreads();
#pragma unroll
            for (int q = 0; q < STEPS; q++) store_step(0, q);
            __syncthreads();
#pragma unroll
            for (int q = 0; q < 3; q++) { read_a(0, q); read_b(0, q); }
            multiply(0, 2); multiply(2, 0); multiply(1, 1); multiply(0, 1); multiply(1, 0); multiply(0, 0);
        }
    }
    join();
    if constexpr (SUM) {
#pragma unroll
        for (int i = 0; i < TM; i++)
#pragma unroll
            for (int j = 0; j < TN; j++) acc[i][j] += sum[i][j];
    }
    const int row0 = m0 + wm + 4 * (l >> 4), col0 = n0 + wn + (l & 15);
    // Pieces of an infinity, and of what rounds to one, are not numbers, and pieces of a float below 2^-110 end at the last of a
    // bf16's range, 2^-133, short of its 24 bits: a wave whose results are not all finite, or in part too small to tell that
    // their operands were not (2^-80, as much as 2^30 above), forms them again from the operands as they are.
    constexpr uint32_t kSmall = (127 - 80) << 23;
    bool sound = true;
#pragma unroll
    for (int i = 0; i < TM; i++)
#pragma unroll
        for (int j = 0; j < TN; j++)
#pragma unroll
            for (int e = 0; e < 4; e++) {
                const uint32_t u = __float_as_uint(acc[i][j][e]) & 0x7fffffffu;
                sound &= u - kSmall < 0x7f800000u - kSmall || u == 0 || row0 + 16 * i + e >= g.m || col0 + 16 * j >= g.n;
            }
    if (__any(!sound)) {
#pragma unroll
        for (int i = 0; i < TM; i++)
#pragma unroll
            for (int j = 0; j < TN; j++) acc[i][j] = f32x4{0.f, 0.f, 0.f, 0.f};
        const int s2 = blockIdx.z == gridDim.z - 1 && g.k % BK ? s1 + (SUM ? g.count : 1) : s1;
        for (int s = s0; s < s2; s++) {
            const int seg = !SUM ? blockIdx.y : s < s1 ? s / per_seg : s - s1;
            const int k0 = (s >= s1 ? per_seg : SUM ? s % per_seg : s) * BK;
            const float *a = g.a[seg], *b = g.b[seg];
            for (int kk = k0; kk < min(k0 + BK, g.k); kk += 4) {
                const int k = kk + (l >> 4);
                const size_t kc = min(k, g.k - 1);
                float av[TM], bv[TN];
#pragma unroll
                for (int i = 0; i < TM; i++) {
                    const size_t r = min(m0 + wm + 16 * i + (l & 15), g.m - 1);
                    av[i] = k < g.k ? (OP == 2 ? a[kc * lda + r] : a[r * lda + kc]) : 0.f;
                }
#pragma unroll
                for (int j = 0; j < TN; j++) {
                    const size_t r = min(n0 + wn + 16 * j + (l & 15), g.n - 1);
                    bv[j] = k < g.k ? (OP == 0 ? b[r * ldb + kc] : b[kc * ldb + r]) : 0.f;
                }
#pragma unroll
                for (int i = 0; i < TM; i++)
#pragma unroll
                    for (int j = 0; j < TN; j++)
                        acc[i][j] = __builtin_amdgcn_mfma_f32_16x16x4f32(av[i], bv[j], acc[i][j], 0, 0, 0);
            }
        }
    }
    const bool part = g.splits > 1, b16 = OP == 0 && ((g.bf16_mask >> blockIdx.y) & 1);
    float *c = part ? g.part + (size_t)blockIdx.z * g.m * g.n : reinterpret_cast<float *>(g.c[OP == 1 ? 0 : blockIdx.y]);
#pragma unroll
    for (int i = 0; i < TM; i++)
#pragma unroll
        for (int j = 0; j < TN; j++) {
            const int col = col0 + 16 * j;
#pragma unroll
            for (int e = 0; e < 4; e++) {
                const int row = row0 + 16 * i + e;
                if (row < g.m && col < g.n) {
                    if (b16) reinterpret_cast<uint16_t *>(c)[(size_t)row * g.n + col] = f32_to_bf16_rne(acc[i][j][e]);
                    else c[(size_t)row * g.n + col] = acc[i][j][e];
                }
            }
        }
}

template <int V>
__global__ __launch_bounds__(256) void group_sum_kernel(const float *__restrict__ part, float *__restrict__ c, long long n, int splits) {
    using Vec = __attribute__((ext_vector_type(V))) float;
    const long long i = (long long)blockIdx.x * 256 + threadIdx.x;
    if (i >= n / V) return;
    Vec s = 0.f;
    for (int z = 0; z < splits; z++) s += reinterpret_cast<const Vec *>(part + z * n)[i];
    reinterpret_cast<Vec *>(c)[i] = s;
}

enum Tile { kHuge, kBig, kSmall };
template <int OP, bool SUM>
void launch(const GroupArgs &g, Tile tile, int ny) {
    const dim3 grid((unsigned)(8 * ceil_div(g.tiles, 8)), (unsigned)ny, (unsigned)g.splits);
    if constexpr (!SUM) {
        if (tile == kHuge) hipLaunchKernelGGL((group_gemm_kernel<OP, SUM, 256, 128, 4, 2>), grid, dim3(512), 0, stream(), g);
    }
    if (tile == kBig) hipLaunchKernelGGL((group_gemm_kernel<OP, SUM, 128, 128, 4, 2>), grid, dim3(512), 0, stream(), g);
    if (tile == kSmall) hipLaunchKernelGGL((group_gemm_kernel<OP, SUM, 64, 64, 2, 2>), grid, dim3(256), 0, stream(), g);
    check_launch("group_gemm_kernel");
}

// Sizes are checked; a, b, c are in g.
void products(GroupArgs g, int op) {
    const ErrorScope es;
    // Tile and split: the fullest compute unit's time, from what a step takes with every compute unit busy (4096^3: 229, 199
    // and 150 TFLOP/s) and what filling and storing a tile takes (512 x 32000 x 512: 95 us with the largest tile, 112 and 132
    // with the others; twelve products of 512^3: 42, 28, 28).  Single products and a sum over products (op 1) have few output
    // tiles: their contraction is split until one workgroup (64-wide tiles: two) per compute unit is there, for another
    // pass over the parts (512 x 512 x 32000: 101 us in 32 parts of the largest tile, 115 in 16 of the next).
    const bool sum = op == 1 && g.count > 1;
    const int cus = compute_units(), ny = op == 1 ? 1 : g.count, total = ceil_div(g.k, BK) * (op == 1 ? g.count : 1);
    constexpr int kRows[3] = {256, 128, 64}, kCols[3] = {128, 128, 64}, kPerCu[3] = {1, 1, 2}, kSplits[3] = {32, 16, 16};
    constexpr double kStep[3] = {2.35, 1.35, 0.44}, kTile[3] = {9, 5, 1.5};   // us
    double best = 0;
    Tile tile = kSmall;
    // The largest tile has no registers for a second sum: below 128 terms it would round more often than term by term sums.
    for (int t = kSmall; t >= (sum || g.k < 128 ? kBig : kHuge); t--) {
        const int tiles = ceil_div(g.m, kRows[t]) * ceil_div(g.n, kCols[t]);
        int s = ny == 1 && !g.bf16_mask ? kPerCu[t] * cus / tiles : 1;
        s = std::max(1, std::min({s, total / 4, kSplits[t]}));
        const double time = ceil_div((long long)tiles * ny * s, cus) * (ceil_div(total, s) * kStep[t] + kTile[t])
                          + (s > 1 ? 4 + 2e-6 * s * g.m * g.n : 0);
        if (t == kSmall || time < best) {
            best = time;
            tile = (Tile)t;
            g.tiles = tiles;
            g.tiles_m = ceil_div(g.m, kRows[t]);
            g.splits = s;
        }
    }
    const long long n = (long long)g.m * g.n;
    if (g.splits > 1) {
        g.part = scratch(37, g.splits * n * sizeof(float));
        if (es.failed()) return;
    }
    KernelTimer kt("group_gemm_kernel");
    if (op == 0) launch<0, false>(g, tile, ny);
    else if (op == 2) launch<2, false>(g, tile, ny);
    else if (sum) launch<1, true>(g, tile, ny);
    else launch<1, false>(g, tile, ny);
    if (g.splits > 1) {
        float *c = reinterpret_cast<float *>(g.c[0]);
        if (n % 4 == 0 && (uintptr_t)c % 16 == 0)
            hipLaunchKernelGGL(group_sum_kernel<4>, dim3((unsigned)((n / 4 + 255) / 256)), dim3(256), 0, stream(), g.part, c, n, g.splits);
        else
            hipLaunchKernelGGL(group_sum_kernel<1>, dim3((unsigned)((n + 255) / 256)), dim3(256), 0, stream(), g.part, c, n, g.splits);
        check_launch("group_sum_kernel");
    }
}

}  // namespace
}  // namespace nlh

extern "C" void linear_group_f32_rocm(int op, int count, const float *const *a, const float *const *b, void *const *c,
                                      unsigned bf16_mask, int m, int n, int k) {
    using namespace nlh;
    const char *fn = "linear_group_f32_rocm";
    if (op < 0 || op > 2 || count < 1 || count > kMaxGroup || m < 0 || n < 1 || k < 1) {
        fail("%s: op=%d (0..2), count=%d (1..%d), m=%d, n=%d, k=%d.", fn, op, count, kMaxGroup, m, n, k);
        return;
    }
    if (n % 4 || (op == 2 ? m : k) % 4) {
        fail("%s: n=%d and %s=%d must be multiples of 4.", fn, n, op == 2 ? "m" : "k", op == 2 ? m : k);
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
    g.count = count; g.m = m; g.n = n; g.k = k;
    products(g, op);
}

extern "C" void product_f32_rocm(int op, const float *a, const float *b, float *c, int m, int n, int k) {
    using namespace nlh;
    if (op < 0 || op > 2 || m < 0 || n < 0 || k < 1) {
        fail("product_f32_rocm: op=%d (0..2), m=%d, n=%d, k=%d.", op, m, n, k);
        return;
    }
    if (m == 0 || n == 0) return;
    GroupArgs g{};
    g.a[0] = a; g.b[0] = b; g.c[0] = c;
    g.count = 1; g.m = m; g.n = n; g.k = k;
    products(g, op);
}
