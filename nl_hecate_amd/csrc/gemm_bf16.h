// Small products on the bf16 matrix cores (gemm_bf16.hip).
#pragma once

namespace nlh {

// op 0: a [m, k], b [n, k]; op 1: a [m, k], b [k, n]; op 2: a [k, m], b [k, n]; rows lda, ldb elements apart; c [m, n] fp32.
// An operand that is not bf16 is fp32.  b2: contraction indices from k_first on (op 1, 2), null if b holds all of them.
struct ProductBf16 {
    const void *a, *b, *b2;
    float *c;
    long long lda, ldb;
    int m, n, k, k_first;
    bool a_bf16, b_bf16;
};
// Sizes, alignments and places (c apart from the operands) that these kernels take, and sizes that they take faster than the
// library.
bool product_bf16_serves(const ProductBf16 &p, int op);
void product_bf16(const ProductBf16 &p, int op);   // scratch slot 30 where the contraction is split
// op 1 of a and op 2 of b, both served: side by side in one launch where neither's result meets what the other reads or writes
// and the types are those of a projection's gradients, one after the other elsewhere.
void product_bf16_pair(const ProductBf16 &a, const ProductBf16 &b);

}  // namespace nlh
