// Which pieces of eight weights the backward of the attention reads whole.  The weight tensor is heads x s rows of ws slots; a
// piece at an end of a row's window hangs over into the rows next to it (the foreign slots are masked where the piece is used),
// and only the tensor's own two ends have nothing to read behind them.
#pragma once

namespace nlh {
namespace {

// Heads whose pieces are looked at one by one: the first and the last, and all where a head holds fewer slots than a piece
// can hang over, so that it would reach through the neighbour.
__host__ __device__ __forceinline__ bool edge_head(int head, int heads, int s, int ws) {
    return head == 0 || head == heads - 1 || (long long)s * ws < 8;
}
__host__ __device__ __forceinline__ int at_most_8(int x) { return x < 8 ? x : 8; }
// Whether eight slots from `slot` on of query t's row, some of them the row's own, lie inside a head of s rows of ws slots.
__host__ __device__ __forceinline__ bool piece_inside(int t, int s, int ws, int slot) {
    return at_most_8(t) * ws + slot >= 0 && (at_most_8(s - 1 - t) + 1) * ws - slot >= 8;
}

}  // namespace
}  // namespace nlh
