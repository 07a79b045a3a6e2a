// The exact Titans / Delta rule in chunk-parallel matrix form (exact_mm.hip): head sizes 64 and 32; frozen: the frozen-M0
// chunkwise rule with chunks of C tokens in the same kernels, at head size 32 only.
#pragma once

namespace nlh {

// Backward from states kept every C <= 64 tokens, m_ckpt / s_ckpt [batch][n_ckpt_count(seq_len, C)][d*d] (C = 1: the full
// trajectory).  Sums in float64 at head size 32 and below 32 tokens an interval, in fp32 otherwise.
bool exact_mm_applies(int d, int C);
// faster than the sequential kernel at this shape (tested: under a clip or a bound)
bool exact_backward_mm_pays(int seq_len, int batch, int d, int C, bool tested, bool frozen);
// error_clip / m_norm_guard > 0: the pass also leaves the error and state norms behind and ends with the test of
// whether a coupling could have fired, BEFORE anything is added to d_m_initial / d_s_initial; false: one may have,
// the caller runs the kernels that apply the couplings, which overwrite every other output.  s_ckpt, eta, d_eta,
// d_s_initial null without momentum (has_s false).
bool exact_backward_mm(const char *fn, bool has_s, bool frozen, int d, const float *k, const float *v, const float *q, const float *alpha,
                       const float *theta, const float *eta, const float *m_ckpt, const float *s_ckpt, const float *d_y,
                       float *d_k, float *d_v, float *d_q, float *d_alpha, float *d_theta, float *d_eta, float *d_m_initial,
                       float *d_s_initial, int seq_len, int batch, int C, float error_clip, float m_norm_guard);

// Forward: the states at the starts of all runs of `run` tokens (kExactChunk, or the frozen rule's chunk), run c's at
// element offset c * sstep * d*d of its chain's m_states / s_states (chain stride state_stride), from the initial states
// (chain stride m_stride; s_initial null: zero).  No clip, no projection.  The runs' tokens are then independent walks
// (FwdArgs::sub_chunks).  sstep 0: the states after the last token instead.
// false, and nothing launched: there is no scratch for it (scratch_if_free: under capture, on a second stream), the caller
// walks the tokens.  The runs go through that scratch in stretches that fit it.
constexpr int kExactChunk = 64;
// kept_bytes: states that the walk of the tokens writes
bool exact_forward_mm_pays(int seq_len, int batch, int d, bool final_only, int run, long long kept_bytes);
bool exact_forward_states(bool has_s, bool frozen, int d, int run, const float *k, const float *v, const float *alpha, const float *theta,
                          const float *eta, const float *m_initial, const float *s_initial, long long m_stride, float *m_states,
                          float *s_states, long long state_stride, int sstep, int seq_len, int input_stride, int batch);

}  // namespace nlh
