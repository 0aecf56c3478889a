// What the whole-step entry point shares with the entry points of its stages.
#pragma once
#include "common.hpp"

namespace clgrpo {

// A choice of rows of a [total, H] array: row n of a kernel's compact problem is row order[n] of the array
// (and entry order[n] of every per-token array); order == nullptr: row n itself.  The kernels that take one put
// the row into a 32-bit offset, so total * H * sizeof(dtype) stays within kMaxOrderedBytes.
struct RowOrder {
  const int32_t* order;
  int64_t total;
};
constexpr int64_t kMaxOrderedBytes = 0x7f000000;

// Forward of the a->T rows of `rows`; per-token outputs and labels are indexed by order[n], kept logits by n.
int head_forward(const char* who, const clgrpo_lmhead_fwd_args* a, int64_t vocab_begin, void* record, const RowOrder& rows,
                 hipStream_t stream);
// Both operands of the dW contraction, kept beyond the call: d(logits) in units and hidden^T K-blocked, `ld` tokens each, of
// which the first `k` (a multiple of 64) are in use.  A backward that is given one leaves its rows behind those and computes no dW.
struct DwOperands {
  void *dzt, *hidt;
  int64_t ld, k;
};
// Backward of the a->T rows of `rows`; hidden, per-token arrays and dhidden are indexed by order[n] (dhidden rows outside
// `rows` are left alone), kept logits by n.  An order and kept dW operands need kept logits.
int head_backward(const char* who, const clgrpo_lmhead_bwd_args* a, int64_t vocab_begin, const RowOrder& rows,
                  hipStream_t stream, const DwOperands* kept = nullptr);
// What a step of several chunks reports once its last chunk's loss is known, from the sums and flag words of all of them
// (`sums` and `flags` begin with the first chunk's, `chunk` others come before this one's); `result` NULL: nothing.
// result: [0..7] the chunks' sums added up, [8] pg, [9] kl, [10] entropy mean, [11] total loss, [12] flags, [13] masked tokens
struct StepResult {
  const double* sums;
  const int32_t* flags;
  int chunk;
  double scale, kl_coef, entropy_coef;
  double* result;
};
// clgrpo_policy_loss with the scratch memory named apart.
int head_policy_loss(const char* who, const clgrpo_policy_loss_args* a, void* workspace, size_t workspace_bytes,
                     hipStream_t stream, const StepResult& step = StepResult{});

}  // namespace clgrpo
