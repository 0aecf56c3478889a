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
// Both operands of the dW contraction, kept beyond the call: K-blocked with `ld` tokens, of which the first `k` (a
// multiple of 64) are in use.  A backward that is given one leaves its rows behind those and computes no dW.
struct DwOperands {
  void *dzt, *hidt;
  int64_t ld, k;
};
// Backward of the a->T rows of `rows`; hidden, per-token arrays and dhidden are indexed by order[n] (dhidden rows outside
// `rows` are left alone), kept logits by n.  An order and kept dW operands need kept logits.
int head_backward(const char* who, const clgrpo_lmhead_bwd_args* a, int64_t vocab_begin, const RowOrder& rows,
                  hipStream_t stream, const DwOperands* kept = nullptr);
// clgrpo_policy_loss with the scratch memory named apart.
int head_policy_loss(const char* who, const clgrpo_policy_loss_args* a, void* workspace, size_t workspace_bytes,
                     hipStream_t stream);

}  // namespace clgrpo
