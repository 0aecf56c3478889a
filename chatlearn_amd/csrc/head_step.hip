// One token chunk of a training step of the head in a single call: forward, policy loss, backward, enqueued back to
// back on the caller's stream.  The arithmetic is that of the stages' own entry points; what this file adds is
// the order of rows.  Rows that carry no gradient (loss mask zero) come last in `row_order`, so that the kept
// logits, both backward GEMMs and the d(logits) pass see a dense problem of the first n_live rows, while every
// per-token array and the hidden states stay where the caller has them: the forward's operand loads, the
// transposition of the hidden states and the dhidden stores go through the order themselves.  That takes the
// place of nine launches and two [T, H] copies (gathers, scatters, zero fills) that cost a 16384-token micro-batch
// at H = 4096 0.35 ms, and of the host's work on them: a 200-token step took 433 us, most of it on the host,
// 268 us with this call.
#include "head_internal.hpp"

namespace clgrpo {

// Rows without a gradient: dhidden zero, and the per-token outputs of a forward that left them out.
struct MaskedRows {
  const int32_t* rows;
  char* dhidden;          // or nullptr
  int64_t row_bytes;      // a multiple of 16
  float *logprob, *entropy, *lse;   // or nullptr
};
__global__ __launch_bounds__(256) void masked_rows_kernel(MaskedRows p) {
  typedef uint32_t u32x4 __attribute__((ext_vector_type(4)));
  const int64_t t = p.rows[blockIdx.x];
  if (p.dhidden) {
    u32x4* row = reinterpret_cast<u32x4*>(p.dhidden + t * p.row_bytes);
    for (int64_t i = threadIdx.x; i < p.row_bytes / 16; i += 256) row[i] = u32x4{0, 0, 0, 0};
  }
  if (threadIdx.x == 0 && p.logprob) { p.logprob[t] = 0.f; p.entropy[t] = 0.f; p.lse[t] = 0.f; }
}

__global__ __launch_bounds__(256) void zero_floats_kernel(float* p, int64_t n) {
  for (int64_t i = (int64_t)blockIdx.x * 256 + threadIdx.x; i < n; i += (int64_t)gridDim.x * 256) p[i] = 0.f;
}

// Scratch memory: the forward's records and the backward's operands one after the other in the same place, the
// loss's own and the upstream gradient of the entropy beside them.
struct StepPlan {
  size_t off_loss, off_gent, off_big, big_bytes, total;
};
static StepPlan step_plan(int64_t T, int64_t n_live, int64_t H, int64_t V, int64_t B, int32_t dtype, int32_t flags, size_t cap) {
  StepPlan pl;
  size_t off = 0;
  pl.off_loss = off; off += align_up(clgrpo_policy_loss_workspace_bytes(T, B), 256);
  pl.off_gent = off; off += align_up((size_t)T * sizeof(float), 256);
  pl.off_big = off;
  size_t big = clgrpo_lmhead_fwd_workspace_bytes(T, H, V, dtype);
  if (n_live > 0) {
    size_t bwd = clgrpo_lmhead_bwd_workspace_bytes(n_live, H, V, dtype, n_live, flags);
    for (int64_t chunk = n_live; !(flags & 1) && bwd > cap && chunk > 256;) {     // recomputed logits: halve the chunk until it fits
      chunk = (chunk / 2 + 255) / 256 * 256;
      if (chunk < 256) chunk = 256;
      bwd = clgrpo_lmhead_bwd_workspace_bytes(n_live, H, V, dtype, chunk, flags);
    }
    if (bwd > big) big = bwd;
  }
  pl.big_bytes = align_up(big, 256);
  pl.total = off + pl.big_bytes;
  return pl;
}

}  // namespace clgrpo

using namespace clgrpo;

extern "C" size_t clgrpo_head_step_workspace_bytes(int64_t T, int64_t n_live, int64_t H, int64_t V, int64_t B, int32_t dtype,
                                                   int32_t flags, size_t recompute_cap) {
  if (T <= 0 || n_live < 0 || n_live > T || H <= 0 || V <= 0 || B <= 0 || (dtype != CLGRPO_BF16 && dtype != CLGRPO_F32)) return 0;
  return step_plan(T, n_live, H, V, B, dtype, flags, recompute_cap).total;
}

extern "C" int64_t clgrpo_head_step_max_ordered_bytes(void) { return kMaxOrderedBytes; }

extern "C" int clgrpo_head_step(const clgrpo_head_step_args* a, void* stream) {
  static const char* who = "clgrpo_head_step";
  CLGRPO_REQUIRE_PTR(a, "args");
  if (a->T <= 0 || a->n_live < 0 || a->n_live > a->T || a->B <= 0)
    return fail(CLGRPO_EINVAL, "%s: T=%lld n_live=%lld B=%lld", who, (long long)a->T, (long long)a->n_live, (long long)a->B);
  if (a->dtype != CLGRPO_BF16 && a->dtype != CLGRPO_F32) return fail(CLGRPO_EDTYPE, "%s: dtype %d", who, a->dtype);
  if (a->n_live < a->T) CLGRPO_REQUIRE_PTR(a->row_order, "row_order");
  CLGRPO_REQUIRE_PTR(a->workspace, "workspace");
  CLGRPO_REQUIRE_PTR(a->labels, "labels");
  CLGRPO_REQUIRE_PTR(a->g_logprob, "g_logprob");
  const bool saved = a->saved_logits != nullptr;
  const bool keep_dw = a->kept_dzt != nullptr;
  const int64_t n_fwd = a->forward_live_only ? a->n_live : a->T;
  // What a stage would refuse only behind the launches of the ones before it, or not at all.
  if ((a->stages & 5) && saved && a->n_live > 0 && a->saved_rows < round_up64(a->n_live, 256))
    return fail(CLGRPO_ESHAPE, "%s: saved_rows=%lld, but %lld rows keep their logits (rounded up to 256)", who,
                (long long)a->saved_rows, (long long)a->n_live);
  if ((a->stages & 1) && n_fwd < a->T) {       // the other rows' outputs are cleared
    CLGRPO_REQUIRE_PTR(a->logprob, "logprob");
    CLGRPO_REQUIRE_PTR(a->entropy, "entropy");
    CLGRPO_REQUIRE_PTR(a->lse, "lse");
  }
  if (a->stages & 2) {
    CLGRPO_REQUIRE_PTR(a->cu_seqlens, "cu_seqlens");
    CLGRPO_REQUIRE_PTR(a->sums, "sums");
    CLGRPO_REQUIRE_PTR(a->flags, "flags");
    if (a->chunk < 0) return fail(CLGRPO_EINVAL, "%s: chunk=%lld", who, (long long)a->chunk);
  }
  if (keep_dw) CLGRPO_REQUIRE_PTR(a->kept_hidt, "kept_hidt");
  if ((a->stages & 4) && a->n_live > 0) {
    if (!saved && (a->row_order != nullptr || keep_dw))
      return fail(CLGRPO_ESHAPE, "%s: a row order and kept dweight operands need kept logits", who);
    if (keep_dw && (a->kept_k < 0 || a->kept_k % 64 != 0 || a->kept_ld % 64 != 0 || a->kept_k + round_up64(a->n_live, 64) > a->kept_ld))
      return fail(CLGRPO_ESHAPE, "%s: %lld tokens do not fit behind the %lld of %lld kept for dweight", who, (long long)a->n_live,
                  (long long)a->kept_k, (long long)a->kept_ld);
    if (a->dhidden == nullptr && a->dweight == nullptr && !keep_dw)
      return fail(CLGRPO_ENULL, "%s: both dhidden and dweight are NULL", who);
  }
  const int32_t flags = (saved ? 1 : 0) | (a->weight_t ? 2 : 0) | (keep_dw ? 4 : 0);
  const StepPlan pl = step_plan(a->T, a->n_live, a->H, a->V, a->B, a->dtype, flags, a->recompute_cap);
  if (a->workspace_bytes < pl.total)
    return fail(CLGRPO_EWORKSPACE, "%s: workspace %zu < %zu bytes", who, a->workspace_bytes, pl.total);
  char* ws = static_cast<char*>(a->workspace);
  hipStream_t s = static_cast<hipStream_t>(stream);
  const RowOrder rows{a->row_order, a->T};
  float* g_entropy = a->entropy_coef > 0 ? reinterpret_cast<float*>(ws + pl.off_gent) : nullptr;

  if ((a->stages & 1) && n_fwd > 0) {
    clgrpo_lmhead_fwd_args f = {};
    f.hidden = a->hidden; f.weight = a->weight; f.labels = a->labels;
    f.T = n_fwd; f.H = a->H; f.V = a->V; f.dtype = a->dtype; f.inv_temperature = a->inv_temperature;
    f.logprob = a->logprob; f.entropy = a->entropy; f.lse = a->lse;
    f.workspace = ws + pl.off_big; f.workspace_bytes = pl.big_bytes;
    if (saved && a->n_live > 0) {
      f.saved_logits = a->saved_logits; f.ld_saved = a->ld_saved; f.saved_rows = a->n_live;
    }
    const int rc = head_forward(who, &f, 0, nullptr, rows, s);
    if (rc) return rc;
  }
  const bool clear_outputs = (a->stages & 1) && n_fwd < a->T;
  const bool clear_dhidden = a->dhidden && (a->stages & (a->stages & 8 ? 1 : 4));
  if (a->n_live < a->T && (clear_outputs || clear_dhidden)) {
    MaskedRows m = {};
    m.rows = a->row_order + a->n_live;
    if (clear_dhidden) { m.dhidden = static_cast<char*>(a->dhidden); m.row_bytes = a->H * (int64_t)dtype_bytes(a->dtype); }
    if (clear_outputs) { m.logprob = a->logprob; m.entropy = a->entropy; m.lse = a->lse; }
    hipLaunchKernelGGL(masked_rows_kernel, dim3((unsigned)(a->T - a->n_live)), dim3(256), 0, s, m);
    const int rc = check_launch("masked_rows_kernel");
    if (rc) return rc;
  }
  if (a->stages & 2) {
    clgrpo_policy_loss_args p = {};
    p.mode = a->mode; p.compute_dtype = a->compute_dtype; p.n = a->T; p.B = a->B; p.cu_seqlens = a->cu_seqlens;
    p.logprob = a->logprob; p.old_logprob = a->old_logprob; p.ref_logprob = a->ref_logprob; p.entropy = a->entropy;
    p.loss_mask = a->loss_mask; p.advantages = a->advantages;
    p.diff_clip_ratio = a->diff_clip_ratio; p.pos_clip_ratio = a->pos_clip_ratio; p.neg_clip_ratio = a->neg_clip_ratio;
    p.final_clip_ratio = a->final_clip_ratio; p.kl_coef = a->kl_coef; p.entropy_coef = a->entropy_coef;
    p.grad_scale = a->grad_scale;
    p.loss = a->loss; p.kl = a->ref_logprob ? a->kl : nullptr; p.g_logprob = a->g_logprob; p.g_entropy = g_entropy;
    p.sums = a->sums + 8 * a->chunk; p.flags = a->flags + a->chunk; p.token_offset = a->token_offset;
    const StepResult step{a->sums, a->flags, (int)a->chunk, a->grad_scale, a->kl_coef, a->entropy_coef, a->result};
    const int rc = head_policy_loss(who, &p, ws + pl.off_loss, pl.off_gent - pl.off_loss, s, step);
    if (rc) return rc;
  }
  if (a->stages & 4) {
    if (a->n_live > 0) {
      clgrpo_lmhead_bwd_args b = {};
      b.hidden = a->hidden; b.weight = a->weight; b.labels = a->labels; b.lse = a->lse; b.entropy = a->entropy;
      b.g_logprob = a->g_logprob; b.g_entropy = g_entropy;
      b.T = a->n_live; b.H = a->H; b.V = a->V; b.dtype = a->dtype; b.inv_temperature = a->inv_temperature;
      b.dhidden = a->dhidden; b.dweight = a->dweight; b.accumulate_dweight = a->accumulate_dweight;
      b.workspace = ws + pl.off_big; b.workspace_bytes = pl.big_bytes;
      b.saved_logits = a->saved_logits; b.ld_saved = a->ld_saved; b.saved_rows = a->saved_rows;
      b.weight_t = a->weight_t; b.weight_t_ready = a->weight_t_ready;
      const DwOperands kept{a->kept_dzt, a->kept_hidt, a->kept_ld, a->kept_k};
      return head_backward(who, &b, 0, rows, s, keep_dw ? &kept : nullptr);
    }
    if (a->dweight && !a->accumulate_dweight && !keep_dw) {
      hipLaunchKernelGGL(zero_floats_kernel, dim3(4096), dim3(256), 0, s, a->dweight, a->V * a->H);
      return check_launch("zero_floats_kernel");
    }
  }
  return CLGRPO_OK;
}
