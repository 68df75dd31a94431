// Dense attention for few query rows against a long key range (decode steps
// and short chunks): the plan and launcher behind cab_flash_attn_fwd and
// cab_flash_attn_scores_fwd. Internal to libcab_hip.so.
#pragma once

#include "cab_internal.h"

namespace cab {

struct RowAttnProblem {
  cab_dtype_t dtype;
  int64_t B, H, Hkv, Nq, Nk, D;
  const void* q;
  const void* k;
  const void* v;
  void* out;
  float* lse;  // may be null
  int64_t qs[3], ks[3], vs[3], os[3];
  float scale;
  int causal;
  // Per-key totals (scores null: none): scores = old (keys below n_old, else
  // 0) + the softmax totals of this call; old may be scores itself.
  const float* old_scores;
  int64_t olds[2], n_old;
  float* scores;
  int64_t ss[2];
};

// Whether the few-row kernels take this problem's sizes and strides.
bool row_attn_applies(cab_dtype_t dtype, int64_t B, int64_t H, int64_t Hkv, int64_t Nq, int64_t Nk,
                      int64_t D, const int64_t* k_strides, const int64_t* v_strides, bool scores);
// Workspace bytes of such a problem (16-byte aligned).
size_t row_attn_workspace(int64_t B, int64_t H, int64_t Hkv, int64_t Nq, int64_t Nk, int64_t D,
                          bool scores);
cab_status_t row_attn_launch(const char* fn, const RowAttnProblem& p, void* ws, hipStream_t s);

}  // namespace cab
