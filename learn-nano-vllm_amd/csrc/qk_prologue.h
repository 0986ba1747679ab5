// Internal: the fused prologue (csrc/qk_prologue.hip) as the attention entry
// points that run it themselves call it.  Not part of the C ABI.
#pragma once

#include <stdint.h>

// The arguments of nvk_qk_norm_rope_store.
struct QkPrologue {
  const void* qkv;
  int64_t qkv_row_stride, n_tokens;
  const int64_t* positions;
  const void *q_norm_weight, *k_norm_weight;
  float eps;
  const float* cos_sin;
  int64_t cos_sin_stride, max_position;
  int32_t num_q_heads, num_kv_heads, head_dim;
  void* q_out;
  int64_t q_out_stride_tok, q_out_stride_head;
  void* k_out;  // null: not written
  int64_t k_out_stride_tok, k_out_stride_head;
  void *k_cache, *v_cache;
  const int32_t* slot_mapping;  // null: no store
  int64_t cache_slots;
  int32_t dtype;
  // decode steps: tokens whose context length is 0 (graph padding) store nothing,
  // and q_out is the attention's output, its rows in any order and any number;
  // null: no decode step
  const int32_t* context_lens = nullptr;
};

// Checks the arguments and launches.  with_q false: the q rows are left to the
// caller (q_out unused); nothing is launched when neither k nor v goes
// anywhere.  Returns NVK_OK or an error.
int qk_prologue_launch(const QkPrologue& p, bool with_q, void* stream);
