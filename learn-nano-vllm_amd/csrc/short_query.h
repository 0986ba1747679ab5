// Internal: attention for steps whose query ranges are short (at most 16 rows
// of query tokens x query heads per kv head): speculative-decode verification
// (nvk_varlen_prefill) and the decode of models with many query heads per kv
// head (nvk_paged_decode).  Not part of the C ABI.
#pragma once

#include <hip/hip_runtime.h>
#include <stddef.h>
#include <stdint.h>

struct ShortQueryParams {
  const uint16_t* q;
  int64_t q_stride_tok, q_stride_head;
  const uint16_t* k_cache;
  const uint16_t* v_cache;
  const int32_t* cu_q;
  const int32_t* cu_k;
  // uniform form: n_query queries per sequence (rows s * n_query .. of q) at the
  // end of its context_lens[s] keys, cu_q / cu_k unused; else null
  const int32_t* context_lens = nullptr;
  int n_query = 1;
  bool decode = false;  // a decode (uniform form, n_query 1): probabilities in two parts
  int batch;
  const int32_t* block_tables;
  int64_t bt_stride;
  int max_blocks, block_size, num_blocks;
  int num_q_heads, num_kv_heads;
  float scale;
  uint16_t* out;
  int64_t out_stride_tok, out_stride_head;
  bool f16;  // elements are f16 (else bf16)
};

// True when the short-query kernels cover a launch of these sizes: keys in pages
// of a multiple of 32 keys, max_seqlen_q * G <= 16 rows, head_dim 128.
bool short_query_applies(bool paged, int block_size, int max_seqlen_q, int num_q_heads,
                         int num_kv_heads, int head_dim, int batch);

// True when a decode of these sizes runs here rather than on the decode
// kernel: paged keys in pages of a multiple of 32 keys, head_dim 128, and 4 or
// more query heads per kv head.  The decode kernel's dot products cost VALU
// time per query head (8 heads: twice the stream's time).  Measured on MI355X,
// graph replays over inputs past the Infinity Cache, decode kernel / these:
//   16/2 heads: 1 x 100 keys 15.0 / 8.9 us, 16 x U{100..2048} 22.5 / 14.3,
//     64 x U{100..2048} 39.1 / 24.0, 192 x U{256..4096} 119.8 / 81.5;
//   16/4: 11.8 / 9.2, 19.1 / 16.7, 37.9 / 36.6, 158.9 / 149.2 us;
//   16/8 (stays): 9.6 / 9.3, 20.0 / 22.8, 57.5 / 57.2, 284.9 / 281.8 us;
//   16/16 (stays): 33 x U{100..300} 16.4 / 17.7, 48 x U{100..500} 27.8 / 27.6, 64
//     x U{100..2048} 90.2 / 87.5, 192 x U{256..4096} 485 / 479 us, and with the
//     prologue 18.4 / 21.6, 29.3 / 31.4, 91.5 / 91.0, 491 / 483 us.
// With the prologue (nvk_paged_decode_prologue), 16/2: 1 x 100 18.5 / 11.6,
// 32 x U{100..2048} 42.9 / 22.3 us; 16/4: 13.2 / 12.4, 29.0 / 27.1 us, 64 x
// U{100..2048} 37.9 / 35.6.  One or two long sequences of 4 heads are the exception
// there (16/4, 1 x 12000 keys 18.9 / 20.0 us, 2 x U{3000..4000} 14.9-16.4 / 16.1;
// without the prologue 18.1 / 16.9, 15.2 / 13.2): the host knows no lengths, and
// both forms take one kernel, so that they give the same bits.
constexpr int kDecodeKernelGroup = 2;
bool short_query_decode_applies(int block_size, int num_blocks, int num_q_heads, int num_kv_heads,
                                int head_dim, int batch);

// Workspace bytes (descriptors + partial records) for these static sizes.
// n_query 0: the varlen form; else the uniform form (of which a decode needs
// no more than nvk_paged_decode_workspace_size: at most as many waves, the same
// records).
size_t short_query_ws_bytes(int batch, int64_t max_keys, int num_q_heads, int num_kv_heads,
                            int n_query = 0);

// Enqueues the two kernels (stream-K pass, combine).  ws: 256-byte aligned,
// short_query_ws_bytes() bytes.  Returns NVK_OK or a hipError_t.
int short_query_launch(const ShortQueryParams& p, int64_t max_keys, void* ws, hipStream_t s);
