// What the attention entry points call: one launcher per head dimension, each with its kernel instances in
// a source file of its own (flash_attention_d*.hip, flash_attention_below*.hip, flash_attention_wide.hip).
#pragma once

#include "common.hpp"

namespace tfk {

struct AttentionCall {
  const void *Q, *K, *V;
  void* O;
  int batch, Lq, Lkv, d;
  float scale_log2;
  bool bf16, k_transposed, v_transposed, causal;   // K as [D][Lkv]; V as [Dv][Lkv]; not both
  int rows;                                        // query rows per workgroup: 256, 128 or 64 (wide, causal: 64)
  bool paired;                                     // causal: two query tiles per workgroup (even tile counts)
  hipStream_t stream;
  float* part = nullptr;                           // splits > 1 (no mask, V as it comes): parts of `chunk` keys, workgroups
  int splits = 1, chunk = 0;                       // of 64 queries; room for their fp32 rows
};
int run_attention_d64(const AttentionCall& c);
int run_attention_d96(const AttentionCall& c);
int run_attention_d128(const AttentionCall& c);
// rows of c.d elements, a multiple of 8: 40..56, 72..88, 104..120; K and V as they come
int run_attention_below64(const AttentionCall& c);
int run_attention_below96(const AttentionCall& c);
int run_attention_below128(const AttentionCall& c);
int run_attention_wide(const AttentionCall& c, int D);   // 160, 192, 256; V as it comes

}  // namespace tfk
