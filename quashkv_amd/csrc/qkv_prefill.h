// Attention of many query rows per kv head over the compressed store
// (qkv_prefill.hip): prompts and prompt chunks.
#pragma once

#include "qkv_attn_dev.h"

struct QkvPrefillArgs {
  const void* q;
  int q_dtype;
  qkv_attn::KVLayers kv;  // entry 0; paged or contiguous, key ranges, causal position
  int64_t t_stride, T;
  int B, Hq, Hkv, Q, d, kbits, vbits;  // kbits: key MSE bits
  const float* pi;
  const float* kcent;  // host codebooks
  const float* vcent;
  const float* signs;
  float qjl_scale, scale;
  int causal;
  void* out;
  int out_dtype;
  int n_splits;
  float* part_o;   // split partials (n_splits > 1)
  float* part_ml;
};

// Query rows per kv head below which no call is worth a 128-row workgroup.
constexpr int kPrefillMinRows = 48;

// Whether the kernel takes these codebooks (symmetric, with f16 levels).
bool qkv_prefill_ok(int d, int kbits, int vbits, const float* kcent, const float* vcent,
                    float qjl_scale);
// Splits of T for R query rows in each of bh (sequence, kv head) groups.
int qkv_prefill_splits(int64_t bh, int R, int d, int64_t T);
int qkv_prefill(const QkvPrefillArgs& a, hipStream_t s);
