// The pointwise part of the CCGQA prep backward (ccgqa_prep_bwd.hip), shared
// with the bf16 whole-backward path (ccgqa_conv_bwd.hip).
#pragma once

#include <hip/hip_runtime.h>
#include <stdint.h>

namespace hydra {

struct PrepBwdArgs {
  const void* qkv;
  int64_t qkv_rs;
  const void *y2q, *y2k;          // conv outputs (element type of qkv), or null without convs
  int64_t yq_b, yk_b, y_h, y_s;   // their batch (q, k), head and token strides (elements)
  const void* temp;
  const float *cs, *sn;
  int64_t cs_rs;
  const void *dq, *dk, *dv;       // [B, H, S, hd]
  void* dy;                       // [B, S, L + K] gradient of the conv outputs, or null
  void* dqkv;
  int64_t dqkv_rs;
  float* dtemp_tok;               // [B * S] or null
  int B, S, Hq, Hkv, hd, flags, dtype;
  hipStream_t st;
};

int launch_prep_bwd(const PrepBwdArgs& a);

}  // namespace hydra
