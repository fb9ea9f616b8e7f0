// Attention forward and backward on the fp32 matrix instructions
// (attn_f32.hip), for the element types, head dims and strides that the bf16
// MFMA kernels do not take; head_dim <= kAttnF32MaxHd.
#pragma once

#include <hip/hip_runtime.h>
#include <stdint.h>

namespace hydra {

constexpr int kAttnF32MaxHd = 128;

struct AttnF32Args {
  const void *q, *k, *v, *dout;  // dout: backward only
  void *o, *dq, *dk, *dv;        // o: forward only; dq, dk, dv: backward only
  float* lse;                    // forward, optional
  const float *dvec, *lse2;      // backward: rowsum(dO * O) and lse * log2(e), [B, Hq, S]
  const uint8_t* kmask;          // [B, S], nonzero = keep; null without a mask
  int mask_mode;
  int B, Hq, Hkv, S, hd;
  // strides of the batch, head and row (elements); v's also along head_dim
  const int64_t *qs, *ks, *vs, *os, *dos, *dqs, *dks, *dvs;
  bool causal;
  float scale;
  int dtype;
  hipStream_t st;
};

int attn_fwd_f32(const AttnF32Args& a);
// Scratch of the backward (fp32 partials) for these sizes; with less of it
// the walks are not cut.
size_t attn_bwd_f32_workspace(int B, int Hq, int Hkv, int S, int hd, bool causal, int mask_mode);
int attn_bwd_f32(const AttnF32Args& a, float* part, size_t part_bytes);

}  // namespace hydra
