// Cross-entropy rows of the chunked LM-head loss on gfx950.
// Reference semantics: chunked_cross_entropy / ChunkedCrossEntropyFunction
// (hydra/kernels/fused_ops.py:1303-1379, 1382-1531): per token row of logits
// x[0..V), with target t (ignore_index rows contribute nothing; other
// targets are clamped to [0, V), :1407-1422),
//   loss_row = logsumexp(x) - x[t],
// and for the backward (:1459-1531), grad_x = (softmax(x) - onehot(t)) * scale
// with scale = grad_output / n_valid, and zero rows for ignored tokens.
// The projections around it (logits = h W^T, grad_h = grad_x W,
// grad_W = grad_x^T h) are plain GEMMs and stay on hipBLASLt.
//
// One 256-thread workgroup per row: an online (max, sum-exp) pass with
// 16-byte loads, a workgroup reduction, then (backward) the row rewritten
// in place.  HBM-bound: a row is read once and written once -- rows of up to
// 32 16-byte chunks per thread (vocab <= 32768 fp32 / 65536 bf16) are held
// in registers between the two phases, longer rows are read a second time.
//
// For 16-bit hidden states and weights the backward's two GEMMs run on the
// bf16 matrix cores: ce_planes kernels write the gradient of the fp32 logits
// as two bf16 planes, hi and residual (16 significant bits together), instead
// of one fp32 row -- the same bytes, and in the logits' own memory where a row
// fits the registers.  Products of bf16 values are exact in the
// GEMMs' fp32 accumulation, so the error of the 16-bit gradients against 64
// bits stays at their rounding (1.7e-3 both), and the three fp32 GEMMs of a
// chunk (4096 tokens x 32000 x 768: 4.4 ms at 140 TFLOP/s) become 1.3 ms of
// bf16 ones.
#include "common.h"

namespace hydra {
namespace {

constexpr float kLog2e = 1.4426950408889634f;
constexpr float kLn2 = 0.6931471805599453f;

// (m, s) with s = sum exp2(x - m), merged.
__device__ __forceinline__ void lse_merge(float& m, float& s, float m2, float s2) {
  const float mx = fmaxf(m, m2);
  if (mx == -INFINITY) return;  // both empty
  s = s * __builtin_amdgcn_exp2f(m - mx) + s2 * __builtin_amdgcn_exp2f(m2 - mx);
  m = mx;
}

template <typename T, bool VEC, bool GRAD>
__global__ __launch_bounds__(256) void ce_rows_kernel(
    const T* logits, int64_t rs, const int64_t* __restrict__ targets,  // logits may alias grad
    float* __restrict__ loss, float* __restrict__ lse_out, T* grad, int64_t grs,
    const float* __restrict__ grad_scale, int V, int64_t ignore_index) {
  constexpr int E = VEC ? 16 / int(sizeof(T)) : 1;
  __shared__ float red_m[4], red_s[4];
  const int64_t row = blockIdx.x;
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  const T* x = logits + row * rs;
  // Pass 1: online max / sum of exp2 over the row, in log2 units.
  float m = -INFINITY, s = 0.f;
  for (int e = tid * E; e < V; e += 256 * E) {
    float v[E];
    // Streamed once when no gradient pass follows: non-temporal loads.
    if constexpr (VEC) load16<T, !GRAD>(x + e, v);
    else v[0] = to_f32(x[e]);
    float cm = v[0] * kLog2e;
#pragma unroll
    for (int i = 1; i < E; ++i) cm = fmaxf(cm, v[i] * kLog2e);
    if (cm == -INFINITY) continue;  // all -inf: adds nothing (and exp2(-inf + inf) is NaN)
    float cs = 0.f;
#pragma unroll
    for (int i = 0; i < E; ++i) cs += __builtin_amdgcn_exp2f(fmaf(v[i], kLog2e, -cm));
    lse_merge(m, s, cm, cs);
  }
#pragma unroll
  for (int off = 32; off > 0; off >>= 1) {
    const float m2 = __shfl_xor(m, off), s2 = __shfl_xor(s, off);
    lse_merge(m, s, m2, s2);
  }
  // x[t] is read before the barrier: with grad == logits, other threads
  // overwrite the row after it.
  const int64_t t_raw = targets[row];
  const bool valid = t_raw != ignore_index;
  const int t = static_cast<int>(t_raw < 0 ? 0 : (t_raw >= V ? V - 1 : t_raw));
  const float xt = tid == 0 ? to_f32(x[t]) : 0.f;
  if (lane == 0) { red_m[wave] = m; red_s[wave] = s; }
  __syncthreads();
  m = red_m[0];
  s = red_s[0];
#pragma unroll
  for (int w = 1; w < 4; ++w) lse_merge(m, s, red_m[w], red_s[w]);
  const float lse2 = m + __log2f(s);  // log2-domain logsumexp
  if (tid == 0) {
    loss[row] = valid ? (lse2 - xt * kLog2e) * kLn2 : 0.f;
    if (lse_out) lse_out[row] = lse2 * kLn2;
  }
  if constexpr (GRAD) {
    // Pass 2: grad = (softmax - onehot(t)) * scale; ignored rows get zeros.
    // In place is allowed (grad == logits): each element is read before
    // the same thread writes it.
    const float sc = valid ? *grad_scale : 0.f;
    T* g = grad + row * grs;
    for (int e = tid * E; e < V; e += 256 * E) {
      float v[E];
      if constexpr (VEC) load16<T>(x + e, v);
      else v[0] = to_f32(x[e]);
#pragma unroll
      for (int i = 0; i < E; ++i) {
        const float p = __builtin_amdgcn_exp2f(fmaf(v[i], kLog2e, -lse2));
        v[i] = (p - (e + i == t ? 1.f : 0.f)) * sc;
      }
      if constexpr (VEC) store16<T>(g + e, v);
      else g[e] = from_f32<T>(v[0]);
    }
  }
}

// Gradient variant for rows that fit in registers (V <= 256 * NCH * E):
// the row is read from HBM once, kept in VGPRs across the reduction, and
// rewritten from there.
template <typename T, int NCH>
__global__ __launch_bounds__(256) void ce_rows_reg_kernel(
    const T* logits, int64_t rs, const int64_t* __restrict__ targets,  // logits may alias grad
    float* __restrict__ loss, float* __restrict__ lse_out, T* grad, int64_t grs,
    const float* __restrict__ grad_scale, int V, int64_t ignore_index) {
  constexpr int E = 16 / int(sizeof(T));
  __shared__ float red_m[4], red_s[4];
  const int64_t row = blockIdx.x;
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  const T* x = logits + row * rs;
  // The row's chunks stay in registers as loaded (16-bit types packed: 128
  // VGPRs at 32 chunks, where unpacked floats would spill) and are widened
  // where used.
  uint4 raw[NCH];
  auto chunk = [&](int c, float (&f)[E]) {
    const int e = (c * 256 + tid) * E;
    if (e < V) {
      load16<T>(reinterpret_cast<const T*>(&raw[c]), f);
    } else {
#pragma unroll
      for (int i = 0; i < E; ++i) f[i] = -INFINITY;
    }
  };
  float m = -INFINITY, s = 0.f;
#pragma unroll
  for (int c = 0; c < NCH; ++c) {
    const int e = (c * 256 + tid) * E;
    raw[c] = e < V ? ld16raw<true>(x + e) : make_uint4(0, 0, 0, 0);  // read once: non-temporal
  }
#pragma unroll
  for (int c = 0; c < NCH; ++c) {
    float v[E];
    chunk(c, v);
    float cm = v[0] * kLog2e;
#pragma unroll
    for (int i = 1; i < E; ++i) cm = fmaxf(cm, v[i] * kLog2e);
    if (cm == -INFINITY) continue;
    float cs = 0.f;
#pragma unroll
    for (int i = 0; i < E; ++i) cs += __builtin_amdgcn_exp2f(fmaf(v[i], kLog2e, -cm));
    lse_merge(m, s, cm, cs);
  }
#pragma unroll
  for (int off = 32; off > 0; off >>= 1) {
    const float m2 = __shfl_xor(m, off), s2 = __shfl_xor(s, off);
    lse_merge(m, s, m2, s2);
  }
  // x[t] is read before the barrier: with grad == logits, other threads
  // overwrite the row after it.
  const int64_t t_raw = targets[row];
  const bool valid = t_raw != ignore_index;
  const int t = static_cast<int>(t_raw < 0 ? 0 : (t_raw >= V ? V - 1 : t_raw));
  const float xt = tid == 0 ? to_f32(x[t]) : 0.f;
  if (lane == 0) { red_m[wave] = m; red_s[wave] = s; }
  __syncthreads();
  m = red_m[0];
  s = red_s[0];
#pragma unroll
  for (int w = 1; w < 4; ++w) lse_merge(m, s, red_m[w], red_s[w]);
  const float lse2 = m + __log2f(s);
  if (tid == 0) {
    loss[row] = valid ? (lse2 - xt * kLog2e) * kLn2 : 0.f;
    if (lse_out) lse_out[row] = lse2 * kLn2;
  }
  const float sc = valid ? *grad_scale : 0.f;
  T* g = grad + row * grs;
#pragma unroll
  for (int c = 0; c < NCH; ++c) {
    const int e = (c * 256 + tid) * E;
    if (e < V) {
      float v[E], o[E];
      chunk(c, v);
#pragma unroll
      for (int i = 0; i < E; ++i) {
        const float p = __builtin_amdgcn_exp2f(fmaf(v[i], kLog2e, -lse2));
        o[i] = (p - (e + i == t ? 1.f : 0.f)) * sc;
      }
      store16<T, true>(g + e, o);
    }
  }
}

// Row statistics of the planes kernels: log2-domain logsumexp over the
// workgroup of per-thread (m, s).
__device__ __forceinline__ float row_lse2(float m, float s, float (&red_m)[4], float (&red_s)[4]) {
#pragma unroll
  for (int off = 32; off > 0; off >>= 1) {
    const float m2 = __shfl_xor(m, off), s2 = __shfl_xor(s, off);
    lse_merge(m, s, m2, s2);
  }
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  if (lane == 0) { red_m[wave] = m; red_s[wave] = s; }
  __syncthreads();
  m = red_m[0];
  s = red_s[0];
#pragma unroll
  for (int w = 1; w < 4; ++w) lse_merge(m, s, red_m[w], red_s[w]);
  return m + __log2f(s);
}

template <int N>
__device__ __forceinline__ void chunk_stats(const float* v, float& m, float& s) {
  float cm = v[0] * kLog2e;
#pragma unroll
  for (int i = 1; i < N; ++i) cm = fmaxf(cm, v[i] * kLog2e);
  if (cm == -INFINITY) return;  // all -inf: adds nothing (and exp2(-inf + inf) is NaN)
  float cs = 0.f;
#pragma unroll
  for (int i = 0; i < N; ++i) cs += __builtin_amdgcn_exp2f(fmaf(v[i], kLog2e, -cm));
  lse_merge(m, s, cm, cs);
}

// What bf16 leaves of g; an infinity is whole without it.
__device__ __forceinline__ float plane_rest(float g, bf16 hi) {
  const float h = to_f32(hi);
  return fabsf(h) == INFINITY ? 0.f : g - h;
}

// Columns from V on hold nothing.
__device__ __forceinline__ void mask_tail(float* v, int e, int V) {
  if (e + 8 > V)
#pragma unroll
    for (int i = 0; i < 8; ++i) v[i] = e + i < V ? v[i] : -INFINITY;
}

// (softmax - onehot(t)) * scale of 8 logits at column e, as bf16 hi and
// residual vectors.
__device__ __forceinline__ void planes8(const float* v, int e, int t, float lse2, float sc, uint4& hi, uint4& lo) {
  float g[8], r[8];
#pragma unroll
  for (int i = 0; i < 8; ++i) {
    const float p = __builtin_amdgcn_exp2f(fmaf(v[i], kLog2e, -lse2));
    g[i] = (p - (e + i == t ? 1.f : 0.f)) * sc;
    r[i] = plane_rest(g[i], from_f32<bf16>(g[i]));
  }
  hi = pack16<bf16>(g);
  lo = pack16<bf16>(r);
}

struct PlanesArgs {
  const float* logits;
  int64_t rs;
  const int64_t* targets;
  uint16_t* planes;  // plane 0 (hi), then plane 1 at ps elements; rows grs apart
  int64_t grs, ps;
  const float* scale;
  int V;
  int64_t ignore_index;
};

// NCH > 0: the row stays in registers (V <= 2048 NCH, aligned rows of whole
// 8-column pieces), and the planes may take the logits' memory: every thread
// has read its columns before the barrier of row_lse2.  NCH = 0: read twice,
// VEC with 8 columns per thread, else one.
template <int NCH, bool VEC>
__global__ __launch_bounds__(256) void ce_planes_kernel(PlanesArgs a) {
  __shared__ float red_m[4], red_s[4];
  const int64_t row = blockIdx.x;
  const int tid = threadIdx.x, V = a.V;
  const float* x = a.logits + row * a.rs;
  uint16_t* hi = a.planes + row * a.grs;
  uint16_t* lo = hi + a.ps;
  const int64_t t_raw = a.targets[row];
  const bool valid = t_raw != a.ignore_index;
  const int t = static_cast<int>(t_raw < 0 ? 0 : (t_raw >= V ? V - 1 : t_raw));
  const float sc = valid ? *a.scale : 0.f;
  float m = -INFINITY, s = 0.f;
  if constexpr (NCH > 0) {
    uint4 raw[NCH][2];
#pragma unroll
    for (int c = 0; c < NCH; ++c) {
      const int e = (c * 256 + tid) * 8;
      if (e < V) {
        raw[c][0] = ld16raw<true>(x + e);
        raw[c][1] = ld16raw<true>(x + e + 4);
      }
    }
#pragma unroll
    for (int c = 0; c < NCH; ++c)
      if ((c * 256 + tid) * 8 < V) {
        float v[8];
        unpack16<float>(raw[c][0], v);
        unpack16<float>(raw[c][1], v + 4);
        mask_tail(v, (c * 256 + tid) * 8, V);
        chunk_stats<8>(v, m, s);
      }
    const float lse2 = row_lse2(m, s, red_m, red_s);
#pragma unroll
    for (int c = 0; c < NCH; ++c) {
      const int e = (c * 256 + tid) * 8;
      if (e < V) {
        float v[8];
        unpack16<float>(raw[c][0], v);
        unpack16<float>(raw[c][1], v + 4);
        mask_tail(v, e, V);
        uint4 h, l;
        planes8(v, e, t, lse2, sc, h, l);
        st16raw<true>(hi + e, h);
        st16raw<true>(lo + e, l);
      }
    }
  } else if constexpr (VEC) {
    for (int e = tid * 8; e < V; e += 256 * 8) {
      float v[8];
      load16<float>(x + e, v);
      load16<float>(x + e + 4, v + 4);
      chunk_stats<8>(v, m, s);
    }
    const float lse2 = row_lse2(m, s, red_m, red_s);
    for (int e = tid * 8; e < V; e += 256 * 8) {
      float v[8];
      load16<float>(x + e, v);
      load16<float>(x + e + 4, v + 4);
      uint4 h, l;
      planes8(v, e, t, lse2, sc, h, l);
      st16raw<true>(hi + e, h);
      st16raw<true>(lo + e, l);
    }
  } else {
    for (int e = tid; e < V; e += 256) chunk_stats<1>(x + e, m, s);
    const float lse2 = row_lse2(m, s, red_m, red_s);
    for (int e = tid; e < V; e += 256) {
      const float p = __builtin_amdgcn_exp2f(fmaf(x[e], kLog2e, -lse2));
      const float g = (p - (e == t ? 1.f : 0.f)) * sc;
      const bf16 h = from_f32<bf16>(g);
      hi[e] = h.bits;
      lo[e] = from_f32<bf16>(plane_rest(g, h)).bits;
    }
  }
}

template <typename T, bool GRAD>
int launch(const void* logits, int64_t rs, const int64_t* targets, float* loss, float* lse,
           void* grad, int64_t grs, const float* scale, int64_t rows, int V, int64_t ignore,
           hipStream_t st) {
  constexpr int E = 16 / int(sizeof(T));
  const bool vec = V % E == 0 && rs % E == 0 && aligned16(logits) &&
                   (!GRAD || (grs % E == 0 && aligned16(grad)));
  const dim3 grid(static_cast<unsigned>(rows));
  const T* x = static_cast<const T*>(logits);
  T* g = static_cast<T*>(grad);
  if constexpr (GRAD) {
    // Register-resident rows: up to 32 chunks of 16 bytes per thread.
    const int nch = (V / E + 255) / 256;
    if (vec && nch <= 32) {
#define HYDRA_CE_REG(N) \
  ce_rows_reg_kernel<T, N><<<grid, 256, 0, st>>>(x, rs, targets, loss, lse, g, grs, scale, V, ignore)
      if (nch <= 8) HYDRA_CE_REG(8);
      else if (nch <= 16) HYDRA_CE_REG(16);
      else HYDRA_CE_REG(32);
#undef HYDRA_CE_REG
      return check_launch("ce_rows");
    }
  }
  if (vec)
    ce_rows_kernel<T, true, GRAD><<<grid, 256, 0, st>>>(x, rs, targets, loss, lse, g, grs, scale, V, ignore);
  else
    ce_rows_kernel<T, false, GRAD><<<grid, 256, 0, st>>>(x, rs, targets, loss, lse, g, grs, scale, V, ignore);
  return check_launch("ce_rows");
}

}  // namespace
}  // namespace hydra

using namespace hydra;

extern "C" int hydra_ce_rows(const void* logits, int64_t rows, int64_t vocab, int64_t logits_rs,
                             const int64_t* targets, int64_t ignore_index, float* loss,
                             float* lse, void* grad, int64_t grad_rs, const float* grad_scale,
                             int dtype, void* stream) {
  HYDRA_REQUIRE(rows >= 0 && vocab >= 1, "ce_rows: bad size");
  HYDRA_REQUIRE(vocab < (int64_t(1) << 31) && rows < (int64_t(1) << 31), "ce_rows: too large");
  HYDRA_REQUIRE(logits_rs >= vocab && (!grad || grad_rs >= vocab), "ce_rows: row stride < vocab");
  HYDRA_REQUIRE(dtype == HYDRA_F32 || dtype == HYDRA_BF16 || dtype == HYDRA_F16,
                "ce_rows: unknown dtype");
  if (rows == 0) return HYDRA_OK;
  HYDRA_REQUIRE(logits && targets && loss, "ce_rows: null pointer");
  HYDRA_REQUIRE(!grad || grad_scale, "ce_rows: the gradient needs grad_scale");
  auto st = static_cast<hipStream_t>(stream);
  const int V = static_cast<int>(vocab);
#define HYDRA_CE(T)                                                                                  \
  return grad ? launch<T, true>(logits, logits_rs, targets, loss, lse, grad, grad_rs, grad_scale,   \
                                rows, V, ignore_index, st)                                          \
              : launch<T, false>(logits, logits_rs, targets, loss, lse, grad, grad_rs, grad_scale,  \
                                 rows, V, ignore_index, st)
  switch (dtype) {
    case HYDRA_F32: HYDRA_CE(float);
    case HYDRA_BF16: HYDRA_CE(bf16);
    default: HYDRA_CE(f16);
  }
#undef HYDRA_CE
}

extern "C" int hydra_ce_grad_planes(const float* logits, int64_t rows, int64_t vocab, int64_t logits_rs,
                                    const int64_t* targets, int64_t ignore_index, void* planes,
                                    int64_t planes_rs, int64_t plane_stride, const float* grad_scale,
                                    void* stream) {
  HYDRA_REQUIRE(rows >= 0 && vocab >= 1, "ce_grad_planes: bad size");
  HYDRA_REQUIRE(vocab < (int64_t(1) << 31) && rows < (int64_t(1) << 31), "ce_grad_planes: too large");
  HYDRA_REQUIRE(logits_rs >= vocab && planes_rs >= vocab, "ce_grad_planes: row stride < vocab");
  const bool in_place = planes == logits;
  if (in_place)
    HYDRA_REQUIRE(planes_rs == 2 * logits_rs && plane_stride == logits_rs,
                  "ce_grad_planes: in place, a row's planes take the two halves of its bytes");
  else
    HYDRA_REQUIRE(rows <= 1 || plane_stride >= (rows - 1) * planes_rs + vocab, "ce_grad_planes: planes overlap");
  if (rows == 0) return HYDRA_OK;
  HYDRA_REQUIRE(logits && targets && planes && grad_scale, "ce_grad_planes: null pointer");
  const int V = static_cast<int>(vocab);
  const PlanesArgs a{logits, logits_rs, targets, static_cast<uint16_t*>(planes), planes_rs, plane_stride,
                     grad_scale, V, ignore_index};
  // In place the padding of a row up to 8 columns is the row's own.
  const bool vec = (V % 8 == 0 || (in_place && logits_rs >= (vocab + 7) / 8 * 8)) && logits_rs % 4 == 0 &&
                   planes_rs % 8 == 0 && plane_stride % 8 == 0 && aligned16(logits) && aligned16(planes);
  const dim3 grid(static_cast<unsigned>(rows));
  auto st = static_cast<hipStream_t>(stream);
  const int64_t nch = ((vocab + 7) / 8 + 255) / 256;
  if (in_place && (!vec || vocab > HYDRA_CE_IN_PLACE_VOCAB))
    return fail(HYDRA_ERR_UNSUPPORTED, "ce_grad_planes: in place takes aligned rows of up to 32768 columns");
  static_assert(HYDRA_CE_IN_PLACE_VOCAB == 16 * 256 * 8, "the longest rows that stay in registers");
  if (!vec) ce_planes_kernel<0, false><<<grid, 256, 0, st>>>(a);
  else if (nch <= 4) ce_planes_kernel<4, true><<<grid, 256, 0, st>>>(a);
  else if (nch <= 8) ce_planes_kernel<8, true><<<grid, 256, 0, st>>>(a);
  else if (nch <= 16) ce_planes_kernel<16, true><<<grid, 256, 0, st>>>(a);
  else ce_planes_kernel<0, true><<<grid, 256, 0, st>>>(a);
  return check_launch("ce_grad_planes");
}
