// Whole backward of the CCGQA q/k/v preparation in bf16 (hydra_ccgqa_prep_bwd_conv):
// conv pair recomputation, the pointwise chain, and the gradients of both
// convs' inputs and weights (reference: attention.py:205-266 and
// kernels/fused_conv.py:39-62, trained through autograd there).
//
// With x0 = the q (or k) columns of qkv, y2 = conv2(conv1(x0)) and dy2 the
// gradient of y2 from the pointwise chain:
//   pack      the conv weights as 64x64 channel blocks, taps together, in both
//             directions (zeros outside a group), so that staging is a copy
//   conv x2   y1 = conv1(x0), y2 = conv2(y1)
//   pointwise launch_prep_bwd (ccgqa_prep_bwd.hip): dy2, the QK-mean and v
//             parts of grad(qkv), temperature partials per token
//   conv x2   dy1 = conv2^T(dy2), grad(x0) += conv1^T(dy1)
//   wgrad     all four weight gradients, and their reduction
// q and k go through every launch together.
//
// The convs are implicit GEMMs on v_mfma_f32_32x32x16_bf16: a tile of 128
// tokens (two halo rows) by 64 input channels sits in LDS once and serves the
// three taps at three row offsets, where the im2col form writes and reads
// every input three times.  The weight gradients contract over tokens: both
// operands are staged row-major and read as MFMA fragments by the transposing
// LDS read (ds_read_tr16_b64), tap t being a row offset of the input tile;
// token ranges are split over workgroups and summed in order.  What bounds
// them is the launch: at 4096 tokens x 512 + 128 channels (8 GFLOP per dense
// conv) there are 160-640 workgroups of a few microseconds each, so everything
// that used to be a launch of its own (im2col, col2im, transposing copies,
// ~45 launches in all) is part of one of eight.
//
// Measured at B4 x S1024, dim 2048, 8/2 heads x 64 (kernel trace): pack 6 us
// (12 with one packed piece per thread), y1 7 and y2 14 (26 with the staged
// pieces in scratch memory and four waves), pointwise 17 (34 as one token per
// wave), dy1 14, grad(x0) 9, weight gradients 22 + 11; the composed form took
// ~430 us of kernels in ~45 launches.  Whole layer steps: that shape 1.32 ->
// 0.78 ms, padded B8 x S777 4/1 x 64 1.41 -> 0.85, 28/4 heads x 16 at B2 x
// S2048 1.40 -> 0.87 (bound by the host's launches now).
#include "ccgqa_prep_bwd.h"
#include "common.h"

#include <algorithm>

namespace hydra {
namespace {

typedef __attribute__((ext_vector_type(8))) __bf16 bf16x8_t;
typedef __attribute__((ext_vector_type(16))) float f32x16_t;
typedef __attribute__((ext_vector_type(4))) short s16x4_t;

constexpr int kBlk = 64;                        // channels per block
constexpr int kTaps = 3;
constexpr int kWBlk = kTaps * kBlk * kBlk;      // one packed weight block
constexpr int kPitch = kBlk + 8;                // LDS row pitch (elements): 16-byte rows, 4-bank skew
constexpr int kTM = 128;                        // tokens per conv tile
constexpr int kConvThreads = 512;
constexpr int kWT = 64;                         // tokens per weight-gradient step

__device__ __forceinline__ f32x16_t mfma(uint4 a, uint4 b, f32x16_t c) {
  return __builtin_amdgcn_mfma_f32_32x32x16_bf16(__builtin_bit_cast(bf16x8_t, a),
                                                 __builtin_bit_cast(bf16x8_t, b), c, 0, 0, 0);
}
__device__ __forceinline__ f32x16_t zero16() {
  f32x16_t z;
#pragma unroll
  for (int r = 0; r < 16; ++r) z[r] = 0.f;
  return z;
}

// The 64-channel blocks of a conv with C channels in groups of cg: output
// block ob reads input blocks first(ob) .. first(ob) + span - 1.
struct Blocks {
  int C, cg, n, span, dense;
  __host__ __device__ int first(int ob) const { return dense ? 0 : ob / span * span; }
};
Blocks blocks_of(int C, int cg) {
  Blocks b{C, cg, (C + kBlk - 1) / kBlk, 1, cg == C ? 1 : 0};
  b.span = b.dense ? b.n : cg <= kBlk ? 1 : cg / kBlk;
  return b;
}

// ------------------------------------------------------------------- pack
// out[ob][ib][t][o][i]: weight from input channel i to output channel o at tap
// t; transposed: the roles of the conv's channels exchanged.
struct PackJob {
  const bf16* w;  // [C][cg][3]
  uint16_t* out;
  Blocks b;
  int transposed;
  int first;      // its first piece (8 input channels of an output channel)
};
struct PackArgs {
  PackJob job[8];
  int pieces;
};

// A thread takes 8 input channels of one output channel, all taps: forward its
// 24 source values are one run (neighbouring threads: neighbouring runs);
// transposed they lie in 8 source rows, and neighbouring threads take
// neighbouring output channels, so that each row is still read in order.
__global__ __launch_bounds__(256) void conv_pack_kernel(PackArgs a) {
  const int p = blockIdx.x * 256 + threadIdx.x;
  if (p >= a.pieces) return;
  int j = 0;
#pragma unroll
  for (int k = 1; k < 8; ++k) j = p >= a.job[k].first ? k : j;
  const PackJob& q = a.job[j];
  const int e = p - q.first, blk = e / (kBlk * kBlk / 8), rem = e % (kBlk * kBlk / 8);
  const int o = q.transposed ? rem % kBlk : rem / 8, i = 8 * (q.transposed ? rem / kBlk : rem % 8);
  const int ob = blk / q.b.span, ib = q.b.first(ob) + blk % q.b.span;
  const int oc = kBlk * ob + o, ic = kBlk * ib + i;
  uint32_t v[kTaps][8];
  const bool ok = oc < q.b.C && ic < q.b.C && oc / q.b.cg == ic / q.b.cg;  // all 8: groups are of 8 k channels
  if (!ok) {
#pragma unroll
    for (int t = 0; t < kTaps; ++t)
#pragma unroll
      for (int u = 0; u < 8; ++u) v[t][u] = 0;
  } else {
    const int row = q.transposed ? ic : oc, col = (q.transposed ? oc : ic) % q.b.cg;
    const int64_t step = q.transposed ? static_cast<int64_t>(q.b.cg) * kTaps : kTaps;
    const bf16* w = q.w + (static_cast<int64_t>(row) * q.b.cg + col) * kTaps;
#pragma unroll
    for (int u = 0; u < 8; ++u)
#pragma unroll
      for (int t = 0; t < kTaps; ++t) v[t][u] = w[u * step + t].bits;
  }
  uint16_t* out = q.out + static_cast<int64_t>(blk) * kWBlk + o * kBlk + i;
#pragma unroll
  for (int t = 0; t < kTaps; ++t)
    *reinterpret_cast<uint4*>(out + t * kBlk * kBlk) =
        make_uint4(v[t][0] | v[t][1] << 16, v[t][2] | v[t][3] << 16, v[t][4] | v[t][5] << 16, v[t][6] | v[t][7] << 16);
}

// ------------------------------------------------------------------- conv
struct ConvJob {
  const uint16_t* x;  // input rows, xrs apart
  uint16_t* y;        // output rows, yrs apart
  const uint16_t* w;  // packed
  int64_t xrs, yrs;
  Blocks b;
  int first;          // its first workgroup
};
struct ConvArgs {
  ConvJob job[2];
  int S, tiles, ntiles;  // token tiles per sequence, over all sequences
};

// job[second], value by value (an indexed access, or a conditional that names
// the fields, would go through a copy in scratch memory).
template <typename V>
__device__ __forceinline__ V pick(bool second, V q, V p) {
  return second ? q : p;
}
__device__ __forceinline__ ConvJob conv_job(const ConvArgs& a, bool second) {
  const ConvJob &p = a.job[0], &q = a.job[1];
  ConvJob j;
  j.x = pick(second, q.x, p.x);
  j.y = pick(second, q.y, p.y);
  j.w = pick(second, q.w, p.w);
  j.xrs = pick(second, q.xrs, p.xrs);
  j.yrs = pick(second, q.yrs, p.yrs);
  j.b.C = pick(second, q.b.C, p.b.C);
  j.b.cg = pick(second, q.b.cg, p.b.cg);
  j.b.n = pick(second, q.b.n, p.b.n);
  j.b.span = pick(second, q.b.span, p.b.span);
  j.b.dense = pick(second, q.b.dense, p.b.dense);
  j.first = pick(second, q.first, p.first);
  return j;
}

// BACK: tap t reads token s + 2 - t (a conv's transpose), else s - (2 - t).
// ACC: adds to the output rows.
// Eight waves, each 32 tokens x 32 output channels: two per SIMD, which hides
// the LDS and L2 latency of a grid of about one workgroup per CU better than
// four waves of 32 x 64 did (the reads per product go from 1.5 to 2 fragments).
template <bool BACK, bool ACC>
__global__ __launch_bounds__(kConvThreads) void conv_kernel(ConvArgs a) {
  constexpr int NT = kConvThreads;
  constexpr int XR = kTM + kTaps - 1;                          // staged token rows
  constexpr int XU = (XR * (kBlk / 8) + NT - 1) / NT;          // 16-byte pieces per thread
  constexpr int WU = kWBlk / 8 / NT;
  __shared__ __attribute__((aligned(16))) uint16_t xs[XR * kPitch], ws[kTaps * kBlk * kPitch];
  const ConvJob q = conv_job(a, static_cast<int>(blockIdx.x) >= a.job[1].first);
  const int idx = blockIdx.x - q.first;
  // tiles fastest: with a multiple of 8 of them, one tile's input rows stay in
  // one XCD's L2 for all output blocks
  const int tile = idx % a.ntiles, ob = idx / a.ntiles;
  const int b = tile / a.tiles, s0 = kTM * (tile - b * a.tiles);
  const int tid = threadIdx.x, lane = tid & 63, n = lane & 31, hf = lane >> 5;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int wt = 32 * (wave & 3), wc = 32 * (wave >> 2);  // this wave's tokens and channels
  const int ib0 = q.b.first(ob);
  const uint16_t* x = q.x + static_cast<int64_t>(b) * a.S * q.xrs;
  uint4 rx[XU], rw[WU];
  auto fetch = [&](int it) {
    const int c0 = kBlk * (ib0 + it);
#pragma unroll
    for (int u = 0; u < XU; ++u) {
      const int i = tid + NT * u, row = i >> 3, c = c0 + 8 * (i & 7);
      const int s = s0 + row - (BACK ? 0 : kTaps - 1);
      rx[u] = make_uint4(0, 0, 0, 0);
      if (row < XR && s >= 0 && s < a.S && c < q.b.C) rx[u] = ld16raw<false>(x + s * q.xrs + c);
    }
    const uint16_t* w = q.w + static_cast<int64_t>(ob * q.b.span + it) * kWBlk;
#pragma unroll
    for (int u = 0; u < WU; ++u) rw[u] = ld16raw<false>(w + 8 * (tid + NT * u));
  };
  f32x16_t acc = zero16();
  fetch(0);
  for (int it = 0; it < q.b.span; ++it) {
    if (it) __syncthreads();  // the previous tile's readers are done
#pragma unroll
    for (int u = 0; u < XU; ++u) {
      const int i = tid + NT * u, row = i >> 3;
      if (row < XR) *reinterpret_cast<uint4*>(&xs[row * kPitch + 8 * (i & 7)]) = rx[u];
    }
#pragma unroll
    for (int u = 0; u < WU; ++u) {
      const int i = tid + NT * u;
      *reinterpret_cast<uint4*>(&ws[(i >> 3) * kPitch + 8 * (i & 7)]) = rw[u];
    }
    __syncthreads();
    if (it + 1 < q.b.span) fetch(it + 1);
#pragma unroll
    for (int ks = 0; ks < kBlk / 16; ++ks)
#pragma unroll
      for (int t = 0; t < kTaps; ++t) {
        const int xrow = wt + n + (BACK ? kTaps - 1 - t : t);
        const uint4 xf = *reinterpret_cast<const uint4*>(&xs[xrow * kPitch + 16 * ks + 8 * hf]);
        const uint4 wf = *reinterpret_cast<const uint4*>(&ws[(kBlk * t + wc + n) * kPitch + 16 * ks + 8 * hf]);
        acc = mfma(wf, xf, acc);
      }
  }
  // a lane holds one token's channels, four consecutive ones per register group
  const int s = s0 + wt + n;
  if (s >= a.S) return;
  uint16_t* y = q.y + (static_cast<int64_t>(b) * a.S + s) * q.yrs;
#pragma unroll
  for (int j = 0; j < 4; ++j) {
    const int c = kBlk * ob + wc + 8 * j + 4 * hf;
    if (c >= q.b.C) continue;
    float f[4];
#pragma unroll
    for (int r = 0; r < 4; ++r) f[r] = acc[4 * j + r];
    uint2* dst = reinterpret_cast<uint2*>(y + c);
    if constexpr (ACC) {
      const uint2 old = *dst;
      f[0] += __uint_as_float(old.x << 16);
      f[1] += __uint_as_float(old.x & 0xffff0000u);
      f[2] += __uint_as_float(old.y << 16);
      f[3] += __uint_as_float(old.y & 0xffff0000u);
    }
    *dst = make_uint2(pack2<bf16>(f[0], f[1]), pack2<bf16>(f[2], f[3]));
  }
}

// ------------------------------------------------------- weight gradients
struct WgradJob {
  const uint16_t *dy, *x;  // dW[o][i][t] = sum_s dy[s][o] x[s - (2 - t)][i]
  int64_t dyrs, xrs;
  bf16* dw;                // [C][cg][3]
  Blocks b;
  int first;               // its first (output block, input block) pair
};
struct WgradArgs {
  WgradJob job[4];
  int S, tiles, ntiles, pairs, splits;
  float* part;             // [splits][pairs][3][64][64]
};

__device__ __forceinline__ const WgradJob& wgrad_job(const WgradArgs& a, int pair) {
  int j = 0;
#pragma unroll
  for (int k = 1; k < 4; ++k) j = pair >= a.job[k].first ? k : j;
  return a.job[j];
}

// MFMA fragment (32 columns from m0, 16 summed rows from k0) of a row-major
// LDS tile: within each 16 lanes the transposing read takes 4 rows of 16
// columns (lane i: row i / 4, columns 4 (i % 4) ..) and returns column i's
// four rows, so two reads give a lane its eight summed values.
__device__ __forceinline__ uint4 tr_frag(const uint16_t* tile, int k0, int m0, int lane) {
  const uint16_t* p = tile + (k0 + 8 * (lane >> 5) + ((lane & 15) >> 2)) * kPitch + m0 + 16 * ((lane >> 4) & 1) +
                      4 * (lane & 3);
  typedef __attribute__((address_space(3))) s16x4_t* lds_t;
  const s16x4_t lo = __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_t)(p));
  const s16x4_t hi = __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_t)(p + 4 * kPitch));
  const uint2 l = __builtin_bit_cast(uint2, lo), h = __builtin_bit_cast(uint2, hi);
  return make_uint4(l.x, l.y, h.x, h.y);
}

__global__ __launch_bounds__(256) void conv_wgrad_kernel(WgradArgs a) {
  constexpr int XR = kWT + kTaps - 1;
  constexpr int DU = kWT * (kBlk / 8) / 256, XU = (XR * (kBlk / 8) + 255) / 256;
  __shared__ __attribute__((aligned(16))) uint16_t ds[kWT * kPitch], xs[XR * kPitch];
  const int pair = blockIdx.x % a.pairs, sp = blockIdx.x / a.pairs;
  const WgradJob& q = wgrad_job(a, pair);
  const int local = pair - q.first, ob = local / q.b.span, ib = q.b.first(ob) + local % q.b.span;
  const int tid = threadIdx.x, lane = tid & 63, n = lane & 31, hf = lane >> 5;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int wo = 32 * (wave & 1), wi = 32 * (wave >> 1);  // this wave's quarter of the block
  const int begin = static_cast<int>(static_cast<int64_t>(a.ntiles) * sp / a.splits);
  const int end = static_cast<int>(static_cast<int64_t>(a.ntiles) * (sp + 1) / a.splits);
  uint4 rd[DU], rx[XU];
  auto fetch = [&](int tile) {
    const int b = tile / a.tiles, s0 = kWT * (tile - b * a.tiles);
    const uint16_t* dy = q.dy + static_cast<int64_t>(b) * a.S * q.dyrs;
    const uint16_t* x = q.x + static_cast<int64_t>(b) * a.S * q.xrs;
#pragma unroll
    for (int u = 0; u < DU; ++u) {
      const int i = tid + 256 * u, s = s0 + (i >> 3), c = kBlk * ob + 8 * (i & 7);
      rd[u] = s < a.S && c < q.b.C ? *reinterpret_cast<const uint4*>(dy + s * q.dyrs + c) : make_uint4(0, 0, 0, 0);
    }
#pragma unroll
    for (int u = 0; u < XU; ++u) {
      const int i = tid + 256 * u, row = i >> 3, s = s0 + row - (kTaps - 1), c = kBlk * ib + 8 * (i & 7);
      rx[u] = row < XR && s >= 0 && s < a.S && c < q.b.C ? *reinterpret_cast<const uint4*>(x + s * q.xrs + c)
                                                          : make_uint4(0, 0, 0, 0);
    }
  };
  f32x16_t acc[kTaps];
#pragma unroll
  for (int t = 0; t < kTaps; ++t) acc[t] = zero16();
  if (begin < end) fetch(begin);
  for (int tile = begin; tile < end; ++tile) {
    __syncthreads();  // the previous tile's readers are done
#pragma unroll
    for (int u = 0; u < DU; ++u) {
      const int i = tid + 256 * u;
      *reinterpret_cast<uint4*>(&ds[(i >> 3) * kPitch + 8 * (i & 7)]) = rd[u];
    }
#pragma unroll
    for (int u = 0; u < XU; ++u) {
      const int i = tid + 256 * u, row = i >> 3;
      if (row < XR) *reinterpret_cast<uint4*>(&xs[row * kPitch + 8 * (i & 7)]) = rx[u];
    }
    __syncthreads();
    if (tile + 1 < end) fetch(tile + 1);
#pragma unroll
    for (int k0 = 0; k0 < kWT; k0 += 16) {
      const uint4 df = tr_frag(ds, k0, wo, lane);
#pragma unroll
      for (int t = 0; t < kTaps; ++t) acc[t] = mfma(df, tr_frag(xs, k0 + t, wi, lane), acc[t]);
    }
  }
  float* part = a.part + (static_cast<int64_t>(sp) * a.pairs + pair) * kWBlk;
#pragma unroll
  for (int t = 0; t < kTaps; ++t)
#pragma unroll
    for (int r = 0; r < 16; ++r)
      part[t * kBlk * kBlk + (wo + 8 * (r >> 2) + 4 * hf + (r & 3)) * kBlk + wi + n] = acc[t][r];
}

// The splits' partials in order -> the weight gradients; the last workgroup
// sums the temperature's per-token partials.
__global__ __launch_bounds__(256) void conv_wgrad_reduce_kernel(WgradArgs a, const float* __restrict__ dtemp_tok,
                                                                bf16* __restrict__ dtemp, int64_t tokens) {
  const int64_t e = static_cast<int64_t>(blockIdx.x) * 256 + threadIdx.x;
  const int pair = static_cast<int>(e / (kBlk * kBlk)), rem = static_cast<int>(e % (kBlk * kBlk));
  if (pair >= a.pairs) {
    if (dtemp == nullptr) return;
    __shared__ float red[4];
    float s = 0.f;
    for (int64_t i = threadIdx.x; i < tokens; i += 256) s += dtemp_tok[i];
    s = wave_sum(s);
    if ((threadIdx.x & 63) == 0) red[threadIdx.x >> 6] = s;
    __syncthreads();
    if (threadIdx.x == 0) *dtemp = from_f32<bf16>(red[0] + red[1] + red[2] + red[3]);
    return;
  }
  const WgradJob& q = wgrad_job(a, pair);
  const int local = pair - q.first, ob = local / q.b.span, ib = q.b.first(ob) + local % q.b.span;
  const int oc = kBlk * ob + rem / kBlk, ic = kBlk * ib + rem % kBlk;
  if (oc >= q.b.C || ic >= q.b.C || oc / q.b.cg != ic / q.b.cg) return;
  const float* p = a.part + static_cast<int64_t>(pair) * kWBlk + rem;
  const int64_t step = static_cast<int64_t>(a.pairs) * kWBlk;
  float s[kTaps] = {0.f, 0.f, 0.f};
#pragma unroll 4
  for (int sp = 0; sp < a.splits; ++sp)
#pragma unroll
    for (int t = 0; t < kTaps; ++t) s[t] += p[sp * step + t * kBlk * kBlk];
  bf16* out = q.dw + (static_cast<int64_t>(oc) * q.b.cg + ic % q.b.cg) * kTaps;
#pragma unroll
  for (int t = 0; t < kTaps; ++t) out[t] = from_f32<bf16>(s[t]);
}

// --------------------------------------------------------------- the plan
// Workspace: packed weights (q1, q2, k1, k2 forward, then transposed), four
// [tokens, L + K] bf16 buffers (y1, y2, dy2, dy1), the weight gradients'
// partials, the temperature's partials per token.
struct Plan {
  Blocks b[4];            // q1, q2, k1, k2
  int64_t pack[8], act, part, dtemp, bytes;
  int pairs, splits, wtiles;
};

constexpr int64_t up256(int64_t n) { return (n + 255) & ~int64_t(255); }

// The sizes this path takes (the caller has the general one otherwise).
bool supported(int64_t B, int64_t S, int64_t Hq, int64_t Hkv, int64_t hd, int64_t ks, int flags, int dtype) {
  const int64_t L = Hq * hd, K = Hkv * hd;
  return dtype == HYDRA_BF16 && ks == kTaps && (flags & HYDRA_CCGQA_CONVS) &&
         (hd == 8 || hd == 16 || hd == 32 || hd == 64 || hd == 128) && K % 16 == 0 && L + K <= 2048 &&
         B >= 1 && S >= 1 && B * S < (int64_t(1) << 24);
}

Plan plan_of(int64_t B, int64_t S, int64_t Hq, int64_t Hkv, int64_t hd) {
  Plan p{};
  const int L = static_cast<int>(Hq * hd), K = static_cast<int>(Hkv * hd), h = static_cast<int>(hd);
  p.b[0] = blocks_of(L, h);
  p.b[1] = blocks_of(L, L);
  p.b[2] = blocks_of(K, h);
  p.b[3] = blocks_of(K, K);
  int64_t at = 0;
  for (int i = 0; i < 8; ++i) {
    p.pack[i] = at;
    at += up256(int64_t(p.b[i & 3].n) * p.b[i & 3].span * kWBlk * 2);
  }
  p.act = at;
  at += 4 * up256(B * S * (L + K) * 2);
  for (const Blocks& b : p.b) p.pairs += b.n * b.span;
  p.wtiles = static_cast<int>((S + kWT - 1) / kWT);
  // about four workgroups per CU, and at least four token tiles in each (a
  // split writes and re-reads 48 KB per pair)
  const int64_t nt = B * p.wtiles;
  p.splits = static_cast<int>(std::max<int64_t>(
      1, std::min<int64_t>(nt / 4, (4 * int64_t(device_cus()) + p.pairs - 1) / p.pairs)));
  p.part = at;
  at += up256(int64_t(p.splits) * p.pairs * kWBlk * 4);
  p.dtemp = at;
  at += up256(B * S * 4);
  p.bytes = at;
  return p;
}

template <bool BACK, bool ACC>
int launch_conv(const ConvJob& jq, const ConvJob& jk, int64_t B, int64_t S, hipStream_t st) {
  ConvArgs a{};
  a.job[0] = jq;
  a.job[1] = jk;
  a.S = static_cast<int>(S);
  a.tiles = static_cast<int>((S + kTM - 1) / kTM);
  a.ntiles = static_cast<int>(B) * a.tiles;
  a.job[0].first = 0;
  a.job[1].first = jq.b.n * a.ntiles;
  conv_kernel<BACK, ACC><<<dim3(static_cast<unsigned>((jq.b.n + jk.b.n) * a.ntiles)), kConvThreads, 0, st>>>(a);
  return check_launch("ccgqa_conv_bwd: conv");
}

}  // namespace
}  // namespace hydra

using namespace hydra;

extern "C" int64_t hydra_ccgqa_prep_bwd_conv_workspace(int64_t B, int64_t S, int64_t Hq, int64_t Hkv, int64_t hd,
                                                       int64_t ks, int flags, int dtype) {
  if (Hq < 1 || Hkv < 1 || Hq % Hkv != 0 || !supported(B, S, Hq, Hkv, hd, ks, flags, dtype)) return -1;
  return plan_of(B, S, Hq, Hkv, hd).bytes;
}

extern "C" int hydra_ccgqa_prep_bwd_conv(const void* qkv, int64_t qkv_rs, const void* wq1, const void* wq2,
                                         const void* wk1, const void* wk2, const void* temp, const float* cos,
                                         const float* sin, int64_t cs_rs, const void* dq, const void* dk,
                                         const void* dv, void* dqkv, int64_t dqkv_rs, void* dwq1, void* dwq2,
                                         void* dwk1, void* dwk2, void* dtemp, int64_t B, int64_t S, int64_t Hq,
                                         int64_t Hkv, int64_t hd, int64_t ks, int flags, int dtype,
                                         void* workspace, int64_t workspace_bytes, void* stream) {
  HYDRA_REQUIRE(Hq >= 1 && Hkv >= 1 && Hq % Hkv == 0, "ccgqa_prep_bwd_conv: bad head counts");
  if (!supported(B, S, Hq, Hkv, hd, ks, flags, dtype))
    return fail(HYDRA_ERR_UNSUPPORTED, "ccgqa_prep_bwd_conv: sizes or type not taken");
  const int64_t L = Hq * hd, K = Hkv * hd, CW = L + K;
  HYDRA_REQUIRE((flags & ~(127 | HYDRA_CCGQA_ROPE_BF16)) == 0 && !(flags & HYDRA_CCGQA_V_TRANSPOSED), "ccgqa_prep_bwd_conv: bad flags");
  HYDRA_REQUIRE(qkv && wq1 && wq2 && wk1 && wk2 && dq && dk && dv && dqkv && dwq1 && dwq2 && dwk1 && dwk2,
                "ccgqa_prep_bwd_conv: null pointer");
  HYDRA_REQUIRE(qkv_rs >= CW + K && dqkv_rs >= CW + K, "ccgqa_prep_bwd_conv: row stride smaller than L + 2K");
  HYDRA_REQUIRE(!(flags & HYDRA_CCGQA_QK_NORM) || temp, "ccgqa_prep_bwd_conv: temperature required");
  HYDRA_REQUIRE(!(flags & HYDRA_CCGQA_ROPE) || (cos && sin && cs_rs >= hd / 2),
                "ccgqa_prep_bwd_conv: cos/sin [S, hd/2] required");
  if (qkv_rs % 8 != 0 || dqkv_rs % 8 != 0 || !aligned16(qkv) || !aligned16(dqkv) || !aligned16(dq) ||
      !aligned16(dk) || !aligned16(dv) || !aligned16(workspace))
    return fail(HYDRA_ERR_UNSUPPORTED, "ccgqa_prep_bwd_conv: unaligned rows");
  const Plan p = plan_of(B, S, Hq, Hkv, hd);
  if (workspace == nullptr || workspace_bytes < p.bytes)
    return fail(HYDRA_ERR_ARG, "ccgqa_prep_bwd_conv: workspace of " + std::to_string(p.bytes) + " bytes required");
  auto st = static_cast<hipStream_t>(stream);
  char* ws = static_cast<char*>(workspace);
  const bf16* w[4] = {static_cast<const bf16*>(wq1), static_cast<const bf16*>(wq2), static_cast<const bf16*>(wk1),
                      static_cast<const bf16*>(wk2)};
  PackArgs pk{};
  for (int i = 0; i < 8; ++i) {
    pk.job[i] = PackJob{w[i & 3], reinterpret_cast<uint16_t*>(ws + p.pack[i]), p.b[i & 3], i >> 2, pk.pieces};
    pk.pieces += p.b[i & 3].n * p.b[i & 3].span * (kBlk * kBlk / 8);
  }
  conv_pack_kernel<<<dim3(static_cast<unsigned>((pk.pieces + 255) / 256)), 256, 0, st>>>(pk);
  if (int rc = check_launch("ccgqa_conv_bwd: pack")) return rc;

  const int64_t act = up256(B * S * CW * 2);
  auto buf = [&](int i) { return reinterpret_cast<uint16_t*>(ws + p.act + i * act); };
  uint16_t *y1 = buf(0), *y2 = buf(1), *dy2 = buf(2), *dy1 = buf(3);
  auto x0 = static_cast<const uint16_t*>(qkv);
  auto dx = static_cast<uint16_t*>(dqkv);
  float* dtok = reinterpret_cast<float*>(ws + p.dtemp);
  // job of side 0 (q) or 1 (k): conv 1 or 2, packed forward or transposed
  auto job = [&](int side, int conv, bool back, const uint16_t* x, int64_t xrs, uint16_t* y, int64_t yrs) {
    const int i = 2 * side + conv - 1;
    return ConvJob{x + side * L, y + side * L, pk.job[i + (back ? 4 : 0)].out, xrs, yrs, p.b[i], 0};
  };
  if (int rc = launch_conv<false, false>(job(0, 1, false, x0, qkv_rs, y1, CW), job(1, 1, false, x0, qkv_rs, y1, CW), B,
                                         S, st))
    return rc;
  if (int rc = launch_conv<false, false>(job(0, 2, false, y1, CW, y2, CW), job(1, 2, false, y1, CW, y2, CW), B, S, st))
    return rc;
  const PrepBwdArgs pb{qkv, qkv_rs, y2, y2 + L, S * CW, S * CW, hd, CW, temp, cos, sin, cs_rs, dq, dk, dv, dy2, dqkv, dqkv_rs,
                       dtok, static_cast<int>(B), static_cast<int>(S), static_cast<int>(Hq), static_cast<int>(Hkv),
                       static_cast<int>(hd), flags, dtype, st};
  if (int rc = launch_prep_bwd(pb)) return rc;
  if (int rc = launch_conv<true, false>(job(0, 2, true, dy2, CW, dy1, CW), job(1, 2, true, dy2, CW, dy1, CW), B, S, st))
    return rc;
  if (int rc = launch_conv<true, true>(job(0, 1, true, dy1, CW, dx, dqkv_rs), job(1, 1, true, dy1, CW, dx, dqkv_rs), B,
                                       S, st))
    return rc;
  WgradArgs wg{};
  void* dws[4] = {dwq1, dwq2, dwk1, dwk2};
  for (int i = 0; i < 4; ++i) {
    const int64_t off = (i >> 1) * L;
    const bool second = i & 1;
    wg.job[i] = WgradJob{(second ? dy2 : dy1) + off, second ? y1 + off : x0 + off, CW, second ? CW : qkv_rs,
                         static_cast<bf16*>(dws[i]), p.b[i], wg.pairs};
    wg.pairs += p.b[i].n * p.b[i].span;
  }
  wg.S = static_cast<int>(S);
  wg.tiles = p.wtiles;
  wg.ntiles = static_cast<int>(B) * p.wtiles;
  wg.splits = p.splits;
  wg.part = reinterpret_cast<float*>(ws + p.part);
  conv_wgrad_kernel<<<dim3(static_cast<unsigned>(wg.pairs * wg.splits)), 256, 0, st>>>(wg);
  if (int rc = check_launch("ccgqa_conv_bwd: weight gradients")) return rc;
  const bool temp_grad = dtemp != nullptr && (flags & HYDRA_CCGQA_QK_NORM);
  conv_wgrad_reduce_kernel<<<dim3(static_cast<unsigned>(wg.pairs * (kBlk * kBlk / 256) + (temp_grad ? 1 : 0))), 256, 0,
                             st>>>(wg, dtok, temp_grad ? static_cast<bf16*>(dtemp) : nullptr, B * S);
  return check_launch("ccgqa_conv_bwd: weight gradient sums");
}
