// Attention in fp32 arithmetic on 16x16 matrix instructions, for any element
// type, any strides, head_dim up to 128: o = softmax(scale * q k^T [+ masks]) v
// and its gradients, with the semantics of attn_fwd.hip and attn_bwd.hip
// (reference: fused_attention.py:14-110, 113-338, 706-823 and the masked SDPA
// call attention.py:268-299).  fp32 and fp16 calls run here, and bf16 calls
// whose head_dim or strides the bf16 MFMA kernels do not take.
//
// Arithmetic.  fp32 elements: v_mfma_f32_16x16x4_f32 throughout.  16-bit
// elements: q k^T and dO v^T go to the 16-bit instructions as they are (their
// products are exact in fp32), and the fp32 probabilities and score gradients
// go there as two or three 16-bit planes that add up to them to fp32's own
// precision (prob_product, grad_product), so nothing is held to 16 bits.
//
// Rows that a query does not see stay out of its sums whatever they hold, an
// infinity or NaN included, but a product over a whole tile gives them the
// weight 0, and 0 * inf is NaN; so are the planes of an infinity (inf - inf),
// of a score gradient that overflowed and of a probability past what fp16's
// planes hold.  All of these leave a NaN in the accumulators, so a wave that
// ends with one walks its tiles a second time, row by row in fp32, each row
// meeting only the columns that see it (row_dot, add_row).  It is a loop of its
// own after the other: inside that one it would cost 30 to 70 registers there.
// Forward / backward, against a test of every staged tile that 16-bit types
// made before (for overflow alone; fp32 made none): fp16 B8 8/2 heads x 64, S
// 2048 157 / 532 -> 129 / 467 us, fp32 B4 8/2 x 64, S 2048 192 / 615 -> 198 /
// 617.
//
// What bounds it.  fp32: the fp32 matrix rate (256 FLOP per CU and cycle, a
// tenth of bf16's measured rate); a 16x16x4 step takes 32 cycles of a SIMD,
// against one 4-byte LDS read per lane, so LDS and the softmax's VALU work hide
// behind it.  16 bits: VALU (exponentials, splits) and LDS reads.  The 16x16
// tile (and not 32x32) because a wave then holds 16 rows: K and V (or Q and dO)
// fragments and both accumulators of head_dim 128 fit the registers without
// spills.
//
// Layouts.  A fragment of rows X[m][d] (m = lane % 16, g = lane / 16) takes the
// summed index d in runs of R = 4 (fp32, or head_dim 16) or 8 elements, 4 R j +
// R g + i over steps (j, i): one 16-byte LDS read feeds a step, and the resident
// side holds the same order.  A result tile has row 4 g + r in register r and
// column lane % 16, so its registers are the B operand of the next product with
// the summed index in the order 4 g + r, whose A operand is a 4-byte read of
// row 4 g + r of the staged tile (fp32) or a transposing read (16 bits):
// nothing is transposed.  Staged rows are 16 bytes longer than head_dim, which
// puts the row groups of such reads into different banks.
//
// Every wave owns 16 rows (queries forward and for dQ, keys for dK/dV); a
// workgroup's four waves share the staged 32-row tiles of the other side,
// double-buffered, the next tile's loads in flight during the arithmetic.
// dK/dV and dQ walks are cut into chunks of equally many tiles so that the
// launch fills the device; their fp32 partials are summed in chunk order
// (deterministic).
//
// Measured, forward + backward of one call, against what these calls took
// before (16 lanes per query row forward, one thread per row backward, VALU):
// fp16 B2 8/2 heads x 64, S 1500, causal 198.1 -> 0.15 ms (launch-bound); fp32
// B4 8/2 x 64, S 2048, causal 274 -> 0.81 ms; fp32 B1 4/1 x 128, S 1000 172.9 ->
// 0.26 ms; fp32 B2 8/2 x 16, S 512, causal 8.7 -> 0.17 ms (launch-bound).
// Errors against 64 bits: fp32 1.8e-6 -> 5.8e-7, fp16 2.3e-4 (the output's
// rounding) both.  16-bit planes against the fp32 instruction on the converted
// rows, fp16: the first of these calls' kernels forward 71 -> 32, dK/dV 115 ->
// 50, dQ 88 -> 34 us; B8 8/2 x 64, S 2048 1516 -> 596 us; B2 8/2 x 128, S 2048
// 841 -> 318 us; B4 8/2 x 16, S 2048 270 -> 194 us.
#include "attn_f32.h"

#include <algorithm>
#include <cmath>

#include "common.h"

namespace hydra {
namespace {

typedef __attribute__((ext_vector_type(4))) float f32x4;

constexpr float kLog2eF = 1.4426950408889634f;
constexpr float kLn2F = 0.6931471805599453f;
constexpr int kWaves = 4;
constexpr int kThreads = 64 * kWaves;
constexpr int kTile = 32;  // staged rows per step

__device__ __forceinline__ f32x4 mfma4(float a, float b, f32x4 c) {
  return __builtin_amdgcn_mfma_f32_16x16x4f32(a, b, c, 0, 0, 0);
}

struct Strides3 {
  int64_t b, h, s;
};

// One operand of the staged side: rows `row0 ..` of `base`, `rs` apart,
// elements `es` apart; `vec`: 16-byte loads are allowed (hd == HDP, unit
// element stride, aligned rows).
template <typename T>
struct Rows {
  const T* base;
  int64_t rs, es;
};

// How many consecutive elements of a row a lane holds per step of a row
// product, and a row's steps.
template <typename T, int HDP>
struct Row16 {
  static constexpr int R = sizeof(T) == 2 && HDP >= 32 ? 8 : 4;
  static constexpr int N = HDP / (4 * R);
  struct __attribute__((aligned(R * sizeof(T)))) Run {
    T v[R];
  };
};

// fp16's gradient products read the staged rows as two bf16 planes (hi + lo,
// exact), tiles of their own after the staged pair.
template <typename T>
constexpr bool kPlaneTiles = std::is_same<T, f16>::value;

// Registers of one thread's share of a staged tile, and its way to LDS (t:
// the thread's index among the kThreads that stage it).
template <typename T, int HDP>
struct Stage {
  static constexpr int E = 16 / int(sizeof(T));     // elements per 16-byte load
  static constexpr int P = HDP + E;                 // elements per staged row
  static constexpr int VU = (kTile * HDP / E + kThreads - 1) / kThreads;
  static constexpr int SU = kTile * HDP / kThreads;  // scalar path: elements per thread
  static constexpr int N = kTile * P;                // elements per tile
  static constexpr bool WHOLE = (kTile * HDP / E) % kThreads == 0;

  uint4 raw[VU];

  __device__ __forceinline__ void fetch(const Rows<T>& r, int row0, int S, int t) {
#pragma unroll
    for (int u = 0; u < VU; ++u) {
      const int i = t + kThreads * u;
      const int row = i / (HDP / E), c = i - row * (HDP / E);
      const bool ok = (WHOLE || row < kTile) && row0 + row < S;
      raw[u] = make_uint4(0, 0, 0, 0);
      if (ok) raw[u] = ld16raw<false>(r.base + static_cast<int64_t>(row0 + row) * r.rs + c * E);
    }
  }
  // planes: where the bf16 planes go (kPlaneTiles), or null
  __device__ __forceinline__ void land(T* dst, T* planes, int t) const {
#pragma unroll
    for (int u = 0; u < VU; ++u) {
      const int i = t + kThreads * u;
      const int row = i / (HDP / E), c = i - row * (HDP / E);
      if (WHOLE || row < kTile) {
        *reinterpret_cast<uint4*>(&dst[row * P + c * E]) = raw[u];
        if constexpr (kPlaneTiles<T>) {
          if (planes) {
            float f[8], lo[8];
            unpack16<f16>(raw[u], f);
            const uint4 h = pack16<bf16>(f);
            unpack16<bf16>(h, lo);
#pragma unroll
            for (int e = 0; e < 8; ++e) lo[e] = f[e] - lo[e];
            *reinterpret_cast<uint4*>(&planes[row * P + c * E]) = h;
            *reinterpret_cast<uint4*>(&planes[N + row * P + c * E]) = pack16<bf16>(lo);
          }
        }
      }
    }
  }
  // Any strides and head_dim: element by element, straight to LDS.
  static __device__ __forceinline__ void direct(const Rows<T>& r, int row0, int S, int hd, T* dst, T* planes, int t) {
#pragma unroll 4
    for (int u = 0; u < SU; ++u) {
      const int i = t + kThreads * u;
      const int row = i / HDP, d = i - row * HDP;
      const bool ok = row0 + row < S && d < hd;
      T x = from_f32<T>(0.f);
      if (ok) x = r.base[static_cast<int64_t>(row0 + row) * r.rs + d * r.es];
      dst[row * P + d] = x;
      if constexpr (kPlaneTiles<T>) {
        if (planes) {
          const float f = to_f32(x);
          const bf16 h = from_f32<bf16>(f);
          planes[row * P + d].bits = h.bits;
          planes[N + row * P + d].bits = from_f32<bf16>(f - to_f32(h)).bits;
        }
      }
    }
  }
};

// The resident fragment of one row (column lane % 16 of B): elements
// 4 R j + R g + i of the row (R = Row16::R), zero past hd or for a row that is not
// there.  vec: rows of HDP elements, aligned to R of them.
template <typename T, int HDP>
__device__ __forceinline__ void load_frag(const T* row, typename Row16<T, HDP>::Run (&f)[Row16<T, HDP>::N], int g, int hd,
                                          bool ok, bool vec) {
  constexpr int R = Row16<T, HDP>::R;
#pragma unroll
  for (int j = 0; j < Row16<T, HDP>::N; ++j)
#pragma unroll
    for (int i = 0; i < R; ++i) f[j].v[i] = from_f32<T>(0.f);
  if (!ok) return;
  if (vec) {
#pragma unroll
    for (int j = 0; j < Row16<T, HDP>::N; ++j) f[j] = *reinterpret_cast<const typename Row16<T, HDP>::Run*>(row + 4 * R * j + R * g);
  } else {
#pragma unroll
    for (int j = 0; j < Row16<T, HDP>::N; ++j)
#pragma unroll
      for (int i = 0; i < R; ++i) {
        const int d = 4 * R * j + R * g + i;
        if (d < hd) f[j].v[i] = row[d];
      }
  }
}

typedef __attribute__((ext_vector_type(4))) short s16x4;
typedef __attribute__((ext_vector_type(8))) __bf16 bf16x8;
typedef __attribute__((ext_vector_type(4))) _Float16 f16x4;
typedef __attribute__((ext_vector_type(8))) _Float16 f16x8;

__device__ __forceinline__ f32x4 mfma16(f16, uint2 a, uint2 b, f32x4 c) {
  return __builtin_amdgcn_mfma_f32_16x16x16f16(__builtin_bit_cast(f16x4, a), __builtin_bit_cast(f16x4, b), c, 0, 0, 0);
}
__device__ __forceinline__ f32x4 mfma16(bf16, uint2 a, uint2 b, f32x4 c) {
  return __builtin_amdgcn_mfma_f32_16x16x16bf16_1k(__builtin_bit_cast(s16x4, a), __builtin_bit_cast(s16x4, b), c, 0, 0,
                                                   0);
}
__device__ __forceinline__ f32x4 mfma32(f16, uint4 a, uint4 b, f32x4 c) {
  return __builtin_amdgcn_mfma_f32_16x16x32_f16(__builtin_bit_cast(f16x8, a), __builtin_bit_cast(f16x8, b), c, 0, 0, 0);
}
__device__ __forceinline__ f32x4 mfma32(bf16, uint4 a, uint4 b, f32x4 c) {
  return __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(bf16x8, a), __builtin_bit_cast(bf16x8, b), c, 0, 0,
                                                 0);
}

// S and dP tiles (or S alone): 16 staged rows times the resident fragment.
// 16-bit elements go to the 16-bit matrix instructions as they are: their
// products are exact there and the sums fp32.
template <typename T, int HDP>
__device__ __forceinline__ f32x4 row_product(const T* rows, const typename Row16<T, HDP>::Run (&f)[Row16<T, HDP>::N], int n, int g) {
  constexpr int R = Row16<T, HDP>::R;
  f32x4 c = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
  for (int j = 0; j < Row16<T, HDP>::N; ++j) {
    const auto a = *reinterpret_cast<const typename Row16<T, HDP>::Run*>(&rows[n * Stage<T, HDP>::P + 4 * R * j + R * g]);
    if constexpr (sizeof(T) == 4) {
#pragma unroll
      for (int i = 0; i < 4; ++i) c = mfma4(a.v[i], f[j].v[i], c);
    } else if constexpr (R == 4) {
      c = mfma16(T{}, __builtin_bit_cast(uint2, a), __builtin_bit_cast(uint2, f[j]), c);
    } else {
      c = mfma32(T{}, __builtin_bit_cast(uint4, a), __builtin_bit_cast(uint4, f[j]), c);
    }
  }
  return c;
}

// acc[d tile] += rows^T * x in fp32: x a result tile whose rows are 16 staged
// rows of fp32 elements.
template <int HDP>
__device__ __forceinline__ void col_product(f32x4 (&acc)[HDP / 16], const float* rows, const f32x4& x, int n, int g) {
#pragma unroll
  for (int r = 0; r < 4; ++r)
#pragma unroll
    for (int t = 0; t < HDP / 16; ++t)
      acc[t] = mfma4(rows[(4 * g + r) * Stage<float, HDP>::P + 16 * t + n], x[r], acc[t]);
}

// What follows serves the second walk (see the top of the file): one row at a
// time, straight from memory, any type and strides, plain fp32.
// The dot product of a row with the resident fragment of each column.
template <typename T, int HDP>
__device__ __forceinline__ float row_dot(const T* row, const typename Row16<T, HDP>::Run (&f)[Row16<T, HDP>::N], int g,
                                         int hd) {
  constexpr int R = Row16<T, HDP>::R;
  float s = 0.f;
  asm volatile("" : "+v"(g));  // offsets and bounds made here, row by row: kept, they would take 60 registers
#pragma unroll
  for (int j = 0; j < Row16<T, HDP>::N; ++j) {
#pragma unroll
    for (int i = 0; i < R; ++i) {
      const int d = 4 * R * j + R * g + i;
      if (d < hd) s = fmaf(to_f32(f[j].v[i]), to_f32(row[d]), s);
    }
  }
  s += __shfl_xor(s, 16);
  return s + __shfl_xor(s, 32);
}
// acc += w * row, elements es apart.
template <typename T, int HDP>
__device__ __forceinline__ void add_row(f32x4 (&acc)[HDP / 16], const T* row, int64_t es, float w, int g, int hd) {
  asm volatile("" : "+v"(g));
#pragma unroll
  for (int t = 0; t < HDP / 16; ++t) {
#pragma unroll
    for (int r = 0; r < 4; ++r) {
      const int d = 16 * t + 4 * g + r;
      if (d < hd) acc[t][r] = fmaf(w, to_f32(row[d * es]), acc[t][r]);
    }
  }
}

template <int N>
__device__ __forceinline__ bool any_nan(const f32x4 (&a)[N]) {
  bool nan = false;
#pragma unroll
  for (int t = 0; t < N; ++t)
#pragma unroll
    for (int r = 0; r < 4; ++r) nan |= a[t][r] != a[t][r];
  return nan;
}

// The same over a whole staged tile of a 16-bit type, x as planes of 16-bit
// values that add up to it.  The summed index: slot i < 4 of lane group g is
// row 4 g + i, slot 4 + i row 16 + 4 g + i, which is the order the two result
// tiles hold; the transposing LDS read gives the same (16 lanes read 4 rows of
// 16 columns, lane j gets column j's four values).
template <typename T, int HDP>
__device__ __forceinline__ uint4 tile_cols(const T* tile, int t, int n, int g) {
  typedef __attribute__((address_space(3))) s16x4* lds_t;
  constexpr int P = Stage<T, HDP>::P;
  const T* p = tile + (4 * g + (n >> 2)) * P + 16 * t + 4 * (n & 3);
  const uint2 lo = __builtin_bit_cast(uint2, __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_t)(p)));
  const uint2 hi = __builtin_bit_cast(uint2, __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_t)(p + 16 * P)));
  return make_uint4(lo.x, lo.y, hi.x, hi.y);
}

// x as three bf16 planes, exactly: each takes the next 8 bits, rounded to
// nearest, so what is left after it is at most 2^-9 of it (truncation would
// leave 2^-7).  A value past bf16's largest overflows to inf - inf.
__device__ __forceinline__ void split3(const f32x4 (&x)[2], uint4 (&p)[3]) {
  uint32_t w[3][4];
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    float a = x[i >> 1][2 * (i & 1)], b = x[i >> 1][2 * (i & 1) + 1];
#pragma unroll
    for (int k = 0; k < 3; ++k) {
      w[k][i] = pack2<bf16>(a, b);
      a -= __uint_as_float(w[k][i] << 16);
      b -= __uint_as_float(w[k][i] & 0xffff0000u);
    }
  }
#pragma unroll
  for (int k = 0; k < 3; ++k) p[k] = make_uint4(w[k][0], w[k][1], w[k][2], w[k][3]);
}

// Probabilities (0 .. 1): three bf16 planes beside bf16 rows; beside fp16 rows
// two fp16 planes of x * kPScale, whose remainder is under half an fp32 ulp of
// x (under 2^-39 for x below 2^-16, where the second plane goes subnormal).
// Accumulators of either come out times kPScale.
template <typename T>
constexpr float kPScale = std::is_same<T, f16>::value ? 16384.f : 1.f;

template <typename T, int HDP>
__device__ __forceinline__ void prob_product(f32x4 (&acc)[HDP / 16], const T* tile, const f32x4 (&x)[2], int n, int g) {
  if constexpr (std::is_same<T, f16>::value) {
    uint32_t h[4], l[4];
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      const float a = x[i >> 1][2 * (i & 1)] * kPScale<T>, b = x[i >> 1][2 * (i & 1) + 1] * kPScale<T>;
      const f16 ha = from_f32<f16>(a), hb = from_f32<f16>(b);
      h[i] = static_cast<uint32_t>(ha.bits) | (static_cast<uint32_t>(hb.bits) << 16);
      l[i] = pack2<f16>(a - to_f32(ha), b - to_f32(hb));
    }
    const uint4 ph = make_uint4(h[0], h[1], h[2], h[3]), pl = make_uint4(l[0], l[1], l[2], l[3]);
#pragma unroll
    for (int t = 0; t < HDP / 16; ++t) {
      const uint4 a = tile_cols<T, HDP>(tile, t, n, g);
      acc[t] = mfma32(f16{}, a, pl, acc[t]);
      acc[t] = mfma32(f16{}, a, ph, acc[t]);
    }
  } else {
    uint4 p[3];
    split3(x, p);
#pragma unroll
    for (int t = 0; t < HDP / 16; ++t) {
      const uint4 a = tile_cols<T, HDP>(tile, t, n, g);
#pragma unroll
      for (int k = 2; k >= 0; --k) acc[t] = mfma32(bf16{}, a, p[k], acc[t]);
    }
  }
}

// dS of any size: three bf16 planes times bf16 rows, or times the two bf16
// planes of fp16 rows.  The product of the two smallest is left out: 2^-8 of
// the row element times 2^-17 of dS, at most 2^-25 of the sum's terms (over all
// fp16 significands and 4 M of fp32; half of what one fp32 product rounds off).
template <typename T, int HDP>
__device__ __forceinline__ void grad_product(f32x4 (&acc)[HDP / 16], const T* tile, const T* planes,
                                             const f32x4 (&x)[2], int n, int g) {
  uint4 p[3];
  split3(x, p);
#pragma unroll
  for (int t = 0; t < HDP / 16; ++t) {
    const uint4 a = tile_cols<T, HDP>(kPlaneTiles<T> ? planes : tile, t, n, g);
    if constexpr (kPlaneTiles<T>) {
      const uint4 b = tile_cols<T, HDP>(planes + Stage<T, HDP>::N, t, n, g);
      acc[t] = mfma32(bf16{}, b, p[1], acc[t]);
      acc[t] = mfma32(bf16{}, b, p[0], acc[t]);
    }
#pragma unroll
    for (int k = 2; k >= 0; --k) acc[t] = mfma32(bf16{}, a, p[k], acc[t]);
  }
}

// Writes a wave's 16 rows (column n) of accumulators, scaled.
template <typename T, int HDP>
__device__ __forceinline__ void store_rows(T* row, const f32x4 (&acc)[HDP / 16], float scale, int g, int hd) {
#pragma unroll
  for (int t = 0; t < HDP / 16; ++t)
#pragma unroll
    for (int r = 0; r < 4; ++r) {
      const int d = 16 * t + 4 * g + r;
      if (d < hd) row[d] = from_f32<T>(acc[t][r] * scale);
    }
}
template <int HDP>
__device__ __forceinline__ void store_part(float* row, const f32x4 (&acc)[HDP / 16], float f, int g) {
#pragma unroll
  for (int t = 0; t < HDP / 16; ++t)
    *reinterpret_cast<float4*>(row + 16 * t + 4 * g) = make_float4(acc[t][0] * f, acc[t][1] * f, acc[t][2] * f, acc[t][3] * f);
}

// Whether query s sees key t < S (keep: the key mask's flag of t).
__device__ __forceinline__ bool sees(int s, int t, bool keep, bool causal, int mode) {
  if (mode == HYDRA_MASK_REFERENCE_SDPA) return t > s || !keep;
  return (!causal || t <= s) && (mode != HYDRA_MASK_KEY_PADDING || keep);
}

// Queries of a wave: task (16 rows of one query head of the group) of an
// item of kWaves tasks, the group's heads first so that a workgroup's waves
// share the key range.
struct Task {
  int h, q0;
  bool active;
};
__device__ __forceinline__ Task task_of(int task, int ntasks, int kvh, int G) {
  Task t;
  t.active = task < ntasks;
  const int c = t.active ? task : ntasks - 1;
  t.q0 = 16 * (c / G);
  t.h = kvh * G + c % G;
  return t;
}

// ---------------------------------------------------------------- forward
// KG key groups of four waves share an item: group kg walks key tiles kg, kg +
// KG, .. with its own staged tiles, and group 0 folds the others' (O, m, l) in
// group order at the end.  KG > 1 where there are too few items to fill the
// device: their walks are then KG times shorter (see launch_fwd).
template <typename T, int HDP, int KG>
__global__ __launch_bounds__(kThreads * KG) void attn_fwd_f32_kernel(
    const T* __restrict__ q, const T* __restrict__ k, const T* __restrict__ v, T* __restrict__ o,
    float* __restrict__ lse, const uint8_t* __restrict__ kmask, int mode, int Hq, int Hkv, int S, int hd, int G,
    int ntasks, int items, Strides3 qs, Strides3 ks, Strides3 vs, int64_t vs3, Strides3 os, int causal, int vec,
    float scale_log2) {
  using St = Stage<T, HDP>;
  __shared__ __attribute__((aligned(16))) T smem_all[KG][2][2 * St::N];
  __shared__ int keep_all[KG][2][kTile];
  const int kg = KG > 1 ? __builtin_amdgcn_readfirstlane(threadIdx.x / kThreads) : 0;
  const int tid = threadIdx.x - kg * kThreads, lane = tid & 63, n = lane & 15, g = lane >> 4;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  auto& smem = smem_all[kg];
  auto& keepv = keep_all[kg];
  const int BHkv = gridDim.x / items;
  const int bk = blockIdx.x % BHkv;
  const int item = items - 1 - static_cast<int>(blockIdx.x / BHkv);  // longest key ranges first
  const int b = bk / Hkv, kvh = bk - b * Hkv;
  const Task tk = task_of(kWaves * item + wave, ntasks, kvh, G);
  const int qi = tk.q0 + n;
  const bool qok = tk.active && qi < S;
  typename Row16<T, HDP>::Run qf[Row16<T, HDP>::N];
  load_frag<T, HDP>(q + b * qs.b + tk.h * qs.h + static_cast<int64_t>(qok ? qi : 0) * qs.s, qf, g, hd, qok, vec & 2);

  const bool walk = causal && mode != HYDRA_MASK_REFERENCE_SDPA;
  const int last_task = min(kWaves * item + kWaves - 1, ntasks - 1);
  const int kend = walk ? min(16 * (last_task / G) + 16, S) : S;
  const int nt = (kend + kTile - 1) / kTile;
  const int my_end = !tk.active ? 0 : walk ? min(tk.q0 + 16, S) : S;  // keys this wave sees
  const Rows<T> kr{k + b * ks.b + kvh * ks.h, ks.s, 1};
  const Rows<T> vr{v + b * vs.b + kvh * vs.h, vs.s, vs3};

  f32x4 acc[HDP / 16];
#pragma unroll
  for (int t = 0; t < HDP / 16; ++t) acc[t] = f32x4{0.f, 0.f, 0.f, 0.f};
  float m = -INFINITY, l = 0.f;
  St sk, sv;
  int kp = 0;
  auto fetch = [&](int t) {
    if (vec & 1) {
      sk.fetch(kr, kTile * t, S, tid);
      sv.fetch(vr, kTile * t, S, tid);
    }
    if (mode != HYDRA_MASK_NONE && tid < kTile) {
      const int key = kTile * t + tid;
      kp = key < S ? kmask[static_cast<int64_t>(b) * S + key] : 0;
    }
  };
  auto land = [&](int t, int buf) {
    if (vec & 1) {
      sk.land(smem[buf], nullptr, tid);
      sv.land(smem[buf] + St::N, nullptr, tid);
    } else {
      St::direct(kr, kTile * t, S, hd, smem[buf], nullptr, tid);
      St::direct(vr, kTile * t, S, hd, smem[buf] + St::N, nullptr, tid);
    }
    if (mode != HYDRA_MASK_NONE && tid < kTile) keepv[buf][tid] = kp;
  };
  if (kg < nt) {
    fetch(kg);
    land(kg, 0);
  }
  const int steps = (nt + KG - 1) / KG;
  for (int st = 0; st < steps; ++st) {
    __syncthreads();
    const int t = KG * st + kg, buf = st & 1, t0 = kTile * t;
    if (t + KG < nt) fetch(t + KG);
    if (t0 < my_end) {
      const T* Ks = smem[buf];
      const T* Vs = Ks + St::N;
      f32x4 x[2];
      float mt = m;
#pragma unroll
      for (int u = 0; u < 2; ++u) x[u] = row_product<T, HDP>(Ks + 16 * u * St::P, qf, n, g);
      // whole tile visible to every row of the wave: no tests
      const bool plain = mode == HYDRA_MASK_NONE && t0 + kTile - 1 <= (walk ? tk.q0 : S - 1) && t0 + kTile <= S;
#pragma unroll
      for (int u = 0; u < 2; ++u)
#pragma unroll
        for (int r = 0; r < 4; ++r) {
          float xs = x[u][r] * scale_log2;
          if (!plain) {
            const int i = 16 * u + 4 * g + r, key = t0 + i;
            const bool keep = mode == HYDRA_MASK_NONE || keepv[buf][i] != 0;
            if (!(key < S && sees(qi, key, keep, causal, mode))) xs = -INFINITY;
          }
          x[u][r] = xs;
          mt = fmaxf(mt, xs);
        }
      mt = fmaxf(mt, __shfl_xor(mt, 16));
      mt = fmaxf(mt, __shfl_xor(mt, 32));
      const float ms = mt == -INFINITY ? 0.f : mt;  // nothing visible yet: every p is exp2(-inf) = 0
      if (__any(mt > m)) {
        const float alpha = __builtin_amdgcn_exp2f(m - ms);  // m = -inf -> 0
        l *= alpha;
#pragma unroll
        for (int d = 0; d < HDP / 16; ++d) acc[d] *= alpha;
        m = mt;
      }
#pragma unroll
      for (int u = 0; u < 2; ++u) {
#pragma unroll
        for (int r = 0; r < 4; ++r) {
          x[u][r] = __builtin_amdgcn_exp2f(x[u][r] - ms);
          l += x[u][r];
        }
        if constexpr (sizeof(T) == 4) col_product<HDP>(acc, Vs + 16 * u * St::P, x[u], n, g);
      }
      if constexpr (sizeof(T) == 2) prob_product<T, HDP>(acc, Vs, x, n, g);
    }
    if (t + KG < nt) land(t + KG, buf ^ 1);
  }
  if (__any(qok && any_nan(acc))) {  // the second walk
    m = -INFINITY;
    l = 0.f;
#pragma unroll
    for (int d = 0; d < HDP / 16; ++d) acc[d] = f32x4{0.f, 0.f, 0.f, 0.f};
    for (int t = kg; t < nt; t += KG)
#pragma unroll 1
      for (int key = kTile * t; key < min(kTile * t + kTile, S); ++key) {
        const bool keep = mode == HYDRA_MASK_NONE || kmask[static_cast<int64_t>(b) * S + key] != 0;
        const bool see = qok && sees(qi, key, keep, causal, mode);
        if (!__any(see)) continue;
        const float x = row_dot<T, HDP>(kr.base + key * kr.rs, qf, g, hd) * scale_log2;
        if (!see) continue;
        if (x > m) {
          const float alpha = __builtin_amdgcn_exp2f(m - x);  // m = -inf -> 0
          l *= alpha;
#pragma unroll
          for (int d = 0; d < HDP / 16; ++d) acc[d] *= alpha;
          m = x;
        }
        const float p = __builtin_amdgcn_exp2f(x - (m == -INFINITY ? 0.f : m));
        if (g == 0) l += p;  // the row's sum over its four lanes follows
        add_row<T, HDP>(acc, vr.base + key * vr.rs, vr.es, p * kPScale<T>, g, hd);
      }
  }
  if constexpr (KG > 1) {
    constexpr int NA = HDP / 16, XF = 4 * NA + 2;  // floats a lane hands over
    static_assert(kThreads * XF * sizeof(float) <= 4 * St::N * sizeof(T), "the exchange fits a group's tiles");
    __syncthreads();  // every group is done with its tiles
    float* mine = reinterpret_cast<float*>(&smem_all[kg][0][0]);
    if (kg > 0) {
#pragma unroll
      for (int d = 0; d < NA; ++d)
#pragma unroll
        for (int r = 0; r < 4; ++r) mine[(4 * d + r) * kThreads + tid] = acc[d][r];
      mine[4 * NA * kThreads + tid] = m;
      mine[(4 * NA + 1) * kThreads + tid] = l;
    }
    __syncthreads();
    if (kg > 0) return;
#pragma unroll
    for (int o2 = 1; o2 < KG; ++o2) {
      const float* x = reinterpret_cast<const float*>(&smem_all[o2][0][0]);
      const float m2 = x[4 * NA * kThreads + tid], l2 = x[(4 * NA + 1) * kThreads + tid];
      if (m2 == -INFINITY) continue;  // saw no key of this row
      const float mn = fmaxf(m, m2);
      const float s1 = __builtin_amdgcn_exp2f(m - mn), s2 = __builtin_amdgcn_exp2f(m2 - mn);
      l = l * s1 + l2 * s2;
#pragma unroll
      for (int d = 0; d < NA; ++d)
#pragma unroll
        for (int r = 0; r < 4; ++r) acc[d][r] = acc[d][r] * s1 + x[(4 * d + r) * kThreads + tid] * s2;
      m = mn;
    }
  }
  l += __shfl_xor(l, 16);
  l += __shfl_xor(l, 32);
  if (!qok) return;
  const float inv = l > 0.f ? (1.f / kPScale<T>) / l : 0.f;
  store_rows<T, HDP>(o + b * os.b + tk.h * os.h + static_cast<int64_t>(qi) * os.s, acc, inv, g, hd);
  if (lse && g == 0)
    lse[(static_cast<int64_t>(b) * Hq + tk.h) * S + qi] = l > 0.f ? (m + __log2f(l)) * kLn2F : -INFINITY;
}

// --------------------------------------------------------------- backward
// Tiles of 32 queries that reach key group kg (64 keys), per query head.
__host__ __device__ inline int q_tiles(int kg, int S, bool walk) {
  const int all = (S + kTile - 1) / kTile;
  return walk ? all - 2 * kg : all;
}

// Key tiles that item `i`'s queries (kWaves tasks of 16 rows) reach.
__host__ __device__ inline int k_tiles(int i, int ntasks, int G, int S, bool walk) {
  const int last = kWaves * i + kWaves - 1 < ntasks ? kWaves * i + kWaves - 1 : ntasks - 1;
  const int end = walk && 16 * (last / G) + 16 < S ? 16 * (last / G) + 16 : S;
  return (end + kTile - 1) / kTile;
}

// Workgroup id -> (batch x kv head, part i, chunk c of it): the parts' chunks
// of one (batch, head) in a row, the (batch, head) fastest.  Workgroups go to
// the 8 XCDs in turn, so each XCD gets every 8th of equally long chunks (grids
// with empty chunks in them left some XCDs idle: dK/dV 588 us with the chunk
// slowest, 397 with it fastest, 363 so, fp32 B4 8/2 heads x 64, S 2048),
// and with 8 (batch, head) pairs one pair's rows per L2.  64 parts at a time.
template <typename F>
__device__ __forceinline__ bool locate(int id, int BHkv, int n, int ch, F tiles, int& bk, int& i, int& c) {
  bk = id % BHkv;
  int j = id / BHkv;
  const int lane = threadIdx.x & 63;
  for (int base = 0; base < n; base += 64) {
    const int p = base + lane;
    int cum = p < n ? (tiles(p) + ch - 1) / ch : 0;
#pragma unroll
    for (int off = 1; off < 64; off <<= 1) {
      const int up = __shfl_up(cum, off);
      if (lane >= off) cum += up;
    }
    const int all = __builtin_amdgcn_readlane(cum, 63);
    if (j < all) {
      const int at = __popcll(__ballot(cum <= j));  // the first part whose running count passes j
      const int before = at ? __builtin_amdgcn_readlane(cum, at - 1) : 0;
      i = base + at;
      c = j - before;
      return true;
    }
    j -= all;
  }
  return false;
}

// dK/dV: a workgroup takes 64 keys of one (batch, kv head) and a chunk of the
// (head of the group, query tile) walk.
template <typename T, int HDP>
__global__ __launch_bounds__(kThreads) void attn_bwd_f32_dkdv_kernel(
    const T* __restrict__ q, const T* __restrict__ k, const T* __restrict__ v, const T* __restrict__ dout,
    const float* __restrict__ dvec, const float* __restrict__ lse2, const uint8_t* __restrict__ kmask, int mode,
    T* __restrict__ dk, T* __restrict__ dv, float* __restrict__ part, int Hq, int Hkv, int S, int hd, int G,
    int BHkv, int nkg, int ch, int maxch, Strides3 qs, Strides3 ks, Strides3 vs, Strides3 ds, Strides3 dks, Strides3 dvs,
    int causal, int vec, float scale_log2, float scale) {
  using St = Stage<T, HDP>;
  constexpr int NT = kPlaneTiles<T> ? 4 : 2;  // Q, dO, Q's planes
  __shared__ __attribute__((aligned(16))) T smem[2][NT * St::N];
  __shared__ __attribute__((aligned(16))) float rowv[2][2][kTile];  // lse2 and D of the tile's rows
  const int tid = threadIdx.x, lane = tid & 63, n = lane & 15, g = lane >> 4;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const bool walk = causal && mode != HYDRA_MASK_REFERENCE_SDPA;
  int bk, kg, c;
  if (!locate(blockIdx.x, BHkv, nkg, ch, [&](int i) { return G * q_tiles(i, S, walk); }, bk, kg, c)) return;
  bk = __builtin_amdgcn_readfirstlane(bk);
  kg = __builtin_amdgcn_readfirstlane(kg);
  c = __builtin_amdgcn_readfirstlane(c);
  const int rest = bk * nkg + kg, parts = BHkv * nkg;
  const int b = bk / Hkv, kvh = bk - b * Hkv;
  const int qt0 = walk ? 2 * kg : 0;
  const int nq = q_tiles(kg, S, walk);
  const int total = G * nq;
  const int kw0 = 64 * kg + 16 * wave, key = kw0 + n;
  bool keep = key < S;
  if (mode != HYDRA_MASK_NONE && keep) keep = kmask[static_cast<int64_t>(b) * S + key] != 0;
  // Key padding: a lane's key is its own column of every product, so masked
  // lanes store zeros at the end and waves without a key that counts rest.
  const bool pad = mode == HYDRA_MASK_KEY_PADDING;
  const bool wave_any = !pad || __builtin_amdgcn_readfirstlane(__any(keep)) != 0;
  const bool wg_any = !pad || __syncthreads_or(keep) != 0;
  const int kbnd = mode == HYDRA_MASK_REFERENCE_SDPA && !keep ? 0x7fffffff : key;

  typename Row16<T, HDP>::Run kf[Row16<T, HDP>::N], vf[Row16<T, HDP>::N];
  load_frag<T, HDP>(k + b * ks.b + kvh * ks.h + static_cast<int64_t>(key < S ? key : 0) * ks.s, kf, g, hd, key < S, vec & 2);
  load_frag<T, HDP>(v + b * vs.b + kvh * vs.h + static_cast<int64_t>(key < S ? key : 0) * vs.s, vf, g, hd, key < S, vec & 2);
  f32x4 dka[HDP / 16], dva[HDP / 16];
#pragma unroll
  for (int t = 0; t < HDP / 16; ++t) dka[t] = dva[t] = f32x4{0.f, 0.f, 0.f, 0.f};

  St sq, sd;
  float rv = 0.f;
  auto fetch = [&](int step) {
    const int hr = step / nq, row0 = kTile * (qt0 + step - hr * nq), h = kvh * G + hr;
    if (vec & 1) {
      sq.fetch(Rows<T>{q + b * qs.b + h * qs.h, qs.s, 1}, row0, S, tid);
      sd.fetch(Rows<T>{dout + b * ds.b + h * ds.h, ds.s, 1}, row0, S, tid);
    }
    if (tid < 2 * kTile) {  // rows past S: zero, with zero Q and dO they add nothing
      const int row = row0 + (tid & (kTile - 1));
      const float* src = tid < kTile ? lse2 : dvec;
      rv = row < S ? src[(static_cast<int64_t>(b) * Hq + h) * S + row] : 0.f;
    }
  };
  auto land = [&](int step, int buf) {
    T* planes = kPlaneTiles<T> ? smem[buf] + 2 * St::N : nullptr;
    if (vec & 1) {
      sq.land(smem[buf], planes, tid);
      sd.land(smem[buf] + St::N, nullptr, tid);
    } else {
      const int hr = step / nq, row0 = kTile * (qt0 + step - hr * nq), h = kvh * G + hr;
      St::direct(Rows<T>{q + b * qs.b + h * qs.h, qs.s, 1}, row0, S, hd, smem[buf], planes, tid);
      St::direct(Rows<T>{dout + b * ds.b + h * ds.h, ds.s, 1}, row0, S, hd, smem[buf] + St::N, nullptr, tid);
    }
    if (tid < 2 * kTile) rowv[buf][tid / kTile][tid & (kTile - 1)] = rv;
  };
  const int first = c * ch, end = wg_any ? min(first + ch, total) : first;
  if (first < end) {
    fetch(first);
    land(first, 0);
  }
  for (int step = first; step < end; ++step) {
    __syncthreads();
    const int buf = (step - first) & 1;
    if (step + 1 < end) fetch(step + 1);
    const int q0 = kTile * (qt0 + step % nq);
    // causal: a tile before the wave's keys holds nothing of theirs
    if (wave_any && (!walk || q0 + kTile - 1 >= kw0)) {
      const bool plain = walk ? q0 >= kw0 + 15 : mode != HYDRA_MASK_REFERENCE_SDPA;
      f32x4 p[2], dp[2];
#pragma unroll
      for (int u = 0; u < 2; ++u) {
        const T* Qs = smem[buf] + 16 * u * St::P;
        const T* Ds = Qs + St::N;
        p[u] = row_product<T, HDP>(Qs, kf, n, g);
        dp[u] = row_product<T, HDP>(Ds, vf, n, g);
        const float4 l4 = *reinterpret_cast<const float4*>(&rowv[buf][0][16 * u + 4 * g]);
        const float4 d4 = *reinterpret_cast<const float4*>(&rowv[buf][1][16 * u + 4 * g]);
        const float lr[4] = {l4.x, l4.y, l4.z, l4.w}, dr[4] = {d4.x, d4.y, d4.z, d4.w};
#pragma unroll
        for (int r = 0; r < 4; ++r) {
          float e = __builtin_amdgcn_exp2f(fmaf(p[u][r], scale_log2, -lr[r]));
          if (!plain) {
            const int s = q0 + 16 * u + 4 * g + r;
            const bool see = mode == HYDRA_MASK_REFERENCE_SDPA ? s < kbnd : key <= s;
            e = see ? e : 0.f;
          }
          p[u][r] = e;
          dp[u][r] = e * (dp[u][r] - dr[r]);
        }
        if constexpr (sizeof(T) == 4) {
          col_product<HDP>(dva, Ds, p[u], n, g);
          col_product<HDP>(dka, Qs, dp[u], n, g);
        }
      }
      if constexpr (sizeof(T) == 2) {
        const T* Qs = smem[buf];
        prob_product<T, HDP>(dva, Qs + St::N, p, n, g);
        grad_product<T, HDP>(dka, Qs, Qs + 2 * St::N, dp, n, g);
      }
    }
    if (step + 1 < end) land(step + 1, buf ^ 1);
  }
  // The second walk.  Keys that are stored as zeros (padding) or not at all do
  // not count: their weights overflow where a query sees no key.
  if (__any(key < S && (!pad || keep) && (any_nan(dka) || any_nan(dva)))) {
#pragma unroll
    for (int t = 0; t < HDP / 16; ++t) dka[t] = dva[t] = f32x4{0.f, 0.f, 0.f, 0.f};
    for (int step = first; step < end; ++step) {
      const int hr = step / nq, row0 = kTile * (qt0 + step - hr * nq), h = kvh * G + hr;
#pragma unroll 1
      for (int s = row0; s < min(row0 + kTile, S); ++s) {
        const bool see = key < S && (mode == HYDRA_MASK_REFERENCE_SDPA ? s < kbnd : !walk || key <= s);
        if (!__any(see)) continue;
        const T* qr = q + b * qs.b + h * qs.h + s * qs.s;
        const T* dr = dout + b * ds.b + h * ds.h + s * ds.s;
        const int64_t ri = (static_cast<int64_t>(b) * Hq + h) * S + s;
        const float e = __builtin_amdgcn_exp2f(fmaf(row_dot<T, HDP>(qr, kf, g, hd), scale_log2, -lse2[ri]));
        const float grad = e * (row_dot<T, HDP>(dr, vf, g, hd) - dvec[ri]);
        if (!see) continue;
        add_row<T, HDP>(dva, dr, 1, e * kPScale<T>, g, hd);
        add_row<T, HDP>(dka, qr, 1, grad, g, hd);
      }
    }
  }
  if (pad && !keep) {
#pragma unroll
    for (int t = 0; t < HDP / 16; ++t) dka[t] = dva[t] = f32x4{0.f, 0.f, 0.f, 0.f};
  }
  if (maxch > 1) {  // summed by attn_bwd_f32_reduce_kernel
    const int64_t rows = static_cast<int64_t>(parts) * 64;  // of one chunk's partial
    float* pk = part + ((static_cast<int64_t>(c) * 2) * rows + (static_cast<int64_t>(rest) * 64 + 16 * wave + n)) * HDP;
    store_part<HDP>(pk, dka, 1.f, g);
    store_part<HDP>(pk + rows * HDP, dva, 1.f / kPScale<T>, g);
  } else if (key < S) {
    store_rows<T, HDP>(dk + b * dks.b + kvh * dks.h + static_cast<int64_t>(key) * dks.s, dka, scale, g, hd);
    store_rows<T, HDP>(dv + b * dvs.b + kvh * dvs.h + static_cast<int64_t>(key) * dvs.s, dva, 1.f / kPScale<T>, g, hd);
  }
}

// dQ: a workgroup takes an item and a chunk of its key tiles.
template <typename T, int HDP>
__global__ __launch_bounds__(kThreads) void attn_bwd_f32_dq_kernel(
    const T* __restrict__ q, const T* __restrict__ k, const T* __restrict__ v, const T* __restrict__ dout,
    const float* __restrict__ dvec, const float* __restrict__ lse2, const uint8_t* __restrict__ kmask, int mode,
    T* __restrict__ dq, float* __restrict__ part, int Hq, int Hkv, int S, int hd, int G, int BHkv, int ntasks,
    int items, int ch, int maxch, Strides3 qs, Strides3 ks, Strides3 vs, Strides3 ds, Strides3 dqs, int causal, int vec,
    float scale_log2, float scale) {
  using St = Stage<T, HDP>;
  constexpr int NT = kPlaneTiles<T> ? 4 : 2;  // K, V, K's planes
  __shared__ __attribute__((aligned(16))) T smem[2][NT * St::N];
  __shared__ int keepv[2][kTile];
  const int tid = threadIdx.x, lane = tid & 63, n = lane & 15, g = lane >> 4;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const bool walk = causal && mode != HYDRA_MASK_REFERENCE_SDPA;
  int bk, item, c;
  if (!locate(blockIdx.x, BHkv, items, ch, [&](int i) { return k_tiles(i, ntasks, G, S, walk); }, bk, item, c)) return;
  bk = __builtin_amdgcn_readfirstlane(bk);
  item = __builtin_amdgcn_readfirstlane(item);
  c = __builtin_amdgcn_readfirstlane(c);
  const int parts = BHkv * items;
  const int b = bk / Hkv, kvh = bk - b * Hkv;
  const int nt = k_tiles(item, ntasks, G, S, walk);
  const int first = c * ch, end = min(first + ch, nt);
  const Task tk = task_of(kWaves * item + wave, ntasks, kvh, G);
  const int qi = tk.q0 + n;
  const bool qok = tk.active && qi < S;
  const int my_end = !tk.active ? 0 : walk ? min(tk.q0 + 16, S) : S;
  typename Row16<T, HDP>::Run qf[Row16<T, HDP>::N], of[Row16<T, HDP>::N];
  const int64_t qr = qok ? qi : 0;
  load_frag<T, HDP>(q + b * qs.b + tk.h * qs.h + qr * qs.s, qf, g, hd, qok, vec & 2);
  load_frag<T, HDP>(dout + b * ds.b + tk.h * ds.h + qr * ds.s, of, g, hd, qok, vec & 2);
  float l2 = 0.f, dd = 0.f;
  if (qok) {
    const int64_t ri = (static_cast<int64_t>(b) * Hq + tk.h) * S + qi;
    l2 = lse2[ri];
    dd = dvec[ri];
  }
  f32x4 acc[HDP / 16];
#pragma unroll
  for (int t = 0; t < HDP / 16; ++t) acc[t] = f32x4{0.f, 0.f, 0.f, 0.f};
  const Rows<T> kr{k + b * ks.b + kvh * ks.h, ks.s, 1};
  const Rows<T> vr{v + b * vs.b + kvh * vs.h, vs.s, 1};
  St sk, sv;
  int kp = 0;
  auto fetch = [&](int t) {
    if (vec & 1) {
      sk.fetch(kr, kTile * t, S, tid);
      sv.fetch(vr, kTile * t, S, tid);
    }
    if (mode != HYDRA_MASK_NONE && tid < kTile) {
      const int key = kTile * t + tid;
      kp = key < S ? kmask[static_cast<int64_t>(b) * S + key] : 0;
    }
  };
  auto land = [&](int t, int buf) {
    T* planes = kPlaneTiles<T> ? smem[buf] + 2 * St::N : nullptr;
    if (vec & 1) {
      sk.land(smem[buf], planes, tid);
      sv.land(smem[buf] + St::N, nullptr, tid);
    } else {
      St::direct(kr, kTile * t, S, hd, smem[buf], planes, tid);
      St::direct(vr, kTile * t, S, hd, smem[buf] + St::N, nullptr, tid);
    }
    if (mode != HYDRA_MASK_NONE && tid < kTile) keepv[buf][tid] = kp;
  };
  fetch(first);
  land(first, 0);
  for (int t = first; t < end; ++t) {
    __syncthreads();
    const int buf = (t - first) & 1, t0 = kTile * t;
    if (t + 1 < end) fetch(t + 1);
    if (t0 < my_end) {
      const bool plain = mode == HYDRA_MASK_NONE && t0 + kTile - 1 <= (walk ? tk.q0 : S - 1) && t0 + kTile <= S;
      f32x4 dp[2];
#pragma unroll
      for (int u = 0; u < 2; ++u) {
        const T* Ks = smem[buf] + 16 * u * St::P;
        const T* Vs = Ks + St::N;
        const f32x4 p = row_product<T, HDP>(Ks, qf, n, g);
        dp[u] = row_product<T, HDP>(Vs, of, n, g);
#pragma unroll
        for (int r = 0; r < 4; ++r) {
          float e = __builtin_amdgcn_exp2f(fmaf(p[r], scale_log2, -l2));
          if (!plain) {
            const int i = 16 * u + 4 * g + r, key = t0 + i;
            const bool keep = mode == HYDRA_MASK_NONE || keepv[buf][i] != 0;
            e = key < S && sees(qi, key, keep, causal, mode) ? e : 0.f;
          }
          dp[u][r] = e * (dp[u][r] - dd);
        }
        if constexpr (sizeof(T) == 4) col_product<HDP>(acc, Ks, dp[u], n, g);
      }
      if constexpr (sizeof(T) == 2) {
        const T* Ks = smem[buf];
        grad_product<T, HDP>(acc, Ks, Ks + 2 * St::N, dp, n, g);
      }
    }
    if (t + 1 < end) land(t + 1, buf ^ 1);
  }
  if (__any(qok && any_nan(acc))) {  // the second walk
#pragma unroll
    for (int t = 0; t < HDP / 16; ++t) acc[t] = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll 1
    for (int key = kTile * first; key < min(kTile * end, S); ++key) {
      const bool keep = mode == HYDRA_MASK_NONE || kmask[static_cast<int64_t>(b) * S + key] != 0;
      const bool see = qok && sees(qi, key, keep, causal, mode);
      if (!__any(see)) continue;
      const T* krow = kr.base + key * kr.rs;
      const float e = __builtin_amdgcn_exp2f(fmaf(row_dot<T, HDP>(krow, qf, g, hd), scale_log2, -l2));
      const float grad = e * (row_dot<T, HDP>(vr.base + key * vr.rs, of, g, hd) - dd);
      if (see) add_row<T, HDP>(acc, krow, 1, grad, g, hd);
    }
  }
  if (maxch > 1) {
    const int64_t rows = static_cast<int64_t>(parts) * 64;
    store_part<HDP>(part + (static_cast<int64_t>(c) * rows + (static_cast<int64_t>(bk) * items + item) * 64 + 16 * wave + n) * HDP,
                    acc, 1.f, g);
  } else if (qok) {
    store_rows<T, HDP>(dq + b * dqs.b + tk.h * dqs.h + static_cast<int64_t>(qi) * dqs.s, acc, scale, g, hd);
  }
}

// Chunk partials in chunk order -> one gradient row per thread group of
// HDP / 4 threads.  which: 0 dk, 1 dv, 2 dq (blockIdx.y + first).
struct ReduceArgs {
  const float *pkv, *pq;
  void *dk, *dv, *dq;
  Strides3 dks, dvs, dqs;
  int Hq, Hkv, S, hd, G, ntasks, items, nkg, BHkv;
  int ch_kv, max_kv, ch_q, max_q;
  int walk;
  float scale;
};
template <typename T, int HDP>
__global__ __launch_bounds__(256) void attn_bwd_f32_reduce_kernel(ReduceArgs a, int first) {
  constexpr int TPR = HDP / 4;
  const int which = first + blockIdx.y;
  const int64_t i = (static_cast<int64_t>(blockIdx.x) * 256 + threadIdx.x) / TPR;
  const int d = 4 * (threadIdx.x % TPR);
  const int64_t rows = static_cast<int64_t>(a.BHkv) * (which == 2 ? a.items : a.nkg) * 64;
  if (i >= rows) return;
  const int j = static_cast<int>(i / 64), w = static_cast<int>(i % 64);  // tile of 64 rows, row in it
  T* out;
  const float* p;
  int nch;
  int64_t step;
  if (which == 2) {
    const int item = j % a.items, bk = j / a.items, b = bk / a.Hkv, kvh = bk - b * a.Hkv;
    const int task = kWaves * item + w / 16;
    if (task >= a.ntasks) return;
    const int row = 16 * (task / a.G) + w % 16, h = kvh * a.G + task % a.G;
    if (row >= a.S) return;
    nch = (k_tiles(item, a.ntasks, a.G, a.S, a.walk) + a.ch_q - 1) / a.ch_q;
    p = a.pq + i * HDP + d;
    step = rows * HDP;
    out = static_cast<T*>(a.dq) + b * a.dqs.b + h * a.dqs.h + static_cast<int64_t>(row) * a.dqs.s;
  } else {
    const int kg = j % a.nkg, bk = j / a.nkg, b = bk / a.Hkv, kvh = bk - b * a.Hkv;
    const int row = 64 * kg + w;
    if (row >= a.S) return;
    nch = (a.G * q_tiles(kg, a.S, a.walk) + a.ch_kv - 1) / a.ch_kv;
    p = a.pkv + (which * rows + i) * HDP + d;
    step = 2 * rows * HDP;
    const Strides3& s = which ? a.dvs : a.dks;
    out = static_cast<T*>(which ? a.dv : a.dk) + b * s.b + kvh * s.h + static_cast<int64_t>(row) * s.s;
  }
  float4 sum = make_float4(0.f, 0.f, 0.f, 0.f);
#pragma unroll 4
  for (int c = 0; c < nch; ++c) {
    const float4 x = *reinterpret_cast<const float4*>(p + c * step);
    sum.x += x.x; sum.y += x.y; sum.z += x.z; sum.w += x.w;
  }
  const float f = which == 1 ? 1.f : a.scale;
  const float o[4] = {sum.x * f, sum.y * f, sum.z * f, sum.w * f};
#pragma unroll
  for (int r = 0; r < 4; ++r)
    if (d + r < a.hd) out[d + r] = from_f32<T>(o[r]);
}

// How the walks are cut: chunks of equally many tiles, about kRounds times as
// many workgroups as are resident at once (none shorter than kMinTiles), so
// that the dispatcher evens out what causality and partial chunks leave uneven.
// One exact round left the CUs idle 30% (dK/dV) to 50% (dQ) of the launch at
// fp32 B4 8/2 heads x 64, S 2048; the partials of three rounds cost ~30 us of
// HBM there (dK/dV 481 -> 363 us, dQ 499 -> 296).
struct Plan {
  int HDP, G, ntasks, items, nkg, BHkv;
  int ch_kv, max_kv, ch_q, max_q;
  int64_t wg_kv, wg_q;  // workgroups
  size_t kv_floats, q_floats;
};
constexpr int kMinTiles = 6, kRounds = 3;
// Workgroups of each backward kernel resident on a CU, by head_dim 16, 32, 64,
// 128: the fp32 kernels' (148 / 137 registers at head_dim 64).  The 16-bit ones
// (149 / 115) hold one or two fewer at head_dim 16 and one more dQ workgroup at
// 64: one table serves them, since it only scales how many chunks a walk gives.
constexpr int kKvPerCu[4] = {6, 5, 3, 2}, kQPerCu[4] = {7, 5, 3, 2};

// split = false: every walk whole (no partials).
Plan plan_of(int B, int Hq, int Hkv, int S, int hd, bool walk, bool split) {
  Plan p{};
  p.HDP = hd <= 16 ? 16 : hd <= 32 ? 32 : hd <= 64 ? 64 : 128;
  p.G = Hq / Hkv;
  p.BHkv = B * Hkv;
  p.ntasks = p.G * ((S + 15) / 16);
  p.items = (p.ntasks + kWaves - 1) / kWaves;
  p.nkg = (S + 63) / 64;
  const int all = (S + kTile - 1) / kTile;
  const int hi = p.HDP == 16 ? 0 : p.HDP == 32 ? 1 : p.HDP == 64 ? 2 : 3;
  // tiles(i): the walk of part i of n, the same in every (batch, kv head)
  auto cut = [&](int n, auto tiles, int longest, int per_cu, int* ch, int* nch, int64_t* wgs) {
    const int64_t slots = static_cast<int64_t>(per_cu) * device_cus();
    int64_t total = 0;
    for (int i = 0; i < n; ++i) total += tiles(i);
    const int64_t c = std::max<int64_t>((total * p.BHkv + kRounds * slots - 1) / (kRounds * slots), kMinTiles);
    *ch = split ? static_cast<int>(std::min<int64_t>(c, longest)) : longest;
    *nch = (longest + *ch - 1) / *ch;
    *wgs = 0;
    for (int i = 0; i < n; ++i) *wgs += (tiles(i) + *ch - 1) / *ch;
    *wgs *= p.BHkv;
  };
  cut(p.nkg, [&](int g) { return p.G * q_tiles(g, S, walk); }, p.G * all, kKvPerCu[hi], &p.ch_kv, &p.max_kv, &p.wg_kv);
  cut(p.items, [&](int i) { return k_tiles(i, p.ntasks, p.G, S, walk); }, all, kQPerCu[hi], &p.ch_q, &p.max_q, &p.wg_q);
  p.kv_floats = p.max_kv > 1 ? size_t(p.BHkv) * p.nkg * 64 * p.HDP * 2 * p.max_kv : 0;
  p.q_floats = p.max_q > 1 ? size_t(p.BHkv) * p.items * 64 * p.HDP * p.max_q : 0;
  return p;
}

Strides3 s3(const int64_t* s) { return Strides3{s[0], s[1], s[2]}; }

// 16-byte row loads: whole rows of HDP elements, aligned.
bool vec_ok(const void* p, const int64_t* s, int E) {
  return aligned16(p) && s[0] % E == 0 && s[1] % E == 0 && s[2] % E == 0 && s[3] == 1;
}

template <typename T, int HDP>
int launch_fwd(const AttnF32Args& a) {
  constexpr int E = 16 / int(sizeof(T));
  const int G = a.Hq / a.Hkv, ntasks = G * ((a.S + 15) / 16), items = (ntasks + kWaves - 1) / kWaves;
  const int vec = (a.hd == HDP && vec_ok(a.k, a.ks, E) && vec_ok(a.v, a.vs, E) ? 1 : 0) |
                  (a.hd == HDP && vec_ok(a.q, a.qs, E) ? 2 : 0);
  const int64_t blocks = static_cast<int64_t>(items) * a.B * a.Hkv;
  if (blocks >= (int64_t(1) << 31)) return fail(HYDRA_ERR_ARG, "attn_fwd: too many rows");
  // Key groups when the items are fewer than two per resident workgroup
  // (registers: 3 per CU at head_dim 64): the longest walk sets the time then.
  // Two groups at head_dim 128 (LDS), else four.  fp16 B2 8/2 x 64, S 1500
  // (376 items): 104 -> 71 us (33 with the 16-bit rows).
  constexpr int KG = HDP == 128 ? 2 : 4;
  constexpr int per_cu = HDP <= 32 ? 5 : HDP == 64 ? 3 : 2;
  const bool groups = blocks < 2 * int64_t(per_cu) * device_cus();
  auto kern = groups ? attn_fwd_f32_kernel<T, HDP, KG> : attn_fwd_f32_kernel<T, HDP, 1>;
  kern<<<dim3(static_cast<unsigned>(blocks)), kThreads * (groups ? KG : 1), 0, a.st>>>(
      static_cast<const T*>(a.q), static_cast<const T*>(a.k), static_cast<const T*>(a.v), static_cast<T*>(a.o),
      a.lse, a.kmask, a.mask_mode, a.Hq, a.Hkv, a.S, a.hd, G, ntasks, items, s3(a.qs), s3(a.ks), s3(a.vs), a.vs[3],
      s3(a.os), a.causal ? 1 : 0, vec, a.scale * kLog2eF);
  return check_launch("attn_fwd_f32_kernel");
}

template <typename T, int HDP>
int launch_bwd(const AttnF32Args& a, float* part, size_t part_bytes) {
  constexpr int E = 16 / int(sizeof(T));
  const bool walk = a.causal && a.mask_mode != HYDRA_MASK_REFERENCE_SDPA;
  Plan p = plan_of(a.B, a.Hq, a.Hkv, a.S, a.hd, walk, true);
  if ((p.kv_floats + p.q_floats) * sizeof(float) > part_bytes) p = plan_of(a.B, a.Hq, a.Hkv, a.S, a.hd, walk, false);
  const bool qv = a.hd == HDP && vec_ok(a.q, a.qs, E) && vec_ok(a.dout, a.dos, E);
  const bool kv = a.hd == HDP && vec_ok(a.k, a.ks, E) && vec_ok(a.v, a.vs, E);
  const float sl2 = a.scale * kLog2eF;
  if (p.wg_kv >= (int64_t(1) << 31) || p.wg_q >= (int64_t(1) << 31)) return fail(HYDRA_ERR_ARG, "attn_bwd: problem too large");
  const T* q = static_cast<const T*>(a.q);
  const T* k = static_cast<const T*>(a.k);
  const T* v = static_cast<const T*>(a.v);
  const T* d = static_cast<const T*>(a.dout);
  float* pq = part + p.kv_floats;
  attn_bwd_f32_dkdv_kernel<T, HDP><<<dim3(static_cast<unsigned>(p.wg_kv)), kThreads, 0, a.st>>>(
      q, k, v, d, a.dvec, a.lse2, a.kmask, a.mask_mode, static_cast<T*>(a.dk), static_cast<T*>(a.dv), part, a.Hq,
      a.Hkv, a.S, a.hd, p.G, p.BHkv, p.nkg, p.ch_kv, p.max_kv, s3(a.qs), s3(a.ks), s3(a.vs), s3(a.dos), s3(a.dks), s3(a.dvs),
      a.causal ? 1 : 0, (qv ? 1 : 0) | (kv ? 2 : 0), sl2, a.scale);
  if (int rc = check_launch("attn_bwd: f32 dkdv")) return rc;
  attn_bwd_f32_dq_kernel<T, HDP><<<dim3(static_cast<unsigned>(p.wg_q)), kThreads, 0, a.st>>>(
      q, k, v, d, a.dvec, a.lse2, a.kmask, a.mask_mode, static_cast<T*>(a.dq), pq, a.Hq, a.Hkv, a.S, a.hd, p.G,
      p.BHkv, p.ntasks, p.items, p.ch_q, p.max_q, s3(a.qs), s3(a.ks), s3(a.vs), s3(a.dos), s3(a.dqs), a.causal ? 1 : 0,
      (kv ? 1 : 0) | (qv ? 2 : 0), sl2, a.scale);
  if (int rc = check_launch("attn_bwd: f32 dq")) return rc;
  if (p.max_kv == 1 && p.max_q == 1) return HYDRA_OK;
  const ReduceArgs r{part, pq, a.dk, a.dv, a.dq, s3(a.dks), s3(a.dvs), s3(a.dqs), a.Hq, a.Hkv, a.S, a.hd, p.G,
                     p.ntasks, p.items, p.nkg, p.BHkv, p.ch_kv, p.max_kv, p.ch_q, p.max_q, walk ? 1 : 0, a.scale};
  // one launch for the gradients that were cut: dk and dv, dq, or all three
  const int first = p.max_kv > 1 ? 0 : 2, count = (p.max_kv > 1 ? 2 : 0) + (p.max_q > 1 ? 1 : 0);
  const int64_t rows = static_cast<int64_t>(p.BHkv) * 64 * std::max(p.max_kv > 1 ? p.nkg : 0, p.max_q > 1 ? p.items : 0);
  const int64_t blocks = (rows * (HDP / 4) + 255) / 256;
  if (blocks >= (int64_t(1) << 31)) return fail(HYDRA_ERR_ARG, "attn_bwd: problem too large");
  attn_bwd_f32_reduce_kernel<T, HDP><<<dim3(static_cast<unsigned>(blocks), count), 256, 0, a.st>>>(r, first);
  return check_launch("attn_bwd: f32 reduce");
}

}  // namespace

int attn_fwd_f32(const AttnF32Args& a) {
  return HYDRA_DISPATCH_DTYPE(a.dtype, T, [&] {
    if (a.hd <= 16) return launch_fwd<T, 16>(a);
    if (a.hd <= 32) return launch_fwd<T, 32>(a);
    if (a.hd <= 64) return launch_fwd<T, 64>(a);
    return launch_fwd<T, 128>(a);
  });
}

size_t attn_bwd_f32_workspace(int B, int Hq, int Hkv, int S, int hd, bool causal, int mask_mode) {
  const Plan p = plan_of(B, Hq, Hkv, S, hd, causal && mask_mode != HYDRA_MASK_REFERENCE_SDPA, true);
  return (p.kv_floats + p.q_floats) * sizeof(float);
}

int attn_bwd_f32(const AttnF32Args& a, float* part, size_t part_bytes) {
  return HYDRA_DISPATCH_DTYPE(a.dtype, T, [&] {
    if (a.hd <= 16) return launch_bwd<T, 16>(a, part, part_bytes);
    if (a.hd <= 32) return launch_bwd<T, 32>(a, part, part_bytes);
    if (a.hd <= 64) return launch_bwd<T, 64>(a, part, part_bytes);
    return launch_bwd<T, 128>(a, part, part_bytes);
  });
}

}  // namespace hydra
