// What the vision blocks do between their projections and the attention operators, one launch a direction:
//
//   polarity features (layers/polaformer.py:63-84): q / scale and (k + positional) / scale, positive and negative parts to a
//     learned power, the same-sign and opposite-sign pairings and the values as contiguous heads;
//   focused features (layers/focused_la.py:56-74): relu features cubed at constant length, the values, as contiguous heads;
//   rotary features (layers/mlla.py:74-81): elu + 1 of q and k, their 2-D rotation, the values, all as contiguous heads;
//   token interpolation (focused_la.py:88-91, polaformer.py:95-98): reduced values back to the queries' length;
//   keys weighted by a score of the token and both sides turned (layers/rala.py:60-69), on heads;
//   merged heads (polaformer.py:92-104, mlla.py:88-92): heads back to token rows, plus the convolution's rows, times a gate.
//
// All of it is elementwise on token rows and bound by HBM: a lane owns 16 bytes of channels of one token (the next lanes the
// next channels), everything is computed from them in fp32 and rounded once, and nothing between the projection's rows and the
// operator's heads is written.  bf16: polarity (64 x 28x28 x 256) 50 us features (257 MB, 5.1 TB/s), 75 + 9 us their gradients
// (385 MB, 5.1 TB/s), 19 + 33 us the merge; rotary (64 x 56x56 x 64) 33 us features (205 MB, 6.2 TB/s), 45 us gradients (283 MB,
// 6.3 TB/s).  Whole polarity and rotary blocks of 16-bit types with heads of 32 channels do not come here: fbla_rows.hip takes them
// from rows to rows.
#include <hip/hip_runtime.h>

#include <type_traits>

#include "fbla_kernels.h"

namespace fbla {
namespace blocks {

namespace {

constexpr int kThreads = 256;
typedef uint32_t u32x4 __attribute__((ext_vector_type(4)));
typedef float f32x4 __attribute__((ext_vector_type(4)));

template <typename T> struct Piece {
  static constexpr int kVec = 16 / sizeof(T);
  union {
    u32x4 w;
    T e[kVec];
  };
};
template <typename T> __device__ __forceinline__ Piece<T> load(const T* p) {
  Piece<T> v;
  v.w = *reinterpret_cast<const u32x4*>(p);
  return v;
}
template <typename T> __device__ __forceinline__ void store(T* p, const Piece<T>& v) {
  *reinterpret_cast<u32x4*>(p) = v.w;
}

// a^p for a >= 0, p >= 1.  16-bit results: the hardware's exp2 and log2, whose error (2^-22 of p log2 a) is far below the
// result's rounding; a result below 2^-126 is 0.
template <typename T> __device__ __forceinline__ float power_of(float a, float p) {
  if constexpr (sizeof(T) == 4) return powf(a, p);
  else return __builtin_amdgcn_exp2f(p * __builtin_amdgcn_logf(a));
}
template <typename T> __device__ __forceinline__ float exp_of(float x) {
  if constexpr (sizeof(T) == 4) return expf(x);
  else return __builtin_amdgcn_exp2f(x * 1.44269504088896341f);
}

// fp32 gradients are as far from exact as torch's operators leave them and no further: quotients are divided out there, and
// what torch rounds product by product and sums in a tree is kept and summed in 64 bits.  16-bit types, whose results' rounding
// is thousands of times that, multiply by reciprocals and sum in 32 bits.
template <typename T> using Sum = std::conditional_t<sizeof(T) == 4, double, float>;
template <typename T> __device__ __forceinline__ float divisor(T scale) { return sizeof(T) == 4 ? (float)scale : 1.f / (float)scale; }
template <typename T> __device__ __forceinline__ float over(float x, float divisor) {
  return sizeof(T) == 4 ? x / divisor : x * divisor;
}

// What the gradients of a^power need: slope = a^(power - 1), which is 1 for a power of 1 whatever a is, and rise = a^power
// ln a.  log2f, not the bare instruction: that takes a denormal for 0, whose logarithm would make a gradient NaN.  fp32:
// powf(a, power - 1) times a, the product unrounded, is as far from a^power as powf(a, power) (3.34e-8 and 3.48e-8 root mean
// square over a in (0, 3), powers 1 to 5), and a second powf costs 80 us at 64 x 28x28 x 256.
template <typename T> __device__ __forceinline__ void power_slope(float a, float power, float& slope, Sum<T>& rise) {
  if constexpr (sizeof(T) == 4) {
    slope = powf(a, power - 1.f);
    rise = (double)slope * a * logf(a);
  } else {
    const float l = log2f(a), p = power - 1.f;
    slope = p == 0.f ? 1.f : __builtin_amdgcn_exp2f(p * l);
    rise = slope * a * (l * 0.693147180559945309f);
  }
}

// first element of head row (b, h, t) of a [B, heads, n, width] tensor
__device__ __forceinline__ int64_t head_row(const Shape& s, uint32_t b, uint32_t h, uint32_t t, uint32_t n, int width) {
  return (((int64_t)b * s.heads + h) * n + t) * width;
}

// ---------------------------------------------------------------------------------------------------------------
// polarity features
// ---------------------------------------------------------------------------------------------------------------
template <typename T>
__device__ __forceinline__ void split_signs(const float (&y)[Piece<T>::kVec], const Piece<T>& power, Piece<T>& pos,
                                            Piece<T>& neg) {
#pragma unroll
  for (int j = 0; j < Piece<T>::kVec; ++j) {
    const float r = power_of<T>(fabsf(y[j]), (float)power.e[j]);
    pos.e[j] = (T)(y[j] < 0.f ? 0.f : r);  // NaN goes to both
    neg.e[j] = (T)(y[j] > 0.f ? 0.f : r);
  }
}

// pieces [0, q_pieces) are the queries' (gate half untouched), the others the keys' and values'
template <typename T>
__global__ __launch_bounds__(kThreads) void polarity_fwd_kernel(Shape s, Polarity<const T> a, T* __restrict__ q_same,
                                                                T* __restrict__ q_opp, T* __restrict__ k_both,
                                                                T* __restrict__ v_heads, uint32_t q_wgs) {
  constexpr int V = Piece<T>::kVec;
  const bool keys = blockIdx.x >= q_wgs;
  const uint32_t i = (keys ? blockIdx.x - q_wgs : blockIdx.x) * kThreads + threadIdx.x;
  const uint32_t pieces = s.heads * s.d / V, n = keys ? s.Nk : s.N;
  const uint32_t row = i / pieces, c = i % pieces * V;
  if (row >= (uint32_t)s.B * n) return;
  const uint32_t b = row / n, t = row % n, h = c / s.d, j0 = c % s.d, C = s.heads * s.d;
  const Piece<T> scale = load(a.scale + c), power = load(a.power + c);
  const T* src = (keys ? a.kv : a.qg) + (int64_t)row * 2 * C + c;
  const Piece<T> x = load(src);
  float y[V];
#pragma unroll
  for (int j = 0; j < V; ++j) y[j] = (float)x.e[j];
  if (keys) {
    const Piece<T> pe = load(a.pe + (int64_t)t * C + c), v = load(src + C);
#pragma unroll
    for (int j = 0; j < V; ++j) y[j] += (float)pe.e[j];
    store(v_heads + head_row(s, b, h, t, n, s.d) + j0, v);
  }
#pragma unroll
  for (int j = 0; j < V; ++j) y[j] /= (float)scale.e[j];
  Piece<T> pos, neg;
  split_signs<T>(y, power, pos, neg);
  const int64_t at = head_row(s, b, h, t, n, 2 * s.d) + j0;
  if (keys) {
    store(k_both + at, pos);
    store(k_both + at + s.d, neg);
  } else {
    store(q_same + at, pos);
    store(q_same + at + s.d, neg);
    store(q_opp + at, neg);
    store(q_opp + at + s.d, pos);
  }
}

// One piece's gradients: dx = the gradient of x (q, or k and its positional term alike), added to `dscale` the gradient of
// -scale * scale, to `dpower` that of the power.
template <typename T>
__device__ __forceinline__ void polarity_piece_bwd(const float (&x)[Piece<T>::kVec], const float (&scale)[Piece<T>::kVec],
                                                   const float (&power)[Piece<T>::kVec], const float (&gpos)[Piece<T>::kVec],
                                                   const float (&gneg)[Piece<T>::kVec], float (&dx)[Piece<T>::kVec],
                                                   Sum<T> (&dscale)[Piece<T>::kVec], Sum<T> (&dpower)[Piece<T>::kVec]) {
  using A = Sum<T>;
#pragma unroll
  for (int j = 0; j < Piece<T>::kVec; ++j) {
    const float y = over<T>(x[j], scale[j]), a = fabsf(y);
    const float gp = y < 0.f ? 0.f : gpos[j], gn = y > 0.f ? 0.f : gneg[j];  // (NaN is in both parts)
    float slope;
    A rise;
    power_slope<T>(a, power[j], slope, rise);
    const bool zero = a == 0.f;  // both parts are cut off there: no gradient
    const A dy = zero ? A(0) : (A)(gp - gn) * power[j] * slope;
    dx[j] = over<T>((float)dy, scale[j]);
    dscale[j] += dy * x[j];
    dpower[j] += zero ? A(0) : (A)(gp + gn) * rise;
  }
}

// Workgroup = `lanes` pieces of channels (at most 64, blockIdx.y picks them) times kThreads / lanes rows; it walks rows
// gridDim.x apart and keeps the sums over tokens (gradients of scale and power) in registers.  Workgroups [0, q_wgs) take the
// queries, the others the keys: rows there are (token, batch group), a lane adds its token's gradients over the batches of the
// group (gradient of the positional term).  partial: [workgroup][2][C], pe_partial: [group][Nk][C].
template <typename T>
__global__ __launch_bounds__(kThreads) void polarity_bwd_kernel(Shape s, Polarity<const T> a, PolarityGrads<const T> g,
                                                                T* __restrict__ dqg, T* __restrict__ dkv,
                                                                float* __restrict__ partial, float* __restrict__ pe_partial,
                                                                int q_wgs, int groups) {
  constexpr int V = Piece<T>::kVec;
  const int C = s.heads * s.d, pieces = C / V;
  const int lanes = min(pieces - (int)blockIdx.y * 64, 64), rows = kThreads / lanes;
  const int lane = threadIdx.x % lanes, r = threadIdx.x / lanes;
  const bool keys = (int)blockIdx.x >= q_wgs;
  const uint32_t wg = keys ? blockIdx.x - q_wgs : blockIdx.x, wgs = keys ? gridDim.x - q_wgs : q_wgs;
  const int c = (blockIdx.y * 64 + lane) * V, h = c / s.d, j0 = c % s.d;
  Sum<T> dscale[V], dpower[V];
  float scale[V], power[V];
  {
    const Piece<T> sc = load(a.scale + c), pw = load(a.power + c);
#pragma unroll
    for (int j = 0; j < V; ++j) {
      dscale[j] = dpower[j] = 0;
      scale[j] = divisor<T>(sc.e[j]);
      power[j] = (float)pw.e[j];
    }
  }
  if (r < rows && !keys) {
    const uint32_t total = (uint32_t)s.B * s.N;
    for (uint32_t row = wg * rows + r; row < total; row += wgs * rows) {
      const uint32_t b = row / s.N, t = row % s.N;
      const int64_t at = head_row(s, b, h, t, s.N, 2 * s.d) + j0;
      const Piece<T> x = load(a.qg + (int64_t)row * 2 * C + c);
      const Piece<T> s0 = load(g.q_same + at), s1 = load(g.q_same + at + s.d), o0 = load(g.q_opp + at),
                     o1 = load(g.q_opp + at + s.d), gate = load(g.gate + (int64_t)row * C + c);
      float xf[V], gpos[V], gneg[V], dx[V];
#pragma unroll
      for (int j = 0; j < V; ++j) {
        xf[j] = (float)x.e[j];
        gpos[j] = (float)s0.e[j] + (float)o1.e[j];
        gneg[j] = (float)s1.e[j] + (float)o0.e[j];
      }
      polarity_piece_bwd<T>(xf, scale, power, gpos, gneg, dx, dscale, dpower);
      Piece<T> out;
#pragma unroll
      for (int j = 0; j < V; ++j) out.e[j] = (T)dx[j];
      T* to = dqg + (int64_t)row * 2 * C + c;
      store(to, out);
      store(to + C, gate);
    }
  }
  if (r < rows && keys) {
    const uint32_t total = (uint32_t)s.Nk * groups;
    for (uint32_t item = wg * rows + r; item < total; item += wgs * rows) {
      const uint32_t t = item / groups, group = item % groups;
      const Piece<T> pe = load(a.pe + (int64_t)t * C + c);
      float dpe[V];
#pragma unroll
      for (int j = 0; j < V; ++j) dpe[j] = 0.f;
      for (uint32_t b = group; b < (uint32_t)s.B; b += groups) {
        const int64_t row = (int64_t)b * s.Nk + t, at = head_row(s, b, h, t, s.Nk, 2 * s.d) + j0;
        const Piece<T> x = load(a.kv + row * 2 * C + c);
        const Piece<T> g0 = load(g.k_both + at), g1 = load(g.k_both + at + s.d),
                       vh = load(g.v_heads + head_row(s, b, h, t, s.Nk, s.d) + j0), vr = load(g.v_rows + row * C + c);
        float xf[V], gpos[V], gneg[V], dx[V];
#pragma unroll
        for (int j = 0; j < V; ++j) {
          xf[j] = (float)x.e[j] + (float)pe.e[j];
          gpos[j] = (float)g0.e[j];
          gneg[j] = (float)g1.e[j];
        }
        polarity_piece_bwd<T>(xf, scale, power, gpos, gneg, dx, dscale, dpower);
        Piece<T> out, v;
#pragma unroll
        for (int j = 0; j < V; ++j) {
          out.e[j] = (T)dx[j];
          dpe[j] += dx[j];
          v.e[j] = (T)((float)vh.e[j] + (float)vr.e[j]);
        }
        T* to = dkv + row * 2 * C + c;
        store(to, out);
        store(to + C, v);
      }
      float* to = pe_partial + ((int64_t)group * s.Nk + t) * C + c;
#pragma unroll
      for (int j = 0; j < V; j += 4) *reinterpret_cast<f32x4*>(to + j) = f32x4{dpe[j], dpe[j + 1], dpe[j + 2], dpe[j + 3]};
    }
  }
  // the rows of the workgroup, in order
  __shared__ Sum<T> sums[kThreads * V];
  float* out = partial + (int64_t)blockIdx.x * 2 * C;
#pragma unroll
  for (int which = 0; which < 2; ++which) {
    __syncthreads();
    if (r < rows)
#pragma unroll
      for (int j = 0; j < V; ++j) sums[(r * lanes + lane) * V + j] = which ? dpower[j] : dscale[j];
    __syncthreads();
    for (int i = threadIdx.x; i < lanes * V; i += kThreads) {
      Sum<T> v = 0;
      for (int q = 0; q < rows; ++q) v += sums[q * lanes * V + i];
      out[which * C + blockIdx.y * 64 * V + i] = (float)v;
    }
  }
}

// Sums over the partials in order, four neighbouring results per lane, 16 lanes of a column; workgroups [0, stat_wgs): the
// `stats` C sums of the scale (times its reciprocal square or, `by` 1, its reciprocal) and the power, the others the Nk C
// sums of the positional term.
template <typename T>
__global__ __launch_bounds__(kThreads) void features_finish_kernel(int C, int stats_of, int by, int wgs, const float* __restrict__ partial,
                                                                   const T* __restrict__ scale, const T* __restrict__ raw_power,
                                                                   float alpha, T* __restrict__ dscale, T* __restrict__ dpower, int stat_wgs, int groups,
                                                                   int64_t pe_count, const float* __restrict__ pe_partial,
                                                                   T* __restrict__ dpe) {
  constexpr int kParts = 16, kLanes = kThreads / kParts;
  using A = Sum<T>;
  __shared__ A sums[kParts][kLanes][4];
  const bool stats = (int)blockIdx.x < stat_wgs;
  const int lane = threadIdx.x % kLanes, part = threadIdx.x / kLanes;
  const int64_t at = ((int64_t)(stats ? blockIdx.x : blockIdx.x - stat_wgs) * kLanes + lane) * 4;
  const int64_t count = stats ? (int64_t)stats_of * C : pe_count;
  const int terms = stats ? wgs : groups;
  const float* src = stats ? partial : pe_partial;
  A sum[4] = {0, 0, 0, 0};
  if (at < count)
#pragma unroll 4
    for (int i = part; i < terms; i += kParts) {
      const f32x4 v = *reinterpret_cast<const f32x4*>(src + (int64_t)i * count + at);
#pragma unroll
      for (int j = 0; j < 4; ++j) sum[j] += v[j];
    }
#pragma unroll
  for (int j = 0; j < 4; ++j) sums[part][lane][j] = sum[j];
  __syncthreads();
  if (part != 0 || at >= count) return;
  for (int i = 1; i < kParts; ++i)
#pragma unroll
    for (int j = 0; j < 4; ++j) sum[j] += sums[i][lane][j];
#pragma unroll
  for (int j = 0; j < 4; ++j) {
    const int64_t c = at + j;
    if (!stats) dpe[c] = (T)sum[j];
    else if (c >= C) {
      const float s = raw_power ? sigmoid((float)raw_power[c - C]) : 0.f;
      dpower[c - C] = (T)(raw_power ? sum[j] * (A)(alpha * s * (1.f - s)) : sum[j]);
    } else {
      const float p = (float)scale[c];
      const A inv = A(1) / (A)(raw_power ? softplus(p) : p), d = by == 1 ? -sum[j] * inv : -sum[j] * inv * inv;
      dscale[c] = (T)(raw_power ? d * (A)sigmoid(p) : d);
    }
  }
}

// ---------------------------------------------------------------------------------------------------------------
// rotary features
// ---------------------------------------------------------------------------------------------------------------
template <typename T> __device__ __forceinline__ float phi(float x) { return x > 0.f ? x + 1.f : exp_of<T>(x); }

// cos and sin of the piece's channel pairs: rot [N][rot_channels / 2][2]
template <typename T>
__device__ __forceinline__ void load_rotation(const float* __restrict__ rot, int rot_channels, uint32_t t, uint32_t c,
                                              float (&cs)[Piece<T>::kVec]) {
  const float* p = rot + (int64_t)t * rot_channels + c % rot_channels;
#pragma unroll
  for (int j = 0; j < Piece<T>::kVec; j += 4) {
    const f32x4 v = *reinterpret_cast<const f32x4*>(p + j);
#pragma unroll
    for (int e = 0; e < 4; ++e) cs[j + e] = v[e];
  }
}

template <typename T>
__global__ __launch_bounds__(kThreads) void rotary_fwd_kernel(Shape s, const T* __restrict__ qk, const T* __restrict__ x,
                                                              const float* __restrict__ rot, int rot_channels,
                                                              T* __restrict__ q, T* __restrict__ k, T* __restrict__ q_rot,
                                                              T* __restrict__ k_rot, T* __restrict__ v) {
  constexpr int V = Piece<T>::kVec;
  const uint32_t C = s.heads * s.d, pieces = C / V, i = blockIdx.x * kThreads + threadIdx.x;
  const uint32_t row = i / pieces, c = i % pieces * V;
  if (row >= (uint32_t)s.B * s.N) return;
  const uint32_t b = row / s.N, t = row % s.N;
  const Piece<T> in[2] = {load(qk + (int64_t)row * 2 * C + c), load(qk + (int64_t)row * 2 * C + C + c)};
  const Piece<T> vin = load(x + (int64_t)row * C + c);
  float cs[V];
  load_rotation<T>(rot, rot_channels, t, c, cs);
  const int64_t at = head_row(s, b, c / s.d, t, s.N, s.d) + c % s.d;
#pragma unroll
  for (int w = 0; w < 2; ++w) {
    Piece<T> plain, turned;
#pragma unroll
    for (int j = 0; j < V; j += 2) {
      const float re = phi<T>((float)in[w].e[j]), im = phi<T>((float)in[w].e[j + 1]);
      plain.e[j] = (T)re;
      plain.e[j + 1] = (T)im;
      turned.e[j] = (T)(re * cs[j] - im * cs[j + 1]);
      turned.e[j + 1] = (T)(re * cs[j + 1] + im * cs[j]);
    }
    store((w ? k : q) + at, plain);
    store((w ? k_rot : q_rot) + at, turned);
  }
  store(v + at, vin);
}

template <typename T>
__global__ __launch_bounds__(kThreads) void rotary_bwd_kernel(Shape s, const T* __restrict__ qk,
                                                              const float* __restrict__ rot, int rot_channels,
                                                              RotaryGrads<const T> g, T* __restrict__ dqk,
                                                              T* __restrict__ dx) {
  constexpr int V = Piece<T>::kVec;
  const uint32_t C = s.heads * s.d, pieces = C / V, i = blockIdx.x * kThreads + threadIdx.x;
  const uint32_t row = i / pieces, c = i % pieces * V;
  if (row >= (uint32_t)s.B * s.N) return;
  const uint32_t b = row / s.N, t = row % s.N;
  const int64_t at = head_row(s, b, c / s.d, t, s.N, s.d) + c % s.d, from = (int64_t)row * 2 * C + c;
  const Piece<T> in[2] = {load(qk + from), load(qk + from + C)};
  const Piece<T> plain[2] = {load(g.q + at), load(g.k + at)}, turned[2] = {load(g.q_rot + at), load(g.k_rot + at)};
  const Piece<T> vh = load(g.v + at), vr = load(g.v_rows + (int64_t)row * C + c);
  float cs[V];
  load_rotation<T>(rot, rot_channels, t, c, cs);
#pragma unroll
  for (int w = 0; w < 2; ++w) {
    Piece<T> out;
#pragma unroll
    for (int j = 0; j < V; j += 2) {
      const float gre = (float)turned[w].e[j], gim = (float)turned[w].e[j + 1];
      const float re = (float)plain[w].e[j] + gre * cs[j] + gim * cs[j + 1];
      const float im = (float)plain[w].e[j + 1] + gim * cs[j] - gre * cs[j + 1];
      const float x0 = (float)in[w].e[j], x1 = (float)in[w].e[j + 1];
      out.e[j] = (T)(x0 > 0.f ? re : re * exp_of<T>(x0));
      out.e[j + 1] = (T)(x1 > 0.f ? im : im * exp_of<T>(x1));
    }
    store(dqk + from + (w ? C : 0), out);
  }
  Piece<T> v;
#pragma unroll
  for (int j = 0; j < V; ++j) v.e[j] = (T)((float)vh.e[j] + (float)vr.e[j]);
  store(dx + (int64_t)row * C + c, v);
}

// Keys weighted per token and both sides turned, on heads (layers/rala.py:60-69): k_out = k * weight, q_rot = R q,
// k_rot = R k_out; weight [B, heads, N].  32 x 28x28 x 256 in bf16: 12 us forward, 15 us backward; torch's products,
// complex products in fp32 and copies 58 and 150 us.
template <typename T>
__device__ __forceinline__ void turn(const float (&x)[Piece<T>::kVec], const float (&cs)[Piece<T>::kVec], float sign,
                                     float (&out)[Piece<T>::kVec]) {
#pragma unroll
  for (int j = 0; j < Piece<T>::kVec; j += 2) {
    out[j] = x[j] * cs[j] - sign * x[j + 1] * cs[j + 1];
    out[j + 1] = x[j + 1] * cs[j] + sign * x[j] * cs[j + 1];
  }
}
template <typename T> __device__ __forceinline__ Piece<T> rounded(const float (&x)[Piece<T>::kVec]) {
  Piece<T> out;
#pragma unroll
  for (int j = 0; j < Piece<T>::kVec; ++j) out.e[j] = (T)x[j];
  return out;
}

template <typename T>
__global__ __launch_bounds__(kThreads) void turn_fwd_kernel(Shape s, const T* __restrict__ q, const T* __restrict__ k,
                                                            const T* __restrict__ weight, const float* __restrict__ rot,
                                                            T* __restrict__ k_out, T* __restrict__ q_rot,
                                                            T* __restrict__ k_rot) {
  constexpr int V = Piece<T>::kVec;
  const uint32_t pieces = s.d / V, i = blockIdx.x * kThreads + threadIdx.x;
  const uint32_t row = i / pieces, j0 = i % pieces * V;
  if (row >= (uint32_t)s.B * s.heads * s.N) return;
  const int64_t at = (int64_t)row * s.d + j0;
  const Piece<T> qi = load(q + at), ki = load(k + at);
  const float w = (float)weight[row];
  float cs[V], qf[V], kf[V], out[V];
  load_rotation<T>(rot, s.d, row % s.N, j0, cs);
#pragma unroll
  for (int j = 0; j < V; ++j) {
    qf[j] = (float)qi.e[j];
    kf[j] = (float)ki.e[j] * w;
  }
  store(k_out + at, rounded<T>(kf));
  turn<T>(qf, cs, 1.f, out);
  store(q_rot + at, rounded<T>(out));
  turn<T>(kf, cs, 1.f, out);
  store(k_rot + at, rounded<T>(out));
}

// dq = R^T dq_rot, dk = weight (dk_out + R^T dk_rot), dweight = the sum of k (dk_out + R^T dk_rot) over the d / V lanes of a
// row (a power of two up to 64)
template <typename T>
__global__ __launch_bounds__(kThreads) void turn_bwd_kernel(Shape s, const T* __restrict__ k, const T* __restrict__ weight,
                                                            const float* __restrict__ rot, const T* __restrict__ dk_out,
                                                            const T* __restrict__ dq_rot, const T* __restrict__ dk_rot,
                                                            T* __restrict__ dq, T* __restrict__ dk, T* __restrict__ dweight) {
  constexpr int V = Piece<T>::kVec;
  const uint32_t pieces = s.d / V, i = blockIdx.x * kThreads + threadIdx.x;
  const uint32_t row = i / pieces, j0 = i % pieces * V;
  const bool real = row < (uint32_t)s.B * s.heads * s.N;
  float sum = 0.f;
  if (real) {
    const int64_t at = (int64_t)row * s.d + j0;
    const Piece<T> ki = load(k + at), g = load(dk_out + at), qr = load(dq_rot + at), kr = load(dk_rot + at);
    const float w = (float)weight[row];
    float cs[V], in[V], out[V];
    load_rotation<T>(rot, s.d, row % s.N, j0, cs);
#pragma unroll
    for (int j = 0; j < V; ++j) in[j] = (float)qr.e[j];
    turn<T>(in, cs, -1.f, out);
    store(dq + at, rounded<T>(out));
#pragma unroll
    for (int j = 0; j < V; ++j) in[j] = (float)kr.e[j];
    turn<T>(in, cs, -1.f, out);
#pragma unroll
    for (int j = 0; j < V; ++j) {
      out[j] += (float)g.e[j];
      sum = fmaf(out[j], (float)ki.e[j], sum);
      out[j] *= w;
    }
    store(dk + at, rounded<T>(out));
  }
  for (int m = 1; m < (int)pieces; m *= 2) sum += __shfl_xor(sum, m);
  if (real && j0 == 0) dweight[row] = (T)sum;
}

// ---------------------------------------------------------------------------------------------------------------
// merged heads
// ---------------------------------------------------------------------------------------------------------------
// Where the piece of channels c of token (b, t) lies in the heads: o [B, heads, N, d], or with o2 the channels of a head in
// two halves o, o2 [B, heads, N, d / 2].
template <typename T>
__device__ __forceinline__ T* head_piece(const Shape& s, T* o, T* o2, uint32_t b, uint32_t t, uint32_t c) {
  const uint32_t h = c / s.d, j = c % s.d;
  if (!o2) return o + head_row(s, b, h, t, s.N, s.d) + j;
  const uint32_t half = s.d / 2;
  return j < half ? o + head_row(s, b, h, t, s.N, half) + j : o2 + head_row(s, b, h, t, s.N, half) + j - half;
}

template <typename T>
__global__ __launch_bounds__(kThreads) void merge_fwd_kernel(Shape s, Merge<const T> a, T* __restrict__ out) {
  constexpr int V = Piece<T>::kVec;
  const uint32_t C = s.heads * s.d, pieces = C / V, i = blockIdx.x * kThreads + threadIdx.x;
  const uint32_t row = i / pieces, c = i % pieces * V;
  if (row >= (uint32_t)s.B * s.N) return;
  const Piece<T> o = load(head_piece<const T>(s, a.o, a.o2, row / s.N, row % s.N, c));
  const Piece<T> l = load(a.local + (int64_t)row * C + c);
  Piece<T> r;
#pragma unroll
  for (int j = 0; j < V; ++j) r.e[j] = (T)((float)o.e[j] + (float)l.e[j]);
  if (a.gate) {
    const Piece<T> gate = load(a.gate + (int64_t)row * a.gate_row + c);
#pragma unroll
    for (int j = 0; j < V; ++j) r.e[j] = (T)(((float)o.e[j] + (float)l.e[j]) * (float)gate.e[j]);
  }
  store(out + (int64_t)row * C + c, r);
}

// dlocal = dout * gate (also as heads), dgate = dout * (heads + local); without a gate dlocal is dout and is not written
template <typename T>
__global__ __launch_bounds__(kThreads) void merge_bwd_kernel(Shape s, Merge<const T> a, const T* __restrict__ dout,
                                                             T* __restrict__ d_o, T* __restrict__ d_o2,
                                                             T* __restrict__ dlocal, T* __restrict__ dgate) {
  constexpr int V = Piece<T>::kVec;
  const uint32_t C = s.heads * s.d, pieces = C / V, i = blockIdx.x * kThreads + threadIdx.x;
  const uint32_t row = i / pieces, c = i % pieces * V;
  if (row >= (uint32_t)s.B * s.N) return;
  const uint32_t b = row / s.N, t = row % s.N;
  const int64_t at = (int64_t)row * C + c;
  Piece<T> g = load(dout + at);
  if (a.gate) {
    const Piece<T> gate = load(a.gate + (int64_t)row * a.gate_row + c), l = load(a.local + at),
                   o = load(head_piece<const T>(s, a.o, a.o2, b, t, c));
    Piece<T> dg;
#pragma unroll
    for (int j = 0; j < V; ++j) {
      dg.e[j] = (T)((float)g.e[j] * ((float)o.e[j] + (float)l.e[j]));
      g.e[j] = (T)((float)g.e[j] * (float)gate.e[j]);
    }
    store(dgate + at, dg);
    store(dlocal + at, g);
  }
  store(head_piece<T>(s, d_o, d_o2, b, t, c), g);
}

// ---------------------------------------------------------------------------------------------------------------
// token interpolation
// ---------------------------------------------------------------------------------------------------------------
// Output token t of `to` lies at (t + 1/2) from / to - 1/2 between the input tokens (not before the first): token i0 with
// weight 1 - f, the next one (the last has none) with f.  Whole numbers: the place times 2 to is (2 t + 1) from - to.
struct Place {
  int i0;
  float f;
};
__device__ __forceinline__ Place place_of(int t, int from, int to) {
  const int at = max((2 * t + 1) * from - to, 0), i0 = min(at / (2 * to), from - 1);
  return {i0, (float)(at - i0 * 2 * to) / (float)(2 * to)};
}

// torch's kernels walk batch and channels in every thread (forward 7.2 ms, backward 252 ms for 64 x 196 -> 784 tokens of 256
// channels in fp16, read transposed); here a lane owns one output piece either way (10 and 12 us).
template <typename T>
__global__ __launch_bounds__(kThreads) void interpolate_fwd_kernel(const T* __restrict__ x, int64_t x_batch, int64_t x_row,
                                                                   int B, int from, int to, int C, T* __restrict__ y) {
  constexpr int V = Piece<T>::kVec;
  const uint32_t pieces = C / V, i = blockIdx.x * kThreads + threadIdx.x;
  const uint32_t row = i / pieces, c = i % pieces * V;
  if (row >= (uint32_t)B * to) return;
  const Place at = place_of(row % to, from, to);
  const T* src = x + (int64_t)(row / to) * x_batch + c;
  const Piece<T> a = load(src + at.i0 * x_row), b = load(src + min(at.i0 + 1, from - 1) * x_row);
  Piece<T> out;
#pragma unroll
  for (int j = 0; j < V; ++j) out.e[j] = (T)((1.f - at.f) * (float)a.e[j] + at.f * (float)b.e[j]);
  store(y + (int64_t)row * C + c, out);
}

// input token i takes part in the outputs whose place lies between i - 1 and i + 1
template <typename T>
__global__ __launch_bounds__(kThreads) void interpolate_bwd_kernel(const T* __restrict__ g, int B, int from, int to, int C,
                                                                   T* __restrict__ dx) {
  constexpr int V = Piece<T>::kVec;
  const uint32_t pieces = C / V, n = blockIdx.x * kThreads + threadIdx.x;
  const uint32_t row = n / pieces, c = n % pieces * V;
  if (row >= (uint32_t)B * from) return;
  const int i = row % from;
  // (2 t + 1) from - to > 2 to (i - 1)  and  < 2 to (i + 1), one token more on either side; the first and the last input
  // token also stand for what lies before and behind them
  const int first = i == 0 ? 0 : max((to * (2 * i - 1) - from) / (2 * from) - 1, 0);
  const int last = i == from - 1 ? to - 1 : min((to * (2 * i + 3) - from) / (2 * from) + 1, to - 1);
  const T* src = g + (int64_t)(row / from) * to * C + c;
  float sum[V];
#pragma unroll
  for (int j = 0; j < V; ++j) sum[j] = 0.f;
#pragma unroll 4
  for (int t = first; t <= last; ++t) {
    const Place at = place_of(t, from, to);
    const float w = (at.i0 == i ? 1.f - at.f : 0.f) + (min(at.i0 + 1, from - 1) == i ? at.f : 0.f);
    const Piece<T> v = load(src + (int64_t)t * C);
    if (w != 0.f)
#pragma unroll
      for (int j = 0; j < V; ++j) sum[j] = fmaf(w, (float)v.e[j], sum[j]);
  }
  Piece<T> out;
#pragma unroll
  for (int j = 0; j < V; ++j) out.e[j] = (T)sum[j];
  store(dx + (int64_t)row * C + c, out);
}

// ---------------------------------------------------------------------------------------------------------------
// rows that are normalised over all their channels
// ---------------------------------------------------------------------------------------------------------------
// `lanes` (a power of two, 8 .. 64) neighbouring lanes share a row, PER pieces each: piece p of lane l is piece p lanes + l.
// The row stays in registers between the sums and the result.
__device__ __forceinline__ float row_sum(float v, int lanes) {
  for (int m = 1; m < lanes; m *= 2) v += __shfl_xor(v, m);
  return v;
}
__device__ __forceinline__ float row_max(float v, int lanes) {
  for (int m = 1; m < lanes; m *= 2) v = fmaxf(v, __shfl_xor(v, m));
  return v;
}

// ---------------------------------------------------------------------------------------------------------------
// focused features (layers/focused_la.py:56-74)
// ---------------------------------------------------------------------------------------------------------------
// t = (relu(x) + 1e-6) / scale; the feature is t^3 brought to t's length over all channels of the token.  With s = t times
// the power of two that brings max t to [0.5, 1) (exact, and nothing under- or overflows) and n = |s|, m = |s^3|:
// feature = s^3 |t| / m, and for its gradient g, G = sum g s^3:
// dt = 3 n s^2 g / m + G (s / (n m) - 3 n s^5 / m^3).
// 64 x 28x28 x 256, bf16: 38 us (154 MB, 4 TB/s) and 83 + 9 us (231 MB, 2.8 TB/s); torch's operators 279 and 851 us.
// Rows of workgroup [0, q_wgs): the queries, the others the keys with the values beside them.
template <typename T> __device__ __forceinline__ float focus_input(float x, float scale) {
  return ((x < 0.f ? 0.f : x) + 1e-6f) / scale;
}
// exponent of the largest t, such that 2^-exponent and 2^exponent are numbers
__device__ __forceinline__ int focus_exponent(float top) { return min(max(__builtin_amdgcn_frexp_expf(top), -126), 126); }

template <typename T, int PER>
__global__ __launch_bounds__(kThreads) void focus_fwd_kernel(Shape s, Focus<const T> a, int lanes, unsigned q_wgs,
                                                             T* __restrict__ q_out, T* __restrict__ k_out,
                                                             T* __restrict__ v_out) {
  constexpr int V = Piece<T>::kVec;
  const bool keys = blockIdx.x >= q_wgs;
  const int lane = threadIdx.x % lanes, per_wg = kThreads / lanes, C = s.heads * s.d;
  const uint32_t n = keys ? s.Nk : s.N;
  const uint32_t row = (keys ? blockIdx.x - q_wgs : blockIdx.x) * per_wg + threadIdx.x / lanes;
  const bool real = row < (uint32_t)s.B * n;
  const uint32_t b = row / n, tok = row % n;
  float t[PER][V], top = 0.f;
#pragma unroll
  for (int p = 0; p < PER; ++p) {
    const int c = (p * lanes + lane) * V;
#pragma unroll
    for (int j = 0; j < V; ++j) t[p][j] = 0.f;
    if (!real || c >= C) continue;
    const Piece<T> x = load((keys ? a.kv + (int64_t)row * 2 * C : a.q + (int64_t)row * C) + c), sc = load(a.scale + c);
    Piece<T> pe;
    pe.w = u32x4{0u, 0u, 0u, 0u};
    if (keys) {
      pe = load(a.pe + (int64_t)tok * C + c);
      store(v_out + head_row(s, b, c / s.d, tok, n, s.d) + c % s.d, load(a.kv + (int64_t)row * 2 * C + C + c));
    }
#pragma unroll
    for (int j = 0; j < V; ++j) {
      t[p][j] = focus_input<T>((float)x.e[j] + (float)pe.e[j], (float)sc.e[j]);
      top = fmaxf(top, t[p][j]);
    }
  }
  top = row_max(top, lanes);
  const int exponent = focus_exponent(top);
  const float down = ldexpf(1.f, -exponent);
  float n2 = 0.f, m2 = 0.f;
#pragma unroll
  for (int p = 0; p < PER; ++p)
#pragma unroll
    for (int j = 0; j < V; ++j) {
      const float v = t[p][j] * down, cube = v * v * v;
      n2 = fmaf(v, v, n2);
      m2 = fmaf(cube, cube, m2);
      t[p][j] = cube;
    }
  const float r = ldexpf(sqrtf(row_sum(n2, lanes) / row_sum(m2, lanes)), exponent);
#pragma unroll
  for (int p = 0; p < PER; ++p) {
    const int c = (p * lanes + lane) * V;
    if (!real || c >= C) continue;
    Piece<T> out;
#pragma unroll
    for (int j = 0; j < V; ++j) out.e[j] = (T)(t[p][j] * r);
    store((keys ? k_out : q_out) + head_row(s, b, c / s.d, tok, n, s.d) + c % s.d, out);
  }
}

// Sums over tokens and batches as in polarity_bwd_kernel; partial: [workgroup][C]
template <typename T, int PER>
__global__ __launch_bounds__(kThreads) void focus_bwd_kernel(Shape s, Focus<const T> a, FocusGrads<const T> g, int lanes,
                                                             T* __restrict__ dq, T* __restrict__ dkv,
                                                             float* __restrict__ partial, float* __restrict__ pe_partial,
                                                             int q_wgs, int groups) {
  constexpr int V = Piece<T>::kVec;
  const bool keys = (int)blockIdx.x >= q_wgs;
  const int lane = threadIdx.x % lanes, per_wg = kThreads / lanes, C = s.heads * s.d, own = threadIdx.x / lanes;
  const uint32_t wg = keys ? blockIdx.x - q_wgs : blockIdx.x, wgs = keys ? gridDim.x - q_wgs : q_wgs;
  const uint32_t n = keys ? s.Nk : s.N;
  // queries: items are rows, one "batch" each; keys: items are (token, batch group)
  const uint32_t items = keys ? n * groups : (uint32_t)s.B * n;
  float scale[PER][V];
  Sum<T> dscale[PER][V];
#pragma unroll
  for (int p = 0; p < PER; ++p) {
    const int c = (p * lanes + lane) * V;
    Piece<T> sc;
    sc.w = u32x4{0u, 0u, 0u, 0u};
    if (c < C) sc = load(a.scale + c);
#pragma unroll
    for (int j = 0; j < V; ++j) {
      scale[p][j] = c < C ? divisor<T>(sc.e[j]) : 1.f;
      dscale[p][j] = 0;
    }
  }
  // every group of lanes makes the same number of trips, so that all lanes of a wave reach the shuffles
  for (uint32_t first = wg * per_wg; first < items; first += wgs * per_wg) {
    const uint32_t item = first + own;
    const bool real = item < items;
    const uint32_t tok = keys ? item / groups : item % n;
    const uint32_t b0 = keys ? item % groups : item / n, b_step = keys ? groups : s.B;
    float dpe[PER][V];
#pragma unroll
    for (int p = 0; p < PER; ++p)
#pragma unroll
      for (int j = 0; j < V; ++j) dpe[p][j] = 0.f;
    const uint32_t trips = keys ? (s.B + groups - 1) / groups : 1;
    for (uint32_t trip = 0; trip < trips; ++trip) {
      const uint32_t b = b0 + trip * b_step;
      const bool here = real && b < (uint32_t)s.B;
      const int64_t row = (int64_t)b * n + tok;
      float t[PER][V], gf[PER][V], top = 0.f;
      uint32_t positive[PER];
#pragma unroll
      for (int p = 0; p < PER; ++p) {
        const int c = (p * lanes + lane) * V;
        positive[p] = 0;
#pragma unroll
        for (int j = 0; j < V; ++j) t[p][j] = gf[p][j] = 0.f;
        if (!here || c >= C) continue;
        const int64_t head = head_row(s, b, c / s.d, tok, n, s.d) + c % s.d;
        const Piece<T> x = load((keys ? a.kv + row * 2 * C : a.q + row * C) + c), gi = load((keys ? g.k : g.q) + head);
        Piece<T> pe;
        pe.w = u32x4{0u, 0u, 0u, 0u};
        if (keys) {
          pe = load(a.pe + (int64_t)tok * C + c);
          const Piece<T> vh = load(g.v + head), vr = load(g.v_rows + row * C + c);
          Piece<T> v;
#pragma unroll
          for (int j = 0; j < V; ++j) v.e[j] = (T)((float)vh.e[j] + (float)vr.e[j]);
          store(dkv + row * 2 * C + C + c, v);
        }
#pragma unroll
        for (int j = 0; j < V; ++j) {
          const float xf = (float)x.e[j] + (float)pe.e[j];
          if (!(xf <= 0.f)) positive[p] |= 1u << j;
          t[p][j] = over<T>((xf < 0.f ? 0.f : xf) + 1e-6f, scale[p][j]);
          top = fmaxf(top, t[p][j]);
          gf[p][j] = (float)gi.e[j];
        }
      }
      top = row_max(top, lanes);
      const float down = ldexpf(1.f, -focus_exponent(top));
      float n2 = 0.f, m2 = 0.f, G = 0.f;
#pragma unroll
      for (int p = 0; p < PER; ++p)
#pragma unroll
        for (int j = 0; j < V; ++j) {
          const float v = t[p][j] * down, cube = v * v * v;
          n2 = fmaf(v, v, n2);
          m2 = fmaf(cube, cube, m2);
          G = fmaf(gf[p][j], cube, G);
        }
      n2 = row_sum(n2, lanes);
      m2 = row_sum(m2, lanes);
      G = row_sum(G, lanes);
      const float nn = sqrtf(n2), mm = sqrtf(m2);
      const float c2 = 3.f * nn / mm, c1 = G / (nn * mm), c5 = G * 3.f * nn / (mm * m2);
#pragma unroll
      for (int p = 0; p < PER; ++p) {
        const int c = (p * lanes + lane) * V;
        if (!here || c >= C) continue;
        Piece<T> out;
#pragma unroll
        for (int j = 0; j < V; ++j) {
          const float v = t[p][j] * down, v2 = v * v;
          const float dt = c2 * v2 * gf[p][j] + c1 * v - c5 * v2 * v2 * v;
          dscale[p][j] += (Sum<T>)dt * t[p][j];
          const float dx = (positive[p] >> j & 1) ? over<T>(dt, scale[p][j]) : 0.f;
          dpe[p][j] += dx;
          out.e[j] = (T)dx;
        }
        store((keys ? dkv + row * 2 * C : dq + row * C) + c, out);
      }
    }
    if (keys && real) {
#pragma unroll
      for (int p = 0; p < PER; ++p) {
        const int c = (p * lanes + lane) * V;
        if (c >= C) continue;
        float* to = pe_partial + ((int64_t)b0 * n + tok) * C + c;
#pragma unroll
        for (int j = 0; j < V; j += 4)
          *reinterpret_cast<f32x4*>(to + j) = f32x4{dpe[p][j], dpe[p][j + 1], dpe[p][j + 2], dpe[p][j + 3]};
      }
    }
  }
  __shared__ Sum<T> sums[kThreads * V];
#pragma unroll
  for (int p = 0; p < PER; ++p) {
    __syncthreads();
#pragma unroll
    for (int j = 0; j < V; ++j) sums[threadIdx.x * V + j] = dscale[p][j];
    __syncthreads();
    for (int i = threadIdx.x; i < lanes * V; i += kThreads) {
      const int c = p * lanes * V + i;
      Sum<T> v = 0;
      for (int q = 0; q < per_wg; ++q) v += sums[q * lanes * V + i];
      if (c < C) partial[(int64_t)blockIdx.x * C + c] = (float)v;
    }
  }
}

// ---------------------------------------------------------------------------------------------------------------
unsigned wgs_for(int64_t rows, int C, int vec) { return (unsigned)cdiv64(rows * (C / vec), kThreads); }
template <typename F> void by_type(int dtype, F&& f) {
  if (dtype == kF16) f(_Float16{});
  else if (dtype == kBF16) f(__bf16{});
  else f(float{});
}
template <typename T, template <typename> class S> S<const T> typed(const S<const void>& a) {
  return __builtin_bit_cast(S<const T>, a);  // the same pointers, to elements of the tensors' type
}

// Split of the polarity gradient: about two workgroups per CU for each side (each costs 2 C partial sums); the batches of a
// token in as many groups as give the keys that many workgroups.
struct Split {
  int q_wgs, k_wgs, groups, channel_wgs;
};
Split polarity_split(const Shape& s, int vec) {
  const int pieces = s.heads * s.d / vec, channel_wgs = (pieces + 63) / 64;
  const int rows = kThreads / (pieces < 64 ? pieces : 64);
  const int64_t most = 512 / channel_wgs < 1 ? 1 : 512 / channel_wgs;
  const int64_t q = cdiv64((int64_t)s.B * s.N, rows);
  int64_t groups = cdiv64(most * rows, s.Nk);
  groups = groups < s.B ? groups : s.B;
  const int64_t k = cdiv64(s.Nk * groups, rows);
  return {(int)(q < most ? q : most), (int)(k < most ? k : most), (int)groups, channel_wgs};
}

}  // namespace

int vec_of(int dtype) { return dtype == kF32 ? 4 : 8; }

void polarity_fwd(const Shape& s, const Polarity<const void>& a, void* q_same, void* q_opp, void* k_both, void* v_heads,
                  int dtype, hipStream_t st) {
  by_type(dtype, [&](auto tag) {
    using T = decltype(tag);
    const int C = s.heads * s.d;
    const unsigned q_wgs = wgs_for((int64_t)s.B * s.N, C, Piece<T>::kVec),
                   k_wgs = wgs_for((int64_t)s.B * s.Nk, C, Piece<T>::kVec);
    polarity_fwd_kernel<T><<<dim3(q_wgs + k_wgs), dim3(kThreads), 0, st>>>(s, typed<T, Polarity>(a), (T*)q_same, (T*)q_opp,
                                                                          (T*)k_both, (T*)v_heads, q_wgs);
  });
}

size_t polarity_bwd_workspace_bytes(const Shape& s, int dtype) {
  const Split w = polarity_split(s, vec_of(dtype));
  const size_t C = (size_t)s.heads * s.d;
  return sizeof(float) * (2 * C * (w.q_wgs + w.k_wgs) + C * w.groups * s.Nk);
}

void polarity_bwd(const Shape& s, const Polarity<const void>& a, const PolarityGrads<const void>& g, void* dqg, void* dkv,
                  void* dpe, void* dscale, void* dpower, float* workspace, int dtype, hipStream_t st) {
  by_type(dtype, [&](auto tag) {
    using T = decltype(tag);
    const Split w = polarity_split(s, Piece<T>::kVec);
    const int C = s.heads * s.d, wgs = w.q_wgs + w.k_wgs;
    float* pe_partial = workspace + (int64_t)2 * C * wgs;
    polarity_bwd_kernel<T><<<dim3((unsigned)wgs, (unsigned)w.channel_wgs), dim3(kThreads), 0, st>>>(
        s, typed<T, Polarity>(a), typed<T, PolarityGrads>(g), (T*)dqg, (T*)dkv, workspace, pe_partial, w.q_wgs, w.groups);
    features_finish(C, wgs, workspace, a.scale, {}, dscale, dpower, w.groups, (int64_t)s.Nk * C, pe_partial, dpe, dtype, st);
  });
}

void features_finish(int C, int terms, const float* partial, const void* scale, RawPower raw, void* dscale, void* dpower, int groups,
                     int64_t pe_count, const float* pe_partial, void* dpe, int dtype, hipStream_t st) {
  by_type(dtype, [&](auto tag) {
    using T = decltype(tag);
    const int stat_wgs = (2 * C + 63) / 64;
    features_finish_kernel<T><<<dim3((unsigned)(stat_wgs + cdiv64(pe_count, 64))), dim3(kThreads), 0, st>>>(
        C, 2, 2, terms, partial, (const T*)scale, (const T*)raw.power, raw.alpha, (T*)dscale, (T*)dpower, stat_wgs, groups, pe_count, pe_partial, (T*)dpe);
  });
}

void rotary_fwd(const Shape& s, const void* qk, const void* x, const float* rot, int rot_channels, void* q, void* k,
                void* q_rot, void* k_rot, void* v, int dtype, hipStream_t st) {
  by_type(dtype, [&](auto tag) {
    using T = decltype(tag);
    rotary_fwd_kernel<T><<<dim3(wgs_for((int64_t)s.B * s.N, s.heads * s.d, Piece<T>::kVec)), dim3(kThreads), 0, st>>>(
        s, (const T*)qk, (const T*)x, rot, rot_channels, (T*)q, (T*)k, (T*)q_rot, (T*)k_rot, (T*)v);
  });
}

void rotary_bwd(const Shape& s, const void* qk, const float* rot, int rot_channels, const RotaryGrads<const void>& g,
                void* dqk, void* dx, int dtype, hipStream_t st) {
  by_type(dtype, [&](auto tag) {
    using T = decltype(tag);
    rotary_bwd_kernel<T><<<dim3(wgs_for((int64_t)s.B * s.N, s.heads * s.d, Piece<T>::kVec)), dim3(kThreads), 0, st>>>(
        s, (const T*)qk, rot, rot_channels, typed<T, RotaryGrads>(g), (T*)dqk, (T*)dx);
  });
}

void turn_fwd(const Shape& s, const void* q, const void* k, const void* weight, const float* rot, void* k_out, void* q_rot,
              void* k_rot, int dtype, hipStream_t st) {
  by_type(dtype, [&](auto tag) {
    using T = decltype(tag);
    turn_fwd_kernel<T><<<dim3(wgs_for((int64_t)s.B * s.N, s.heads * s.d, Piece<T>::kVec)), dim3(kThreads), 0, st>>>(
        s, (const T*)q, (const T*)k, (const T*)weight, rot, (T*)k_out, (T*)q_rot, (T*)k_rot);
  });
}

void turn_bwd(const Shape& s, const void* k, const void* weight, const float* rot, const void* dk_out, const void* dq_rot,
              const void* dk_rot, void* dq, void* dk, void* dweight, int dtype, hipStream_t st) {
  by_type(dtype, [&](auto tag) {
    using T = decltype(tag);
    turn_bwd_kernel<T><<<dim3(wgs_for((int64_t)s.B * s.N, s.heads * s.d, Piece<T>::kVec)), dim3(kThreads), 0, st>>>(
        s, (const T*)k, (const T*)weight, rot, (const T*)dk_out, (const T*)dq_rot, (const T*)dk_rot, (T*)dq, (T*)dk,
        (T*)dweight);
  });
}

void merge_fwd(const Shape& s, const Merge<const void>& a, void* out, int dtype, hipStream_t st) {
  by_type(dtype, [&](auto tag) {
    using T = decltype(tag);
    merge_fwd_kernel<T><<<dim3(wgs_for((int64_t)s.B * s.N, s.heads * s.d, Piece<T>::kVec)), dim3(kThreads), 0, st>>>(
        s, typed<T, Merge>(a), (T*)out);
  });
}

void merge_bwd(const Shape& s, const Merge<const void>& a, const void* dout, void* d_o, void* d_o2, void* dlocal, void* dgate,
               int dtype, hipStream_t st) {
  by_type(dtype, [&](auto tag) {
    using T = decltype(tag);
    merge_bwd_kernel<T><<<dim3(wgs_for((int64_t)s.B * s.N, s.heads * s.d, Piece<T>::kVec)), dim3(kThreads), 0, st>>>(
        s, typed<T, Merge>(a), (const T*)dout, (T*)d_o, (T*)d_o2, (T*)dlocal, (T*)dgate);
  });
}

// Lanes and pieces of a row that is normalised over its channels
struct Lanes {
  int lanes, per;
};
static Lanes row_lanes(int C, int vec) {
  const int pieces = C / vec;
  int lanes = 8;
  while (lanes < 64 && lanes < pieces) lanes *= 2;
  return {lanes, (pieces + lanes - 1) / lanes};
}
int most_row_channels(int dtype) { return 64 * 4 * vec_of(dtype); }
template <typename F> static void by_pieces(int per, F&& f) {
  if (per == 1) f(std::integral_constant<int, 1>());
  else if (per == 2) f(std::integral_constant<int, 2>());
  else f(std::integral_constant<int, 4>());
}

void focus_fwd(const Shape& s, const Focus<const void>& a, void* q, void* k, void* v, int dtype, hipStream_t st) {
  by_type(dtype, [&](auto tag) {
    using T = decltype(tag);
    const Lanes l = row_lanes(s.heads * s.d, Piece<T>::kVec);
    const int rows = kThreads / l.lanes;
    const unsigned q_wgs = (unsigned)cdiv64((int64_t)s.B * s.N, rows), k_wgs = (unsigned)cdiv64((int64_t)s.B * s.Nk, rows);
    by_pieces(l.per, [&](auto per) {
      focus_fwd_kernel<T, decltype(per)::value><<<dim3(q_wgs + k_wgs), dim3(kThreads), 0, st>>>(
          s, typed<T, Focus>(a), l.lanes, q_wgs, (T*)q, (T*)k, (T*)v);
    });
  });
}

// as polarity_split, for rows of whole tokens
static Split focus_split(const Shape& s, int vec) {
  const int rows = kThreads / row_lanes(s.heads * s.d, vec).lanes;
  const int64_t most = 512, q = cdiv64((int64_t)s.B * s.N, rows);
  int64_t groups = cdiv64(most * rows, s.Nk);
  groups = groups < s.B ? groups : s.B;
  const int64_t k = cdiv64(s.Nk * groups, rows);
  return {(int)(q < most ? q : most), (int)(k < most ? k : most), (int)groups, 1};
}

size_t focus_bwd_workspace_bytes(const Shape& s, int dtype) {
  const Split w = focus_split(s, vec_of(dtype));
  const size_t C = (size_t)s.heads * s.d;
  return sizeof(float) * C * ((size_t)w.q_wgs + w.k_wgs + (size_t)w.groups * s.Nk);
}

void focus_bwd(const Shape& s, const Focus<const void>& a, const FocusGrads<const void>& g, void* dq, void* dkv, void* dpe,
               void* dscale, float* workspace, int dtype, hipStream_t st) {
  by_type(dtype, [&](auto tag) {
    using T = decltype(tag);
    const Split w = focus_split(s, Piece<T>::kVec);
    const int C = s.heads * s.d, wgs = w.q_wgs + w.k_wgs;
    const Lanes l = row_lanes(C, Piece<T>::kVec);
    float* pe_partial = workspace + (int64_t)C * wgs;
    by_pieces(l.per, [&](auto per) {
      focus_bwd_kernel<T, decltype(per)::value><<<dim3((unsigned)wgs), dim3(kThreads), 0, st>>>(
          s, typed<T, Focus>(a), typed<T, FocusGrads>(g), l.lanes, (T*)dq, (T*)dkv, workspace, pe_partial, w.q_wgs, w.groups);
    });
    const int64_t pe_count = (int64_t)s.Nk * C;
    const int stat_wgs = (C + 63) / 64;
    features_finish_kernel<T><<<dim3((unsigned)(stat_wgs + cdiv64(pe_count, 64))), dim3(kThreads), 0, st>>>(
        C, 1, 1, wgs, workspace, (const T*)a.scale, nullptr, 0.f, (T*)dscale, nullptr, stat_wgs, w.groups, pe_count, pe_partial, (T*)dpe);
  });
}

void interpolate_fwd(const void* x, int64_t x_batch, int64_t x_row, int B, int from, int to, int C, void* y, int dtype,
                     hipStream_t st) {
  by_type(dtype, [&](auto tag) {
    using T = decltype(tag);
    interpolate_fwd_kernel<T><<<dim3(wgs_for((int64_t)B * to, C, Piece<T>::kVec)), dim3(kThreads), 0, st>>>(
        (const T*)x, x_batch, x_row, B, from, to, C, (T*)y);
  });
}

void interpolate_bwd(const void* g, int B, int from, int to, int C, void* dx, int dtype, hipStream_t st) {
  by_type(dtype, [&](auto tag) {
    using T = decltype(tag);
    interpolate_bwd_kernel<T><<<dim3(wgs_for((int64_t)B * from, C, Piece<T>::kVec)), dim3(kThreads), 0, st>>>(
        (const T*)g, B, from, to, C, (T*)dx);
  });
}

}  // namespace blocks
}  // namespace fbla
