// The attention of two vision blocks straight on the rows of their projections, 16-bit types, heads of 32 channels: PolaFormer's
// two pairings with their polarity features, gate and local values (layers/polaformer.py:63-104) and MLLA's rotary numerator
// over a plain denominator with its local values (layers/mlla.py:74-92).  Features are computed where they are multiplied and
// nothing is laid out as heads: forward, one pass over keys and values (state) and one over queries (output rows); backward,
// one over queries and output gradients (gradients of queries, gate and local values, sums of the state's gradient) and one over
// keys and values.
//
// What bounds it: vector instructions about as much as HBM (a power costs a logarithm and an exponential per channel and pass, its
// gradient another pair), the matrix products hide behind both.  A wave takes 32 tokens of one head at a time.  Lane (t, kb)
// = (lane % 32, lane / 32) holds of token t the channels 16 s + 8 kb + 0..7, s = 0, 1: the 16-byte pieces of its row, the B operand
// of 32x32x16 with the tokens as columns, and - with the rows of the A operand permuted (row_of) - the 16 accumulators of a
// product's column.  So rows, features, products and results of a token never leave its two lanes; only the sums over tokens
// need the tokens as the contraction, and go through wave-private LDS and its transposing read.  The four waves of a
// workgroup take neighbouring heads (128-byte lines and more of a row at about the same time).
//
// Polarity: features F = pos | neg (64), matrix M = S of the same-sign pairing for the first 16 value channels and S with its halves
// swapped for the last 16, so that F M is both pairings at once, with a denominator for each.  Rotary: F = turned features
// (32), M = S, the denominator from the plain features.  Matrices are operands as hi + lo pairs of 16 bits.
//
// Measured, bf16, heads as kernels of their own (features to heads, both operators, merge and gate, and the gradients of each) ->
// here, with what each reaches of the bytes it moves: PolaFormer's 64 x 28x28 x 256: forward 136 -> 62 us (state 21 us, 2.6 TB/s;
// output 33 us, 3.1 TB/s), backward 270 -> 131 us (queries 61 us, 2.9 TB/s; keys 55 us, 2.6 TB/s; the two finishing launches 5 us
// each), the whole step 750 -> 502 us.  MLLA's 64 x 56x56 x 64: forward 84 -> 48 us (state 17, output 24 us, 3.3 TB/s), backward
// 139 -> 71 us (queries 30, keys 33 us, 3.9 TB/s), the step 371 -> 238 us.  What was tried and cost time: three waves a SIMD for
// state and output (4 spilled registers each: 24 and 35 us), two tiles a wave for the keys (256 registers: 72 us), shuffles of each
// sum by itself at the end of the queries' pass (86 us), LDS addresses kept over the tiles (76 spilled: 141 us).
#include <hip/hip_runtime.h>

#include <algorithm>
#include <type_traits>

#include "fbla_mfma_shared.h"

namespace fbla {
namespace rows {

namespace {

constexpr int kThreads = 256, kWaves = 4, D = 32;
using mfma::f32x16;
using mfma::wave_sync;

typedef uint32_t u32x4 __attribute__((ext_vector_type(4)));
typedef uint32_t u32x2 __attribute__((ext_vector_type(2)));
typedef short i16x2 __attribute__((ext_vector_type(2)));
typedef short i16x4 __attribute__((ext_vector_type(4)));
typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
typedef _Float16 f16x8 __attribute__((ext_vector_type(8)));
typedef float f32x4 __attribute__((ext_vector_type(4)));
typedef float f32x8 __attribute__((ext_vector_type(8)));
template <typename T> struct Vec;
template <> struct Vec<__bf16> { typedef bf16x8 type; };
template <> struct Vec<_Float16> { typedef f16x8 type; };
template <typename T> using V8 = typename Vec<T>::type;

__device__ __forceinline__ f32x16 mma(bf16x8 a, bf16x8 b, f32x16 c) { return __builtin_amdgcn_mfma_f32_32x32x16_bf16(a, b, c, 0, 0, 0); }
__device__ __forceinline__ f32x16 mma(f16x8 a, f16x8 b, f32x16 c) { return __builtin_amdgcn_mfma_f32_32x32x16_f16(a, b, c, 0, 0, 0); }
template <typename T> __device__ __forceinline__ V8<T> load8(const T* p) { return *reinterpret_cast<const V8<T>*>(p); }
template <typename T> __device__ __forceinline__ f32x8 wide(V8<T> v) { return __builtin_convertvector(v, f32x8); }
template <typename T> __device__ __forceinline__ V8<T> narrow(f32x8 v) { return __builtin_convertvector(v, V8<T>); }
__device__ __forceinline__ f32x8 load_f8(const float* p) {
  const f32x4 a = *reinterpret_cast<const f32x4*>(p), b = *reinterpret_cast<const f32x4*>(p + 4);
  return f32x8{a[0], a[1], a[2], a[3], b[0], b[1], b[2], b[3]};
}
__device__ __forceinline__ f32x16 zero16() {
  f32x16 r;
#pragma unroll
  for (int i = 0; i < 16; ++i) r[i] = 0.f;
  return r;
}
__device__ __forceinline__ float both_halves(float x) { return x + __shfl_xor(x, 32); }
__device__ __forceinline__ float sum8(f32x8 v) { return ((v[0] + v[1]) + (v[2] + v[3])) + ((v[4] + v[5]) + (v[6] + v[7])); }

// Output channel of row m of a permuted A operand: accumulator r = 8 s + e of a lane's column is then channel 16 s + 8 kb + e
__device__ __forceinline__ int row_of(int m) { return 16 * (m >> 4) + 8 * ((m >> 2) & 1) + 4 * ((m >> 3) & 1) + (m & 3); }

// ---- LDS tiles [32 tokens][64 or 32 channels of 16 bits]: pieces are written down a column of 32 rows and read four rows at a
// time by the transposing read; both spread over all banks
__device__ __forceinline__ int place64(int row, int ch) {
  return row * 128 + ((ch ^ (((row >> 1) & 1) << 1 | ((row >> 2) & 1) | ((row >> 3) & 1) << 2)) << 4);
}
__device__ __forceinline__ int place32(int row, int ch) { return row * 64 + ((ch ^ ((row >> 2) & 3)) << 4); }
__device__ __forceinline__ u32x2 transposed_read(const unsigned char* at) {
  typedef i16x4 __attribute__((address_space(3))) * lds_ptr;
  return __builtin_bit_cast(u32x2, __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_ptr)(at)));
}
template <bool WIDE> __device__ __forceinline__ int place(int row, int ch) { return WIDE ? place64(row, ch) : place32(row, ch); }
// channels 32 block + lane % 32 (PERMUTED: row_of(lane % 32)) of the tokens 16 ks + 8 kb + 0..7
template <typename T, bool WIDE, bool PERMUTED = false> __device__ __forceinline__ V8<T> tokens_of(const unsigned char* tile, int lane,
                                                                                                    int block, int ks) {
  const int g = lane >> 4, s = lane & 15;
  u32x2 r[2];
#pragma unroll
  for (int h = 0; h < 2; ++h) {
    const int four = PERMUTED ? (s & 1) << 1 | (s >> 1 & 1) : s & 3;
    const int row = 16 * ks + 8 * (g >> 1) + 4 * h + (s >> 2), c = 32 * block + 16 * (g & 1) + 4 * four;
    r[h] = transposed_read(tile + place<WIDE>(row, c >> 3) + ((c >> 2) & 1) * 8);
  }
  return __builtin_bit_cast(V8<T>, u32x4{r[0][0], r[0][1], r[1][0], r[1][1]});
}

// ---- features of a lane's 16 channels of a token
template <typename T> struct Features {
  V8<T> f[4];  // polarity: pos, pos, neg, neg of the two pieces; rotary: turned, turned, plain, plain
};
template <typename T, bool POLA, typename K> __device__ __forceinline__ Features<T> features_of(const f32x8 (&x)[2], const K& k,
                                                                                                 const f32x8 (&cs)[2]) {
  Features<T> r;
#pragma unroll
  for (int s = 0; s < 2; ++s) {
    if constexpr (POLA) {
      const f32x8 inv = k.inv(s), power = k.power(s);
      f32x8 a;
      u32x4 negative;
#pragma unroll
      for (int e = 0; e < 8; ++e) a[e] = __builtin_amdgcn_exp2f(power[e] * __builtin_amdgcn_logf(fabsf(x[s][e] * inv[e])));
#pragma unroll
      for (int e = 0; e < 4; ++e)  // the signs of two channels, spread over their halves of a word
        negative[e] = __builtin_bit_cast(uint32_t, __builtin_bit_cast(i16x2, __builtin_amdgcn_perm(__float_as_uint(x[s][2 * e + 1]),
                                                                                                   __float_as_uint(x[s][2 * e]), 0x07060302u)) >> 15);
      const u32x4 w = __builtin_bit_cast(u32x4, narrow<T>(a));
      r.f[s] = __builtin_bit_cast(V8<T>, w & ~negative);
      r.f[2 + s] = __builtin_bit_cast(V8<T>, w & negative);
    } else {
      f32x8 a, b;
#pragma unroll
      for (int e = 0; e < 8; ++e) b[e] = x[s][e] > 0.f ? x[s][e] + 1.f : __builtin_amdgcn_exp2f(x[s][e] * 1.44269504088896341f);
#pragma unroll
      for (int e = 0; e < 8; e += 2) {
        a[e] = b[e] * cs[s][e] - b[e + 1] * cs[s][e + 1];
        a[e + 1] = b[e] * cs[s][e + 1] + b[e + 1] * cs[s][e];
      }
      r.f[s] = narrow<T>(a);
      r.f[2 + s] = narrow<T>(b);
    }
  }
  return r;
}
// Gradient of x from those of the features' two parts (polarity: pos and neg; rotary: turned and plain).  Polarity, with
// y = x / scale, u the gradient of the part that x is in: dx = +-u power |y|^(power - 1) / scale; the sums for scale and power lack
// the factors that are the same for every token (stats_factors).
template <bool POLA, typename K> __device__ __forceinline__ f32x8 features_grad(f32x8 x, const K& k, int s, f32x8 cs, f32x8 ga, f32x8 gb,
                                                                                f32x8& dscale, f32x8& dpower) {
  f32x8 dx;
  if constexpr (POLA) {
    const f32x8 inv = k.inv(s), power = k.power(s);
#pragma unroll
    for (int e = 0; e < 8; ++e) {
      const float y = x[e] * inv[e];
      // (the bare logarithm takes a denormal for 0: from the smallest normal number up, where the slope is 1 or next to nothing)
      const float l = __builtin_amdgcn_logf(__builtin_amdgcn_fmed3f(fabsf(y), 1.17549435e-38f, 3.4028235e38f));
      const float slope = __builtin_amdgcn_exp2f(fmaf(power[e], l, -l));
      const float u = y < 0.f ? -gb[e] : ga[e];
      const float t = y == 0.f ? 0.f : u * slope;  // both parts are cut off at 0
      dx[e] = t * power[e] * inv[e];
      dscale[e] = fmaf(t, x[e], dscale[e]);
      dpower[e] = fmaf(t * x[e], l, dpower[e]);
    }
  } else {
#pragma unroll
    for (int e = 0; e < 8; e += 2) {
      const float re = gb[e] + ga[e] * cs[e] + ga[e + 1] * cs[e + 1], im = gb[e + 1] + ga[e + 1] * cs[e] - ga[e] * cs[e + 1];
      dx[e] = x[e] > 0.f ? re : re * __builtin_amdgcn_exp2f(x[e] * 1.44269504088896341f);
      dx[e + 1] = x[e + 1] > 0.f ? im : im * __builtin_amdgcn_exp2f(x[e + 1] * 1.44269504088896341f);
    }
  }
  return dx;
}

template <typename K> __device__ __forceinline__ void stats_factors(const K& k, f32x8 (&dscale)[2], f32x8 (&dpower)[2]) {
#pragma unroll
  for (int s = 0; s < 2; ++s) {
    dscale[s] *= k.power(s);
    dpower[s] *= k.inv(s) * 0.693147180559945309f;
  }
}

// the wave's place: head h of batch b, every TI-th tile of 32 tokens from its own
struct Place {
  int lane, t, kb, h, sub, subs;
  __device__ __forceinline__ Place(int heads, int group_heads, int group) {
    lane = threadIdx.x & 63;
    t = lane & 31;
    kb = lane >> 5;
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    h = group * group_heads + wave % group_heads;
    sub = wave / group_heads;
    subs = kWaves / group_heads;
  }
};
// 1 / scale and power of the head's channels from their parameters, in LDS (64 floats a wave): registers are what these kernels are short of
template <typename T, bool POLA> struct Constants {
  float* at;
  int c0;
  __device__ __forceinline__ Constants(float* to, const Attn& a, const Place& p) : at(to), c0(8 * p.kb) {
    if constexpr (POLA) {
      const int c = p.h * D + p.t;
      at[p.lane] = p.kb ? 1.f + a.alpha * blocks::sigmoid((float)((const T*)a.power)[c]) : 1.f / blocks::softplus((float)((const T*)a.scale)[c]);
    }
  }
  __device__ __forceinline__ f32x8 inv(int s) const { return POLA ? load_f8(at + 16 * s + c0) : f32x8{}; }
  __device__ __forceinline__ f32x8 power(int s) const { return POLA ? load_f8(at + 32 + 16 * s + c0) : f32x8{}; }
};
// The lane's pieces of token t0 + tt: the tile's address is the wave's, the lane adds 32 bits
template <typename P> __device__ __forceinline__ P* piece(P* head0, int64_t row, int t0, int tt, int kb) {
  return head0 + (int64_t)t0 * row + (uint32_t)(tt * (int)row + 8 * kb);
}
template <typename T, bool POLA> __device__ __forceinline__ void load_turns(const Attn& a, const Place& p, int t0, int tt, f32x8 (&cs)[2]) {
  if constexpr (!POLA) {
    const float* at = piece(a.rot + p.h * D, a.heads * D, t0, tt, p.kb);
#pragma unroll
    for (int s = 0; s < 2; ++s) cs[s] = load_f8(at + 16 * s);
  }
}

// sizes of a head's sums: M's rows, and the vector that goes with it
template <bool POLA> constexpr int kFeatures = POLA ? 64 : 32;
template <bool POLA> constexpr int kSlot = kFeatures<POLA> * (D + 1);  // floats of a partial
template <bool POLA> constexpr int kVector = kFeatures<POLA> + 8;       // floats of a head's finished vector: [features], the planes' factor

// ---------------------------------------------------------------------------------------------------------------
// state: partial sums of F^T V and of the denominator's features over `chunk` tokens
// ---------------------------------------------------------------------------------------------------------------
template <typename T, bool POLA>
__global__ __launch_bounds__(kThreads, 2) void state_kernel(Attn a, float* __restrict__ partial, int chunk, int parts, int group_heads) {
  constexpr int KF = kFeatures<POLA> / 32;
  __shared__ __attribute__((aligned(16))) unsigned char smem[kWaves][32 * 128 + 32 * 64];
  __shared__ __attribute__((aligned(16))) float consts[kWaves][64];
  const Place p(a.heads, group_heads, blockIdx.y);
  const int b = blockIdx.z, C = a.heads * D, h0 = p.h * D, n = a.Nk;
  unsigned char* ft = smem[threadIdx.x >> 6];
  unsigned char* vt = ft + 32 * 128;
  const int t_end = min(n, ((int)blockIdx.x + 1) * chunk);
  const Constants<T, POLA> k(consts[threadIdx.x >> 6], a, p);
  wave_sync();
  const T *ks = (const T*)a.k + (int64_t)b * n * a.k_row + h0, *vs = (const T*)a.v + (int64_t)b * n * a.v_row + h0;

  V8<T> one = {};
  if (p.t == 0)
#pragma unroll
    for (int e = 0; e < 8; ++e) one[e] = (T)1.f;
  f32x16 acc[KF], sum[KF];
#pragma unroll
  for (int f = 0; f < KF; ++f) acc[f] = sum[f] = zero16();

  struct Rows {
    V8<T> k[2], v[2], pe[2];
    f32x8 cs[2];
  };
  auto fetch = [&](Rows& r, int t0) {
    const int tt = min(p.t, n - 1 - t0);
#pragma unroll
    for (int s = 0; s < 2; ++s) {
      r.k[s] = load8(piece(ks, a.k_row, t0, tt, p.kb) + 16 * s);
      r.v[s] = load8(piece(vs, a.v_row, t0, tt, p.kb) + 16 * s);
      if constexpr (POLA) r.pe[s] = load8(piece((const T*)a.pe + h0, C, t0, tt, p.kb) + 16 * s);
    }
    load_turns<T, POLA>(a, p, t0, tt, r.cs);
  };
  Rows r;
  int t0 = blockIdx.x * chunk + 32 * p.sub;
  if (t0 < t_end) fetch(r, t0);
  for (; t0 < t_end; t0 += 32 * p.subs) {
    const bool real = t0 + p.t < t_end;
    f32x8 x[2];
#pragma unroll
    for (int s = 0; s < 2; ++s) {
      x[s] = wide<T>(r.k[s]);
      if constexpr (POLA) x[s] += wide<T>(r.pe[s]);
    }
    Features<T> f = features_of<T, POLA>(x, k, r.cs);
    wave_sync();  // the previous tile has been read
#pragma unroll
    for (int i = 0; i < 4; ++i) *reinterpret_cast<V8<T>*>(ft + place64(p.t, 2 * i + p.kb)) = real ? f.f[i] : V8<T>{};
#pragma unroll
    for (int s = 0; s < 2; ++s) *reinterpret_cast<V8<T>*>(vt + place32(p.t, 2 * s + p.kb)) = real ? r.v[s] : V8<T>{};
    if (t0 + 32 * p.subs < t_end) fetch(r, t0 + 32 * p.subs);
    wave_sync();
#pragma unroll
    for (int ks = 0; ks < 2; ++ks) {
      const V8<T> v = tokens_of<T, false>(vt, p.lane, 0, ks);
#pragma unroll
      for (int fb = 0; fb < KF; ++fb) {
        const V8<T> ff = tokens_of<T, true>(ft, p.lane, fb, ks);
        acc[fb] = mma(ff, v, acc[fb]);
        if constexpr (POLA) sum[fb] = mma(ff, one, sum[fb]);
      }
      if constexpr (!POLA) sum[0] = mma(tokens_of<T, true>(ft, p.lane, 1, ks), one, sum[0]);
    }
  }
  float* to = partial + (((int64_t)b * a.heads + p.h) * parts + blockIdx.x * p.subs + p.sub) * kSlot<POLA>;
#pragma unroll
  for (int fb = 0; fb < KF; ++fb)
#pragma unroll
    for (int i = 0; i < 16; ++i) {
      const int f = 32 * fb + 8 * (i >> 2) + 4 * p.kb + (i & 3);
      to[f * D + p.t] = acc[fb][i];
      if (p.t == 0) to[kFeatures<POLA> * D + f] = sum[fb][i];
    }
}

// ---------------------------------------------------------------------------------------------------------------
// the partials' sum, in order, as operands: planes [f][v] hi, lo and [v][f] hi, lo of `scale` times the matrix, brought to a largest
// value of 8 to 16 by a power of two (as 16-bit pairs it would lose to denormals otherwise), and `scale` times the vector, followed by
// the factor that takes the power back.  Forward: M and the mean key; backward, from the sums of M's gradient: S's and the mean
// key's.  Bound by the latency of the partials' loads: four sets of threads share them (one set: 111 us for 392 partials of one head, 7
// us for 512 heads of four), and the result leaves in 16-byte pieces of both orders through LDS (2 bytes at a time: 11 us).  Now 5 us
// for 512 heads of four, 11 to 14 us where a head has its most, kMostParts.
// ---------------------------------------------------------------------------------------------------------------
constexpr int kFinishThreads = 1024, kFinishSets = 4;  // sets of threads that share a head's partials
template <typename T, bool POLA>
__global__ __launch_bounds__(kFinishThreads) void finish_kernel(const float* __restrict__ partial, int parts, float scale, T* __restrict__ planes,
                                                                float* __restrict__ vec) {
  constexpr int F = kFeatures<POLA>, E = F * D, kSet = kFinishThreads / kFinishSets, kEach = E / kSet, kOwn = E / kFinishThreads;
  static_assert(2 * (E / 8) <= kFinishThreads && F <= kSet && kSlot<POLA> == E + F);
  __shared__ float sums[kFinishSets][kSlot<POLA>], largest[kFinishThreads / 64], matrix[F][D + 1];
  const int64_t head = blockIdx.x;
  const int set = threadIdx.x / kSet, t = threadIdx.x % kSet;
  {
    const float* from = partial + head * parts * kSlot<POLA>;
    float x[kEach] = {}, y = 0.f;
#pragma unroll 4
    for (int i = set; i < parts; i += kFinishSets) {
      const float* at = from + (int64_t)i * kSlot<POLA>;
#pragma unroll
      for (int e = 0; e < kEach; ++e) x[e] += at[t + kSet * e];
      if (t < F) y += at[E + t];
    }
#pragma unroll
    for (int e = 0; e < kEach; ++e) sums[set][t + kSet * e] = x[e];
    if (t < F) sums[set][E + t] = y;
  }
  __syncthreads();
  auto total = [&](int at) { return ((sums[0][at] + sums[1][at]) + (sums[2][at] + sums[3][at])) * scale; };
  float x[kOwn], most = 0.f;
#pragma unroll
  for (int e = 0; e < kOwn; ++e) {
    x[e] = total(threadIdx.x + kFinishThreads * e);
    most = fmaxf(most, fabsf(x[e]));
  }
#pragma unroll
  for (int off = 32; off > 0; off >>= 1) most = fmaxf(most, __shfl_xor(most, off));
  if (threadIdx.x % 64 == 0) largest[threadIdx.x / 64] = most;
  __syncthreads();
#pragma unroll
  for (int w = 0; w < kFinishThreads / 64; ++w) most = fmaxf(most, largest[w]);
  float norm = 1.f;  // also when the matrix is zero or not finite
  if (most > 1e-30f && most < 3e38f) {
    int e;
    frexpf(most, &e);
    norm = ldexpf(1.f, 4 - e);
  }
#pragma unroll
  for (int e = 0; e < kOwn; ++e) {
    const int at = threadIdx.x + kFinishThreads * e, f = at / D, v = at % D;
    matrix[POLA && v >= 16 ? f ^ 32 : f][v] = x[e] * norm;  // the last value channels pair with the swapped halves
  }
  __syncthreads();
  T* to = planes + head * 4 * E;
  auto write = [&](T* plane, auto at) {  // 8 values of a row of the plane, hi and lo
    f32x8 z;
#pragma unroll
    for (int e = 0; e < 8; ++e) z[e] = at(e);
    const V8<T> hi = narrow<T>(z);
    *reinterpret_cast<V8<T>*>(plane) = hi;
    *reinterpret_cast<V8<T>*>(plane + E) = narrow<T>(z - wide<T>(hi));
  };
  if (const int q = threadIdx.x; q < E / 8) {
    write(to + 8 * q, [&](int e) { return matrix[q / (D / 8)][8 * (q % (D / 8)) + e]; });
  } else if (const int r = q - E / 8; r < E / 8) {
    write(to + 2 * E + 8 * r, [&](int e) { return matrix[8 * (r % (F / 8)) + e][r / (F / 8)]; });
  }
  if ((int)threadIdx.x < F) vec[head * kVector<POLA> + threadIdx.x] = total(E + threadIdx.x);
  if (threadIdx.x == 0) vec[head * kVector<POLA> + F] = 1.f / norm;
}

// F M for a lane's token: A operand [v][f], hi + lo
template <typename T, bool POLA> struct Numerator {
  static constexpr int kSteps = kFeatures<POLA> / 16;
  V8<T> hi[kSteps], lo[kSteps];
  __device__ __forceinline__ void load(const T* planes, int lane) {
    constexpr int F = kFeatures<POLA>, E = F * D;
    const T* at = planes + 2 * E + row_of(lane & 31) * F + 8 * (lane >> 5);
#pragma unroll
    for (int ks = 0; ks < kSteps; ++ks) {
      hi[ks] = load8(at + 16 * ks);
      lo[ks] = load8(at + E + 16 * ks);
    }
  }
  __device__ __forceinline__ f32x16 operator()(const Features<T>& f) const {
    f32x16 r = zero16();
#pragma unroll
    for (int ks = 0; ks < kSteps; ++ks) r = mma(hi[ks], f.f[ks], r);
#pragma unroll
    for (int ks = 0; ks < kSteps; ++ks) r = mma(lo[ks], f.f[ks], r);
    return r;
  }
};
// The denominators' inverses for both pieces' channels (rotary: the same), by a product too: rows of the mean key, hi and lo (and of
// its swapped halves), every four rows of the operand the same four, so that both lanes of a token have all of them.
template <typename T, bool POLA> struct MeanKey {
  static constexpr int F = kFeatures<POLA>;
  T* at;  // LDS [POLA ? 4 : 2][F]
  __device__ __forceinline__ MeanKey(T* to, const float* km, int lane) : at(to) {
    if (lane < F) {
      const float x = km[lane];
      const T hi = (T)x, lo = (T)(x - (float)hi);
      at[lane] = hi;
      at[F + lane] = lo;
      if constexpr (POLA) {
        at[2 * F + (lane ^ 32)] = hi;
        at[3 * F + (lane ^ 32)] = lo;
      }
    }
  }
  __device__ __forceinline__ void operator()(const Features<T>& f, const Place& p, float eps, float (&rz)[2]) const {
    const T* row = at + (p.t & (POLA ? 3 : 1)) * F + 8 * p.kb;
    f32x16 z = zero16();
#pragma unroll
    for (int ks = 0; ks < F / 16; ++ks) z = mma(load8(row + 16 * ks), f.f[POLA ? ks : 2 + ks], z);
    rz[0] = 1.f / (z[0] + z[1] + eps);
    rz[1] = POLA ? 1.f / (z[2] + z[3] + eps) : rz[0];
  }
};

// ---------------------------------------------------------------------------------------------------------------
// output rows: (F M / z + local) * gate
// ---------------------------------------------------------------------------------------------------------------
template <typename T, bool POLA>
__global__ __launch_bounds__(kThreads, POLA ? 2 : 3) void output_kernel(Attn a, int chunk, int group_heads) {
  constexpr int F = kFeatures<POLA>;
  __shared__ __attribute__((aligned(16))) float consts[kWaves][64];
  __shared__ __attribute__((aligned(16))) T means[kWaves][256];
  const Place p(a.heads, group_heads, blockIdx.y);
  const int b = blockIdx.z, C = a.heads * D, h0 = p.h * D, n = a.N;
  const int64_t head = (int64_t)b * a.heads + p.h;
  const MeanKey<T, POLA> mean(means[threadIdx.x >> 6], a.km + head * kVector<POLA>, p.lane);
  const float undo = a.km[head * kVector<POLA> + F];
  const Constants<T, POLA> k(consts[threadIdx.x >> 6], a, p);
  Numerator<T, POLA> product;
  product.load((const T*)a.planes + head * 4 * F * D, p.lane);
  wave_sync();
  const T *qs = (const T*)a.q + (int64_t)b * n * a.q_row + h0, *ls = (const T*)a.local + (int64_t)b * n * C + h0,
          *gs = POLA ? (const T*)a.gate + (int64_t)b * n * a.gate_row + h0 : nullptr;
  T* os = (T*)a.out + (int64_t)b * n * C + h0;
  struct Rows {
    V8<T> q[2], local[2], gate[2];
    f32x8 cs[2];
  };
  auto fetch = [&](Rows& r, int t0) {
    const int tt = min(p.t, n - 1 - t0);
#pragma unroll
    for (int s = 0; s < 2; ++s) {
      r.q[s] = load8(piece(qs, a.q_row, t0, tt, p.kb) + 16 * s);
      r.local[s] = load8(piece(ls, C, t0, tt, p.kb) + 16 * s);
      if constexpr (POLA) r.gate[s] = load8(piece(gs, a.gate_row, t0, tt, p.kb) + 16 * s);
    }
    load_turns<T, POLA>(a, p, t0, tt, r.cs);
  };
  const int t_end = min(n, ((int)blockIdx.x + 1) * chunk);
  int t0 = blockIdx.x * chunk + 32 * p.sub;
  Rows r;
  if (t0 < t_end) fetch(r, t0);
  for (; t0 < t_end; t0 += 32 * p.subs) {
    const f32x8 x[2] = {wide<T>(r.q[0]), wide<T>(r.q[1])};
    const Features<T> f = features_of<T, POLA>(x, k, r.cs);
    const f32x16 num = product(f);
    float rz[2];
    mean(f, p, a.eps, rz);
    V8<T> y[2];
#pragma unroll
    for (int s = 0; s < 2; ++s) {
      f32x8 v;
      const float by = undo * rz[s];
#pragma unroll
      for (int e = 0; e < 8; ++e) v[e] = num[8 * s + e] * by;
      v += wide<T>(r.local[s]);
      if constexpr (POLA) v *= wide<T>(r.gate[s]);
      y[s] = narrow<T>(v);
    }
    if (t0 + 32 * p.subs < t_end) fetch(r, t0 + 32 * p.subs);
    if (t0 + p.t < t_end)
#pragma unroll
      for (int s = 0; s < 2; ++s) *reinterpret_cast<V8<T>*>(piece(os, C, t0, p.t, p.kb) + 16 * s) = y[s];
  }
}

// Sums over the 32 tokens of each half of the wave, of 16 values a lane (two pieces' channels).  Each step exchanges the half of the
// values that the other lane keeps: 31 exchanges for 32 values, where five for each would be 160.  Lane t is left with value t % 16.
__device__ __forceinline__ float sum16(const f32x8& a, const f32x8& b, int t) {
  float v[16];
#pragma unroll
  for (int i = 0; i < 16; ++i) v[i] = i < 8 ? a[i & 7] : b[i & 7];
  auto step = [&](auto keep) {
    constexpr int m = decltype(keep)::value;
    const bool upper = t & m;
#pragma unroll
    for (int i = 0; i < m; ++i) {
      const float mine = upper ? v[i + m] : v[i], theirs = upper ? v[i] : v[i + m];
      v[i] = mine + __shfl_xor(theirs, m);
    }
  };
  step(std::integral_constant<int, 8>{});
  step(std::integral_constant<int, 4>{});
  step(std::integral_constant<int, 2>{});
  step(std::integral_constant<int, 1>{});
  return v[0] + __shfl_xor(v[0], 16);
}
// to[16 s + 8 kb + e] = the sum of value e of piece s
__device__ __forceinline__ void store_sums(const f32x8& a, const f32x8& b, float* to, const Place& p) {
  const float v = sum16(a, b, p.t);
  if (p.t < 16) to[16 * (p.t >> 3) + 8 * p.kb + (p.t & 7)] = v;
}
// partial[2][C] of the wave's place
__device__ __forceinline__ void store_stats(const f32x8 (&dscale)[2], const f32x8 (&dpower)[2], float* to, int C, const Place& p) {
  store_sums(dscale[0], dscale[1], to + p.h * D, p);
  store_sums(dpower[0], dpower[1], to + C + p.h * D, p);
}

// ---------------------------------------------------------------------------------------------------------------
// backward over the queries: gradients of queries, gate and local values; partial sums of dM = F^T (do / z) and F^T dz
// ---------------------------------------------------------------------------------------------------------------
template <bool POLA> constexpr int kQueriesWave = 8192 + 2 * 256 + 512 + 2 * D * kFeatures<POLA> * 2;
template <typename T, bool POLA>
__global__ __launch_bounds__(kThreads, 2) void queries_kernel(Attn a, float* __restrict__ partial, float* __restrict__ stats, int chunk,
                                                              int parts, int group_heads) {
  constexpr int F = kFeatures<POLA>, KF = F / 32, E = F * D;
  // per wave: features | e hi and lo | mean key | as operand | constants | the [v][f] planes
  constexpr int kFt = 0, kEt = 4096, kKm = 8192, kMean = kKm + 256, kK = kMean + 512, kM = kK + 256, kWave = kM + 2 * D * F * 2;
  static_assert(kWave == kQueriesWave<POLA>);
  extern __shared__ __attribute__((aligned(16))) unsigned char smem[];
  Place p(a.heads, group_heads, blockIdx.y);
  const int b = blockIdx.z, C = a.heads * D, h0 = p.h * D, n = a.N;
  const int64_t head = (int64_t)b * a.heads + p.h;
  unsigned char* ws = smem + (threadIdx.x >> 6) * kWave;
  unsigned char *ft = ws + kFt, *et = ws + kEt;
  float* km = reinterpret_cast<float*>(ws + kKm);
  const T* planes = (const T*)a.planes + head * 4 * E;
  if (p.lane < F) km[p.lane] = a.km[head * kVector<POLA> + p.lane];
  const float undo = a.km[head * kVector<POLA> + F];
  const MeanKey<T, POLA> mean(reinterpret_cast<T*>(ws + kMean), a.km + head * kVector<POLA>, p.lane);
  // the [v][f] planes in LDS, read by rows and, transposed, by columns
  constexpr int kRow = F * 2;
#pragma unroll
  for (int i = 0; i < 2 * D * F / 8 / 64; ++i) {
    const int q = p.lane + 64 * i, plane = q / (D * F / 8), row = q / (F / 8) % D, ch = q % (F / 8);
    *reinterpret_cast<V8<T>*>(ws + kM + plane * D * kRow + place<POLA>(row, ch)) = load8(planes + (2 + plane) * E + row * F + 8 * ch);
  }
  const Constants<T, POLA> k(reinterpret_cast<float*>(ws + kK), a, p);
  wave_sync();

  const T *qs = (const T*)a.q + (int64_t)b * n * a.q_row + h0, *ds = (const T*)a.dout + (int64_t)b * n * C + h0,
          *ls = POLA ? (const T*)a.local + (int64_t)b * n * C + h0 : nullptr,
          *gs = POLA ? (const T*)a.gate + (int64_t)b * n * a.gate_row + h0 : nullptr;
  T *dqs = (T*)a.dq + (int64_t)b * n * a.dq_row + h0, *dls = POLA ? (T*)a.dlocal + (int64_t)b * n * C + h0 : nullptr,
    *dgs = POLA ? (T*)a.dgate + (int64_t)b * n * a.dgate_row + h0 : nullptr;

  f32x16 acc[KF];
#pragma unroll
  for (int f = 0; f < KF; ++f) acc[f] = zero16();
  f32x8 dkm[2 * KF] = {};  // polarity: pos, pos, neg, neg of the two pieces
  f32x8 dscale[2] = {}, dpower[2] = {};
  struct Rows {
    V8<T> q[2], d[2];
    f32x8 cs[2];
  };
  auto fetch = [&](Rows& r, int t0) {
    const int tt = min(p.t, n - 1 - t0);
#pragma unroll
    for (int s = 0; s < 2; ++s) {
      r.q[s] = load8(piece(qs, a.q_row, t0, tt, p.kb) + 16 * s);
      r.d[s] = load8(piece(ds, C, t0, tt, p.kb) + 16 * s);
    }
    load_turns<T, POLA>(a, p, t0, tt, r.cs);
  };
  const int t_end = min(n, ((int)blockIdx.x + 1) * chunk);
  int t0 = blockIdx.x * chunk + 32 * p.sub;
  Rows r, next;
  if (t0 < t_end) fetch(r, t0);
  for (; t0 < t_end; t0 += 32 * p.subs) {
    // Seen anew in each tile, or the compiler keeps some forty LDS addresses for the whole loop and spills them
    asm volatile("" : "+v"(p.lane), "+v"(p.t), "+v"(p.kb));
    V8<T> local[2], gate[2];
    if constexpr (POLA) {
      const int tt = min(p.t, n - 1 - t0);
#pragma unroll
      for (int s = 0; s < 2; ++s) {
        local[s] = load8(piece(ls, C, t0, tt, p.kb) + 16 * s);
        gate[s] = load8(piece(gs, a.gate_row, t0, tt, p.kb) + 16 * s);
      }
    }
    const bool real = t0 + p.t < t_end;
    const f32x8 x[2] = {wide<T>(r.q[0]), wide<T>(r.q[1])};
    const Features<T> f = features_of<T, POLA>(x, k, r.cs);
    f32x16 num = zero16();
#pragma unroll
    for (int plane = 0; plane < 2; ++plane)
#pragma unroll
      for (int ks = 0; ks < F / 16; ++ks)
        num = mma(*reinterpret_cast<const V8<T>*>(ws + kM + plane * D * kRow + place<POLA>(row_of(p.t), 2 * ks + p.kb)), f.f[ks], num);
    float rz[2], dz[2];
    mean(f, p, a.eps, rz);
    V8<T> g16[2], eh[2], el[2];
#pragma unroll
    for (int s = 0; s < 2; ++s) {
      f32x8 o, g = wide<T>(r.d[s]);
      const float by = undo * rz[s];
#pragma unroll
      for (int e = 0; e < 8; ++e) o[e] = num[8 * s + e] * by;
      g16[s] = r.d[s];
      if constexpr (POLA) {
        const V8<T> dgate = narrow<T>(g * (o + wide<T>(local[s]))), dl = narrow<T>(g * wide<T>(gate[s]));
        if (real) {
          *reinterpret_cast<V8<T>*>(piece(dgs, a.dgate_row, t0, p.t, p.kb) + 16 * s) = dgate;
          *reinterpret_cast<V8<T>*>(piece(dls, C, t0, p.t, p.kb) + 16 * s) = dl;
        }
        g16[s] = dl;
      }
      if (!real) g16[s] = V8<T>{};
      g = wide<T>(g16[s]);
      dz[s] = sum8(g * o);
      const f32x8 ez = g * rz[s];
      eh[s] = narrow<T>(ez);
      el[s] = narrow<T>(ez - wide<T>(eh[s]));
    }
    if constexpr (POLA) {
      dz[0] = -both_halves(dz[0]) * rz[0];
      dz[1] = -both_halves(dz[1]) * rz[1];
    } else {
      dz[0] = dz[1] = -both_halves(dz[0] + dz[1]) * rz[0];
    }
    __builtin_amdgcn_sched_barrier(0);  // (registers: one part after the other)
#pragma unroll
    for (int s = 0; s < 2; ++s) {
      const f32x8 fb = wide<T>(f.f[2 + s]);
      if constexpr (POLA) {
        const f32x8 fa = wide<T>(f.f[s]);
        dkm[s] += fa * dz[0] + fb * dz[1];
        dkm[2 * KF - 2 + s] += fb * dz[0] + fa * dz[1];
      } else {
        dkm[s] += fb * dz[0];
      }
    }
    __builtin_amdgcn_sched_barrier(0);
    wave_sync();  // the previous tile has been read
#pragma unroll
    for (int i = 0; i < 4; ++i) *reinterpret_cast<V8<T>*>(ft + place64(p.t, 2 * i + p.kb)) = real ? f.f[i] : V8<T>{};
#pragma unroll
    for (int s = 0; s < 2; ++s) {
      *reinterpret_cast<V8<T>*>(et + place64(p.t, 2 * s + p.kb)) = eh[s];
      *reinterpret_cast<V8<T>*>(et + place64(p.t, 4 + 2 * s + p.kb)) = el[s];
    }
    wave_sync();
#pragma unroll
    for (int ks = 0; ks < 2; ++ks) {
      const V8<T> th = tokens_of<T, true>(et, p.lane, 0, ks), tl = tokens_of<T, true>(et, p.lane, 1, ks);
#pragma unroll
      for (int fb = 0; fb < KF; ++fb) {
        const V8<T> ff = tokens_of<T, true>(ft, p.lane, fb, ks);
        acc[fb] = mma(ff, th, acc[fb]);
        acc[fb] = mma(ff, tl, acc[fb]);
      }
    }
    __builtin_amdgcn_sched_barrier(0);
    // gradient of the features: M^T (do / z) + dz (mean key); the denominator goes with the value channels, 16 a step
    f32x16 df[KF];
#pragma unroll
    for (int fb = 0; fb < KF; ++fb) {
#pragma unroll
      for (int ks = 0; ks < 2; ++ks) {
        const unsigned char* m = ws + kM;
        const f32x16 part = mma(tokens_of<T, POLA, true>(m + D * kRow, p.lane, fb, ks), g16[ks],
                                mma(tokens_of<T, POLA, true>(m, p.lane, fb, ks), g16[ks], zero16()));
        const float by = undo * rz[ks];
#pragma unroll
        for (int i = 0; i < 16; ++i) df[fb][i] = ks ? fmaf(part[i], by, df[fb][i]) : part[i] * by;
      }
    }
    if (t0 + 32 * p.subs < t_end) fetch(next, t0 + 32 * p.subs);
    __builtin_amdgcn_sched_barrier(0);
#pragma unroll
    for (int s = 0; s < 2; ++s) {
      const f32x8 ka = load_f8(km + 16 * s + 8 * p.kb);
      f32x8 ga, gb;
      if constexpr (POLA) {
        const f32x8 kn = load_f8(km + 32 + 16 * s + 8 * p.kb);
        ga = ka * dz[0] + kn * dz[1];
        gb = kn * dz[0] + ka * dz[1];
      } else {
        ga = f32x8{};
        gb = ka * dz[0];
      }
#pragma unroll
      for (int e = 0; e < 8; ++e) {
        ga[e] += df[0][8 * s + e];
        if constexpr (POLA) gb[e] += df[KF - 1][8 * s + e];
      }
      const V8<T> dx = narrow<T>(features_grad<POLA>(wide<T>(r.q[s]), k, s, r.cs[s], ga, gb, dscale[s], dpower[s]));
      if (real) *reinterpret_cast<V8<T>*>(piece(dqs, a.dq_row, t0, p.t, p.kb) + 16 * s) = dx;
      __builtin_amdgcn_sched_barrier(0);
    }
    r = next;
  }
  const int part = blockIdx.x * p.subs + p.sub;
  float* to = partial + (head * parts + part) * kSlot<POLA>;
#pragma unroll
  for (int fb = 0; fb < KF; ++fb)
#pragma unroll
    for (int i = 0; i < 16; ++i) {
      const int ff = 32 * fb + 8 * (i >> 2) + 4 * p.kb + (i & 3);
      to[ff * D + p.t] = acc[fb][i];
    }
#pragma unroll
  for (int i = 0; i < KF; ++i) store_sums(dkm[2 * i], dkm[2 * i + 1], to + E + 32 * i, p);
  if constexpr (POLA) {
    stats_factors(k, dscale, dpower);
    store_stats(dscale, dpower, stats + ((int64_t)b * parts + part) * 2 * C, C, p);
  }
}

// ---------------------------------------------------------------------------------------------------------------
// backward over the keys: gradients of keys and values.  A wave keeps one tile of tokens and walks the batches of its group (the
// gradient of the positional term is a sum over them, held in registers).
// ---------------------------------------------------------------------------------------------------------------
template <typename T, bool POLA>
__global__ __launch_bounds__(kThreads, POLA ? 2 : 3) void keys_kernel(Attn a, const T* __restrict__ planes, const float* __restrict__ dkm,
                                                                     float* __restrict__ stats, float* __restrict__ pe_partial, int groups,
                                                                     int group_heads) {
  constexpr int F = kFeatures<POLA>, KF = F / 32, E = F * D;
  __shared__ __attribute__((aligned(16))) float consts[kWaves][128];  // constants | mean key's gradient
  Place p(a.heads, group_heads, blockIdx.y);
  const int C = a.heads * D, h0 = p.h * D, n = a.Nk, t0 = 32 * (blockIdx.x * p.subs + p.sub), tt = min(p.t, n - 1 - t0);
  const Constants<T, POLA> k(consts[threadIdx.x >> 6], a, p);
  float* mean = consts[threadIdx.x >> 6] + 64;
  f32x8 dscale[2] = {}, dpower[2] = {}, dpe[2] = {};
  struct Rows {
    V8<T> k[2], v[2], more[2];
  } r;
  auto fetch = [&](int b) {
#pragma unroll
    for (int s = 0; s < 2; ++s) {
      r.k[s] = load8(piece((const T*)a.k + (int64_t)b * n * a.k_row + h0, a.k_row, t0, tt, p.kb) + 16 * s);
      r.v[s] = load8(piece((const T*)a.v + (int64_t)b * n * a.v_row + h0, a.v_row, t0, tt, p.kb) + 16 * s);
      r.more[s] = load8(piece((const T*)a.dv_more + (int64_t)b * n * C + h0, C, t0, tt, p.kb) + 16 * s);
    }
  };
  const bool real = t0 + p.t < n;
  if (t0 < n) {
    V8<T> pe[2];
    f32x8 cs[2];
    if constexpr (POLA) {
#pragma unroll
      for (int s = 0; s < 2; ++s) pe[s] = load8(piece((const T*)a.pe + h0, C, t0, tt, p.kb) + 16 * s);
    }
    load_turns<T, POLA>(a, p, t0, tt, cs);
    fetch(blockIdx.z);
    for (int b = blockIdx.z; b < a.B; b += groups) {
      asm volatile("" : "+v"(p.lane), "+v"(p.t), "+v"(p.kb));  // (as in the kernel above)
      const int64_t head = (int64_t)b * a.heads + p.h;
      wave_sync();  // (the last batch's has been read)
      if (p.lane < F) mean[p.lane] = dkm[head * kVector<POLA> + p.lane];
      const float undo = dkm[head * kVector<POLA> + F];
      wave_sync();
      f32x8 x[2];
      V8<T> v[2];
#pragma unroll
      for (int s = 0; s < 2; ++s) {
        x[s] = wide<T>(r.k[s]);
        if constexpr (POLA) x[s] += wide<T>(pe[s]);
        v[s] = r.v[s];
      }
      const Features<T> f = features_of<T, POLA>(x, k, cs);
      {
        Numerator<T, POLA> product;
        product.load(planes + head * 4 * E, p.lane);
        const f32x16 dv = product(f);
#pragma unroll
        for (int s = 0; s < 2; ++s) {
          f32x8 y = wide<T>(r.more[s]);
#pragma unroll
          for (int e = 0; e < 8; ++e) y[e] += dv[8 * s + e] * undo;
          if (real) *reinterpret_cast<V8<T>*>(piece((T*)a.dv + (int64_t)b * n * a.dv_row + h0, a.dv_row, t0, tt, p.kb) + 16 * s) = narrow<T>(y);
        }
      }
      __builtin_amdgcn_sched_barrier(0);  // (the two halves' registers one after the other)
      f32x16 df[KF];
#pragma unroll
      for (int fb = 0; fb < KF; ++fb) {
        df[fb] = zero16();
#pragma unroll
        for (int ks = 0; ks < 2; ++ks) {  // A operand [f][v]
          const T* m = planes + head * 4 * E + (32 * fb + row_of(p.t)) * D + 16 * ks + 8 * p.kb;
          df[fb] = mma(load8(m + E), v[ks], mma(load8(m), v[ks], df[fb]));
        }
      }
      if (b + groups < a.B) fetch(b + groups);
#pragma unroll
      for (int s = 0; s < 2; ++s) {
        f32x8 ga, gb;
#pragma unroll
        for (int e = 0; e < 8; ++e) {
          ga[e] = df[0][8 * s + e] * undo;
          gb[e] = POLA ? df[KF - 1][8 * s + e] * undo : 0.f;
        }
        if constexpr (POLA) ga += load_f8(mean + 16 * s + 8 * p.kb);
        gb += load_f8(mean + (POLA ? 32 : 0) + 16 * s + 8 * p.kb);  // (rotary: of the plain features)
        if (!real) ga = gb = f32x8{};
        const f32x8 dx = features_grad<POLA>(x[s], k, s, cs[s], ga, gb, dscale[s], dpower[s]);
        if constexpr (POLA) dpe[s] += dx;
        if (real) *reinterpret_cast<V8<T>*>(piece((T*)a.dk + (int64_t)b * n * a.dk_row + h0, a.dk_row, t0, tt, p.kb) + 16 * s) = narrow<T>(dx);
        __builtin_amdgcn_sched_barrier(0);
      }
    }
  }
  if constexpr (POLA) {
    if (real) {
#pragma unroll
      for (int s = 0; s < 2; ++s) {
        float* to = pe_partial + ((int64_t)blockIdx.z * n + t0 + p.t) * C + h0 + 8 * p.kb + 16 * s;
        const f32x8 v = dpe[s];
        *reinterpret_cast<f32x4*>(to) = f32x4{v[0], v[1], v[2], v[3]};
        *reinterpret_cast<f32x4*>(to + 4) = f32x4{v[4], v[5], v[6], v[7]};
      }
    }
    stats_factors(k, dscale, dpower);
    store_stats(dscale, dpower, stats + (((int64_t)blockIdx.z * gridDim.x + blockIdx.x) * p.subs + p.sub) * 2 * C, C, p);
  }
}

// ---------------------------------------------------------------------------------------------------------------
// host side
// ---------------------------------------------------------------------------------------------------------------
// heads of a workgroup: its waves' where they are whole fours or twos, otherwise the waves take tiles of one head
int group_heads(int heads) { return heads % 4 == 0 ? 4 : heads % 2 == 0 ? 2 : 1; }
// Tokens of a workgroup: `per_cu` workgroups a CU over all, whole tiles of its waves, and where sums are left no more of them than
// `most_parts` a head, which one workgroup adds up (one head, 112 x 112 tokens, rotary: 98 chunks, state 5 + finish 111 us; 25 chunks,
// 7 + 11 us, the queries' pass 7 -> 13 us).
struct Cut {
  int chunk, chunks, parts;
};
constexpr int kMostParts = 128;
Cut cut(int64_t B, int64_t n, int heads, int per_cu, int most_parts) {
  const int g = group_heads(heads), step = 32 * (kWaves / g);
  const int64_t places = B * (heads / g);
  int64_t chunks = 256 * per_cu / places;
  const int64_t most = std::min<int64_t>(cdiv64(n, step), most_parts / (kWaves / g));
  chunks = chunks < 1 ? 1 : chunks > most ? most : chunks;
  const int64_t chunk = cdiv64(cdiv64(n, chunks), step) * step;
  chunks = cdiv64(n, chunk);
  return {(int)chunk, (int)chunks, (int)(chunks * (kWaves / g))};
}
struct Work {  // floats (planes: T) of the workspace, in order
  size_t partial, stats, pe, planes, dkm;
  int key_tiles, groups, query_rows, key_rows;
};
Work work(const Attn& a) {
  const int F = a.pola ? 64 : 32, C = a.heads * D, g = group_heads(a.heads);
  const size_t heads = (size_t)a.B * a.heads;
  const Cut s = cut(a.B, a.Nk, a.heads, 2, kMostParts), q = cut(a.B, a.N, a.heads, 2, kMostParts);
  const size_t slot = F * (D + 1);
  Work w{};
  w.partial = heads * (s.parts > q.parts ? s.parts : q.parts) * slot;
  w.key_tiles = (int)cdiv64(a.Nk, 32 * (kWaves / g));
  const int64_t places = (int64_t)w.key_tiles * (a.heads / g), most = (a.pola ? 2 : 4) * 256 / places;
  const int64_t each = cdiv64(a.B, most < 1 ? 1 : most);  // batches a workgroup, as even as can be
  w.groups = (int)cdiv64(a.B, each);
  w.query_rows = a.B * q.parts;
  w.key_rows = w.groups * w.key_tiles * (kWaves / g);
  w.stats = a.pola ? (size_t)(w.query_rows + w.key_rows) * 2 * C : 0;
  w.pe = a.pola ? (size_t)w.groups * a.Nk * C : 0;
  w.planes = heads * 4 * F * D;
  w.dkm = heads * (F + 8);
  return w;
}

template <typename T, bool POLA> void fwd_t(const Attn& a, hipStream_t st) {
  const int g = group_heads(a.heads);
  const Cut s = cut(a.B, a.Nk, a.heads, 2, kMostParts), o = cut(a.B, a.N, a.heads, POLA ? 2 : 4, 1 << 30);
  const dim3 block(kThreads);
  float* partial = (float*)a.workspace;
  state_kernel<T, POLA><<<dim3(s.chunks, a.heads / g, a.B), block, 0, st>>>(a, partial, s.chunk, s.parts, g);
  finish_kernel<T, POLA><<<dim3(a.B * a.heads), dim3(kFinishThreads), 0, st>>>(partial, s.parts, 1.f / (float)a.Nk, (T*)a.planes, a.km);
  output_kernel<T, POLA><<<dim3(o.chunks, a.heads / g, a.B), block, 0, st>>>(a, o.chunk, g);
}

struct Carved {
  float *partial, *stats, *pe, *dkm;
  void* planes;
};
Carved carve(const Attn& a, const Work& w) {
  Carved c;
  c.partial = (float*)a.workspace;
  c.stats = c.partial + align_up(w.partial, 64);
  c.pe = c.stats + align_up(w.stats, 64);
  c.dkm = c.pe + align_up(w.pe, 64);
  c.planes = c.dkm + align_up(w.dkm, 64);
  return c;
}

template <typename T, bool POLA> int bwd_queries_t(const Attn& a, hipStream_t st) {
  const int g = group_heads(a.heads);
  const Cut q = cut(a.B, a.N, a.heads, 2, kMostParts);
  const Carved c = carve(a, work(a));
  constexpr int kLds = kWaves * kQueriesWave<POLA>;
  static thread_local bool configured = false;
  if (kLds > 64 * 1024 && !configured) {
    const hipError_t e = hipFuncSetAttribute(reinterpret_cast<const void*>(queries_kernel<T, POLA>),
                                             hipFuncAttributeMaxDynamicSharedMemorySize, kLds);
    if (e != hipSuccess) {
      set_error("cannot reserve %d bytes of LDS: %s", kLds, hipGetErrorString(e));
      return kErrLaunch;
    }
    configured = true;
  }
  queries_kernel<T, POLA><<<dim3(q.chunks, a.heads / g, a.B), dim3(kThreads), kLds, st>>>(a, c.partial, c.stats, q.chunk, q.parts, g);
  finish_kernel<T, POLA><<<dim3(a.B * a.heads), dim3(kFinishThreads), 0, st>>>(c.partial, q.parts, 1.f / (float)a.Nk, (T*)c.planes, c.dkm);
  return kOk;
}

template <typename T, bool POLA> void bwd_keys_t(const Attn& a, int dtype, hipStream_t st) {
  const int g = group_heads(a.heads);
  const Work w = work(a);
  const Carved c = carve(a, w);
  keys_kernel<T, POLA><<<dim3(w.key_tiles, a.heads / g, w.groups), dim3(kThreads), 0, st>>>(
      a, (const T*)c.planes, c.dkm, c.stats + (size_t)w.query_rows * 2 * a.heads * D, c.pe, w.groups, g);
  if (POLA)
    blocks::features_finish(a.heads * D, w.query_rows + w.key_rows, c.stats, a.scale, {a.power, a.alpha}, a.dscale, a.dpower, w.groups, (int64_t)a.Nk * a.heads * D,
                            c.pe, a.dpe, dtype, st);
}

template <typename Go> void by_kind(const Attn& a, int dtype, Go go) {
  if (dtype == kF16) a.pola ? go((_Float16*)nullptr, std::true_type{}) : go((_Float16*)nullptr, std::false_type{});
  else a.pola ? go((__bf16*)nullptr, std::true_type{}) : go((__bf16*)nullptr, std::false_type{});
}

}  // namespace

size_t workspace_bytes(const Attn& a) {
  const Work w = work(a);
  return sizeof(float) * (align_up(w.partial, 64) + align_up(w.stats, 64) + align_up(w.pe, 64) + align_up(w.dkm, 64)) + 2 * w.planes;
}
size_t planes_elements(const Attn& a) { return (size_t)a.B * a.heads * 4 * (a.pola ? 64 : 32) * D; }

void forward(const Attn& a, int dtype, hipStream_t st) {
  by_kind(a, dtype, [&](auto* t, auto pola) { fwd_t<std::remove_pointer_t<decltype(t)>, decltype(pola)::value>(a, st); });
}
int backward_queries(const Attn& a, int dtype, hipStream_t st) {
  int rc = kOk;
  by_kind(a, dtype, [&](auto* t, auto pola) { rc = bwd_queries_t<std::remove_pointer_t<decltype(t)>, decltype(pola)::value>(a, st); });
  return rc;
}
void backward_keys(const Attn& a, int dtype, hipStream_t st) {
  by_kind(a, dtype, [&](auto* t, auto pola) { bwd_keys_t<std::remove_pointer_t<decltype(t)>, decltype(pola)::value>(a, dtype, st); });
}

}  // namespace rows
}  // namespace fbla
