// Weight and bias gradient of a projection over token rows: dW[m][n] = sum_t g[t][m] x[t][n], db[m] = sum_t g[t][m],
// (the blocks' nn.Linear layers: layers/mlla.py:56, rala.py:31, focused_la.py:26-27, polaformer.py:24-25).
//
// The contraction runs over the tokens (1e4 .. 1e5), the result is a few hundred on a side: a GEMM that tiles the result
// alone leaves the GPU to a dozen workgroups (the library's, bf16: 128 x 64 over 200704 tokens 419 us, 512 x 256 over
// 50176 tokens 188 us, plus 32 us of column sums each for the bias; here, with the bias, 23 and 35 us).  So the
// tokens are split: a workgroup owns a 128 x 128 tile of the result and one chunk of the tokens, the chunks' fp32 sums
// are added in chunk order by a second kernel and rounded once.
//
// Tile: four waves, each a 64 x 64 quarter.  16 bits: steps of 64 tokens arrive flat (16 bytes per lane, whole rows) and are staged
// in LDS row-major; both operands are read out of it with the transposing read.  Per step a wave reads 16 KiB of LDS for
// 16 MFMAs of 32x32x16, which take about as long: bound by LDS and matrix cores together where the result has many
// tiles, by HBM where it has one or two.  The next step's rows are in registers meanwhile; two LDS buffers, one barrier per
// step.  fp32: steps of 32 tokens, the fp32 matrix instruction takes its operands from the rows as they lie;
// bound by it where there are tiles enough (512 x 256 over 50176 tokens 558 + 32 -> 136 us, 104 TFLOP/s of 153).
#include <hip/hip_runtime.h>

#include <type_traits>

#include "fbla_mfma_shared.h"

namespace fbla {
namespace linear {

namespace {

constexpr int kThreads = 256;
constexpr int kTile = 128;               // rows and columns of the result per workgroup
constexpr int kStepBytes = 64 * 128 * 2; // one operand's rows of a step: 64 tokens of 16 bits, 32 of fp32
constexpr int kLeastChunk = 256;
// What sums of g alone and over the chunks are added in: 64 bits for fp32, so that the bias gradient is no further from exact
// than column sums in a tree (50176 tokens x 512: 2.1e-7 in 32 bits, 4.8e-8 so; the library's 1.9e-7), 32 for 16-bit types.
template <typename T> using Sum = std::conditional_t<sizeof(T) == 4, double, float>;
template <typename T> struct Step {
  static constexpr int kVec = 16 / sizeof(T), kRowBytes = kTile * sizeof(T), kTokens = kStepBytes / kRowBytes;
  static constexpr int kRowPieces = kTile / kVec, kRows = kThreads / kRowPieces;  // rows that the threads move at a time
};

typedef uint32_t u32x4 __attribute__((ext_vector_type(4)));
typedef uint32_t u32x2 __attribute__((ext_vector_type(2)));
typedef short i16x4 __attribute__((ext_vector_type(4)));
typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
typedef _Float16 f16x8 __attribute__((ext_vector_type(8)));
typedef float f32x4 __attribute__((ext_vector_type(4)));
using mfma::f32x16;

template <typename T> __device__ __forceinline__ f32x16 mma(u32x4 a, u32x4 b, f32x16 c);
template <> __device__ __forceinline__ f32x16 mma<__bf16>(u32x4 a, u32x4 b, f32x16 c) {
  return __builtin_amdgcn_mfma_f32_32x32x16_bf16(__builtin_bit_cast(bf16x8, a), __builtin_bit_cast(bf16x8, b), c, 0, 0, 0);
}
template <> __device__ __forceinline__ f32x16 mma<_Float16>(u32x4 a, u32x4 b, f32x16 c) {
  return __builtin_amdgcn_mfma_f32_32x32x16_f16(__builtin_bit_cast(f16x8, a), __builtin_bit_cast(f16x8, b), c, 0, 0, 0);
}

// eight tokens of one feature out of a row-major tile: two transposing reads of four
__device__ __forceinline__ u32x4 tr_fragment(const unsigned char* tile, int off0, int off1) {
  typedef i16x4 __attribute__((address_space(3))) * lds_ptr;
  const u32x2 a = __builtin_bit_cast(u32x2, __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_ptr)(tile + off0)));
  const u32x2 b = __builtin_bit_cast(u32x2, __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_ptr)(tile + off1)));
  return u32x4{a[0], a[1], b[0], b[1]};
}

// One step's products for a wave's 64 x 64 quarter (wm, wn).
template <typename T> struct Multiply {
  static constexpr int kRowBytes = Step<T>::kRowBytes;
  // transposing reads: this lane addresses, for element half h, token 4 (s / 4) + 2 (g / 2) + h (+ 16 ks) and the four
  // features 16 (g % 2) + 4 (s % 4) .. + 3 of a fragment of 32 (g = lane / 16, s = lane % 16)
  int goff[2][2], xoff[2][2];
  __device__ __forceinline__ Multiply(int lane, int wm, int wn) {
    const int g16 = lane >> 4, s16 = lane & 15;
#pragma unroll
    for (int h = 0; h < 2; ++h)
#pragma unroll
      for (int a = 0; a < 2; ++a) {
        const int tok = 4 * (s16 >> 2) + 2 * (g16 >> 1) + h, f = 32 * a + 16 * (g16 & 1) + 4 * (s16 & 3);
        const int fg = 64 * wm + f, fx = 64 * wn + f;
        goff[a][h] = mfma::swz<kRowBytes>(tok, fg >> 3) + ((fg >> 2) & 1) * 8;
        xoff[a][h] = mfma::swz<kRowBytes>(tok, fx >> 3) + ((fx >> 2) & 1) * 8;
      }
  }
  static __device__ __forceinline__ int place(int row, int piece) { return mfma::swz<kRowBytes>(row, piece); }
  __device__ __forceinline__ void operator()(const unsigned char* gt, const unsigned char* xt, f32x16 (&acc)[2][2]) const {
#pragma unroll
    for (int ks = 0; ks < Step<T>::kTokens / 16; ++ks) {
      u32x4 ga[2], xb[2];
#pragma unroll
      for (int a = 0; a < 2; ++a) {
        ga[a] = tr_fragment(gt + ks * 16 * kRowBytes, goff[a][0], goff[a][1]);
        xb[a] = tr_fragment(xt + ks * 16 * kRowBytes, xoff[a][0], xoff[a][1]);
      }
#pragma unroll
      for (int a = 0; a < 2; ++a)
#pragma unroll
        for (int b = 0; b < 2; ++b) acc[a][b] = mma<T>(ga[a], xb[b], acc[a][b]);
    }
  }
};
// fp32: the operand of 32x32x2 is one feature per lane and a token per half wave, which is a row of the tile as it lies
template <> struct Multiply<float> {
  int goff, xoff;
  __device__ __forceinline__ Multiply(int lane, int wm, int wn)
      : goff((lane >> 5) * kTile + 64 * wm + (lane & 31)), xoff((lane >> 5) * kTile + 64 * wn + (lane & 31)) {}
  static __device__ __forceinline__ int place(int row, int piece) { return row * Step<float>::kRowBytes + piece * 16; }
  __device__ __forceinline__ void operator()(const unsigned char* gt, const unsigned char* xt, f32x16 (&acc)[2][2]) const {
    const float* g = reinterpret_cast<const float*>(gt) + goff;
    const float* x = reinterpret_cast<const float*>(xt) + xoff;
#pragma unroll
    for (int ks = 0; ks < Step<float>::kTokens / 2; ++ks)
#pragma unroll
      for (int a = 0; a < 2; ++a)
#pragma unroll
        for (int b = 0; b < 2; ++b)
          acc[a][b] = __builtin_amdgcn_mfma_f32_32x32x2f32(g[2 * ks * kTile + 32 * a], x[2 * ks * kTile + 32 * b], acc[a][b],
                                                           0, 0, 0);
  }
};

// partial [chunk][M][N], bias_partial [chunk][M] (null: no bias)
template <typename T>
__global__ __launch_bounds__(kThreads, 2) void wgrad_kernel(const T* __restrict__ g, int64_t g_row, const T* __restrict__ x,
                                                            int64_t x_row, int64_t tokens, int M, int N, int chunk,
                                                            int tiles_n, float* __restrict__ partial,
                                                            float* __restrict__ bias_partial) {
  extern __shared__ __attribute__((aligned(16))) unsigned char smem[];  // 2 x (g step, x step)
  // The tiles of a chunk read the same rows: they run on one XCD (workgroup i is on XCD i % 8), whose L2 then fetches them
  // once.  Chunks beyond the last multiple of eight keep the plain order, and so do chunks of the shortest length, which end
  // before that pays (with / without, bf16 with bias: 512 x 256 over 50176 tokens, chunks of 832, 34.5 / 42.6 us; 640 x 640
  // over 8192, chunks of 448, 24.9 / 29.6; over 4096, chunks of 256, 23.3 / 20.9).
  int tile, c;
  {
    const int tiles = gridDim.x, i = blockIdx.x + tiles * blockIdx.y;
    const int together = chunk > kLeastChunk ? (int)gridDim.y / 8 * 8 * tiles : 0;
    c = i < together ? i / (8 * tiles) * 8 + i % 8 : i / tiles;
    tile = i < together ? i / 8 % tiles : i % tiles;
  }
  const int m0 = tile / tiles_n * kTile, n0 = tile % tiles_n * kTile;
  const int64_t t_begin = (int64_t)c * chunk;
  const int len = (int)min((int64_t)chunk, tokens - t_begin);  // >= 1: the host counts the chunks
  const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int wm = wave >> 1, wn = wave & 1;

  // thread t moves one piece of rows t / kRowPieces + kRows i of a step; what lies outside the matrices or the chunk is zero
  constexpr int V = Step<T>::kVec, kRows = Step<T>::kRows, kTokens = Step<T>::kTokens;
  const int prow = tid / Step<T>::kRowPieces, pch = tid % Step<T>::kRowPieces;
  const bool g_piece = m0 + V * pch < M, x_piece = n0 + V * pch < N;
  const T* gp = g + (t_begin + prow) * g_row + m0 + V * pch;
  const T* xp = x + (t_begin + prow) * x_row + n0 + V * pch;
  auto load_step = [&](u32x4(&dst)[4], const T* src, int64_t row, int base, bool has) {
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      dst[i] = u32x4{0u, 0u, 0u, 0u};
      if (has && base + prow + kRows * i < len) dst[i] = *reinterpret_cast<const u32x4*>(src + (base + kRows * i) * row);
    }
  };
  auto stash = [&](const u32x4(&src)[4], unsigned char* to) {
#pragma unroll
    for (int i = 0; i < 4; ++i) *reinterpret_cast<u32x4*>(to + Multiply<T>::place(prow + kRows * i, pch)) = src[i];
  };

  const Multiply<T> multiply(lane, wm, wn);
  f32x16 acc[2][2];
#pragma unroll
  for (int a = 0; a < 2; ++a)
#pragma unroll
    for (int b = 0; b < 2; ++b)
#pragma unroll
      for (int r = 0; r < 16; ++r) acc[a][b][r] = 0.f;
  const bool with_bias = bias_partial != nullptr && n0 == 0;
  Sum<T> bias[V];
#pragma unroll
  for (int j = 0; j < V; ++j) bias[j] = 0;

  u32x4 grow[4], xrow[4];
  load_step(grow, gp, g_row, 0, g_piece);
  load_step(xrow, xp, x_row, 0, x_piece);
  int buf = 0;
  for (int base = 0; base < len; base += kTokens) {
    unsigned char* gt = smem + buf * 2 * kStepBytes;
    unsigned char* xt = gt + kStepBytes;
    stash(grow, gt);
    stash(xrow, xt);
    if (with_bias) {
      union Row { u32x4 w; T e[V]; };
      if constexpr (sizeof(T) == 4) {  // four rows in a tree, then to the sum
        Row p[4];
#pragma unroll
        for (int i = 0; i < 4; ++i) p[i].w = grow[i];
#pragma unroll
        for (int j = 0; j < V; ++j) bias[j] += (p[0].e[j] + p[1].e[j]) + (p[2].e[j] + p[3].e[j]);
      } else {
#pragma unroll
        for (int i = 0; i < 4; ++i) {
          Row p;
          p.w = grow[i];
#pragma unroll
          for (int j = 0; j < V; ++j) bias[j] += (float)p.e[j];
        }
      }
    }
    load_step(grow, gp, g_row, base + kTokens, g_piece);
    load_step(xrow, xp, x_row, base + kTokens, x_piece);
    __syncthreads();  // the step is in LDS; every wave is done with the step before it, whose buffer is written next
    multiply(gt, xt, acc);
    buf ^= 1;
  }

  float* out = partial + (int64_t)c * M * N;
#pragma unroll
  for (int a = 0; a < 2; ++a)
#pragma unroll
    for (int b = 0; b < 2; ++b)
#pragma unroll
      for (int r = 0; r < 16; ++r) {
        const int m = m0 + 64 * wm + 32 * a + 8 * (r >> 2) + 4 * (lane >> 5) + (r & 3);
        const int n = n0 + 64 * wn + 32 * b + (lane & 31);
        if (m < M && n < N) out[(int64_t)m * N + n] = acc[a][b][r];
      }
  if (with_bias) {
    __syncthreads();  // all waves have read their last step
    Sum<T>* sums = reinterpret_cast<Sum<T>*>(smem);  // [kRows][128]
#pragma unroll
    for (int j = 0; j < V; ++j) sums[prow * kTile + V * pch + j] = bias[j];
    __syncthreads();
    if (tid < kTile && m0 + tid < M) {
      Sum<T> v = 0;
#pragma unroll
      for (int i = 0; i < kRows; ++i) v += sums[i * kTile + tid];
      bias_partial[(int64_t)c * M + m0 + tid] = (float)v;
    }
  }
}

// out[i] = sum over the chunks of partial[chunk][i]; 16 threads share four neighbouring results (chunks part, part + 16,
// ..), their sums are added in order.  Workgroups past the `count` weights take the `bias_count` bias entries.
template <typename T>
__global__ __launch_bounds__(kThreads) void wgrad_finish_kernel(const float* __restrict__ partial, int count,
                                                                T* __restrict__ out, const float* __restrict__ bias_partial,
                                                                int bias_count, T* __restrict__ bias_out, int chunks,
                                                                int weight_wgs) {
  constexpr int kParts = 16, kLanes = kThreads / kParts;
  using A = Sum<T>;
  __shared__ A sums[kParts][kLanes][4];
  int wg = blockIdx.x;
  if (wg >= weight_wgs) {
    wg -= weight_wgs;
    partial = bias_partial;
    count = bias_count;
    out = bias_out;
  }
  const int lane = threadIdx.x % kLanes, part = threadIdx.x / kLanes;
  const int at = (wg * kLanes + lane) * 4;  // counts are multiples of 4
  A sum[4] = {0, 0, 0, 0};
  if (at < count) {
    const float* p = partial + at;
#pragma unroll 4
    for (int c = part; c < chunks; c += kParts) {
      const f32x4 v = *reinterpret_cast<const f32x4*>(p + (int64_t)c * count);
#pragma unroll
      for (int j = 0; j < 4; ++j) sum[j] += v[j];
    }
  }
#pragma unroll
  for (int j = 0; j < 4; ++j) sums[part][lane][j] = sum[j];
  __syncthreads();
  if (part == 0 && at < count) {
    for (int i = 1; i < kParts; ++i)
#pragma unroll
      for (int j = 0; j < 4; ++j) sum[j] += sums[i][lane][j];
#pragma unroll
    for (int j = 0; j < 4; ++j) out[at + j] = (T)sum[j];
  }
}

int tiles(int n) { return (n + kTile - 1) / kTile; }

// Tokens of a chunk: two workgroups per CU over all tiles (one round), whole steps, at least four of them: a chunk costs
// its M x N fp32 sums on the way out and in again.
int chunk_for(int64_t tokens, int M, int N) {
  const int64_t slots = 2 * 256 / ((int64_t)tiles(M) * tiles(N));
  int64_t chunk = cdiv64(tokens, slots < 1 ? 1 : slots);
  if (chunk < kLeastChunk) chunk = kLeastChunk;
  return (int)(cdiv64(chunk, 64) * 64);
}

template <typename T>
void launch(const void* g, int64_t g_row, const void* x, int64_t x_row, int64_t tokens, int M, int N, void* dw, void* db,
            float* workspace, hipStream_t st) {
  const int chunk = chunk_for(tokens, M, N), chunks = (int)cdiv64(tokens, chunk);
  float* bias_partial = db ? workspace + (int64_t)chunks * M * N : nullptr;
  wgrad_kernel<T><<<dim3((unsigned)(tiles(M) * tiles(N)), (unsigned)chunks), dim3(kThreads), 4 * kStepBytes, st>>>(
      (const T*)g, g_row, (const T*)x, x_row, tokens, M, N, chunk, tiles(N), workspace, bias_partial);
  const int weight_wgs = (int)cdiv64((int64_t)M * N, 64), bias_wgs = db ? (M + 63) / 64 : 0;
  wgrad_finish_kernel<T><<<dim3((unsigned)(weight_wgs + bias_wgs)), dim3(kThreads), 0, st>>>(
      workspace, M * N, (T*)dw, bias_partial, M, (T*)db, chunks, weight_wgs);
}

}  // namespace

size_t wgrad_workspace_bytes(int64_t tokens, int M, int N) {
  return sizeof(float) * (size_t)cdiv64(tokens, chunk_for(tokens, M, N)) * ((size_t)M * N + M);
}

void wgrad(const void* g, int64_t g_row, const void* x, int64_t x_row, int64_t tokens, int M, int N, void* dw, void* db,
           float* workspace, int dtype, hipStream_t st) {
  if (dtype == kF16) launch<_Float16>(g, g_row, x, x_row, tokens, M, N, dw, db, workspace, st);
  else if (dtype == kF32) launch<float>(g, g_row, x, x_row, tokens, M, N, dw, db, workspace, st);
  else launch<__bf16>(g, g_row, x, x_row, tokens, M, N, dw, db, workspace, st);
}

}  // namespace linear
}  // namespace fbla
