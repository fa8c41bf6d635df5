// Depth-wise convolution over token rows: x is [B, H*W, C] with the channels adjacent (the layout in which the
// blocks' projections leave their tokens), every channel c convolved on the H x W grid with the K x K taps
// w[c % Cw] (Cw = C: LePE of layers/mlla.py:57,92 and rala.py:32,58; Cw = head dim: the value convolution of the
// PVT-style blocks, focused_la.py:88-93, polaformer.py:97-101, one filter per channel of a head).
//
// Bound: HBM for the bytes (one read, one write) and the vector ALU for the K*K multiply-adds per element, about
// equally at K = 5.  A lane owns 16 bytes of channels and a strip of 7 or 8 neighbouring outputs of one grid row: the
// STRIP + K - 1 input pieces of one tap row sit in registers and serve K * STRIP products, the taps come from LDS as
// fp32 (a piece of them is read once per strip, not once per output).  Rows are re-read K times out of the caches.
// 64 x 28x28 x 256 in bf16, 5x5: 25 us (51 MB, 2.1 TB/s); 64 x 56x56 x 64, 3x3: 18 us.
// No matrix instruction: a depth-wise filter has no channel contraction to give one (the library's implicit-GEMM
// weight gradient spends its time on padding for exactly that reason: 27.7 ms at 64 x 56x56 x 64 channels, 3x3, bf16).
#include <hip/hip_runtime.h>

#include <type_traits>

#include "fbla_kernels.h"

namespace fbla {
namespace dwconv {

namespace {

constexpr int kThreads = 256;
constexpr float kLargest = 3.40282347e38f;  // of fp32
constexpr int kFinishParts = 32;    // threads that share the terms of one filter's gradient
constexpr int kBlockChannels = 64;  // channels of a workgroup: 128-byte (16-bit) or 256-byte (fp32) pieces of a row

typedef uint32_t u32x4 __attribute__((ext_vector_type(4)));

template <typename T> struct Lane {
  static constexpr int kVec = 16 / sizeof(T);
  static constexpr int kLanes = kBlockChannels / kVec;  // lanes across the channels of a workgroup
  static constexpr int kWorkers = kThreads / kLanes;    // strips in flight per workgroup
};

// What the products of one output are added in: 64 bits for fp32 (as torch's convolution adds them; in 32 bits a result is
// 9.1e-8 from exact at 5x5, so it is 2.5e-8; 64 x 28x28 x 256 32 and 39 us), 32 for 16-bit types.
template <typename T> using Sum = std::conditional_t<sizeof(T) == 4, double, float>;
__device__ __forceinline__ float mul_add(float a, float b, float c) { return fmaf(a, b, c); }
__device__ __forceinline__ double mul_add(double a, double b, double c) { return fma(a, b, c); }

template <typename T> union Piece {
  u32x4 w;
  T e[16 / sizeof(T)];
};

// the input pieces [first, first + COUNT) of one grid row; columns outside the grid are zero.  Unconditional loads from
// clamped columns: a guarded load would be waited for before the next one is requested.
template <typename T, int COUNT>
__device__ __forceinline__ void load_row(const T* __restrict__ row, int64_t col_stride, int first, int W,
                                         Piece<T> (&out)[COUNT]) {
#pragma unroll
  for (int i = 0; i < COUNT; ++i) {
    const int col = first + i;
    const int at = col < 0 ? 0 : (col < W ? col : W - 1);
    out[i].w = *reinterpret_cast<const u32x4*>(row + at * col_stride);
  }
#pragma unroll
  for (int i = 0; i < COUNT; ++i) {
    const int col = first + i;
    if (col < 0 || col >= W) out[i].w = u32x4{0, 0, 0, 0};
  }
}

template <typename T, int K, int STRIP>
__global__ __launch_bounds__(kThreads) void conv_kernel(Conv a, int strips_per_row, int nstrips, int flip) {
  constexpr int V = Lane<T>::kVec, P = K / 2, IN = STRIP + K - 1;
  __shared__ float taps[K * K][kBlockChannels];
  __shared__ int endless_of[kThreads / 64];  // a wave staged a tap that is infinite or NaN
  const int c0 = blockIdx.y * kBlockChannels;
  int endless = 0;
  for (int i = threadIdx.x; i < K * K * kBlockChannels; i += kThreads) {
    const int tap = i / kBlockChannels, c = c0 + i % kBlockChannels;
    const T* w = static_cast<const T*>(a.w) + (int64_t)(c % a.Cw) * (K * K);
    const float v = c < a.C ? (float)w[flip ? K * K - 1 - tap : tap] : 0.f;
    taps[tap][i % kBlockChannels] = v;
    endless |= !(fabsf(v) <= kLargest);
  }
  endless = __ballot(endless) != 0;
  if (threadIdx.x % 64 == 0) endless_of[threadIdx.x / 64] = endless;
  __syncthreads();
  const int lane = threadIdx.x % Lane<T>::kLanes, worker = threadIdx.x / Lane<T>::kLanes;
  const int cl = lane * V, c = c0 + cl;
  const int strip = blockIdx.x * Lane<T>::kWorkers + worker;
  if (strip >= nstrips || c >= a.C) return;
  const int sx = strip % strips_per_row, yb = strip / strips_per_row;
  const int y = yb % a.H, b = yb / a.H;
  const int x0 = sx * STRIP;

  using A = Sum<T>;
  A acc[STRIP][V];
  if (a.bias) {
#pragma unroll
    for (int j = 0; j < V; ++j) {
      const A v = (A)static_cast<const T*>(a.bias)[(c + j) % a.Cw];
#pragma unroll
      for (int t = 0; t < STRIP; ++t) acc[t][j] = v;
    }
  } else {
#pragma unroll
    for (int t = 0; t < STRIP; ++t)
#pragma unroll
      for (int j = 0; j < V; ++j) acc[t][j] = 0;
  }

  const T* xb = static_cast<const T*>(a.x) + (int64_t)b * a.x_batch + c;
#pragma unroll 1
  for (int ky = 0; ky < K; ++ky) {
    const int yy = y + ky - P;
    if (yy < 0 || yy >= a.H) continue;
    Piece<T> in[IN];
    load_row<T, IN>(xb + (int64_t)yy * a.W * a.x_row, a.x_row, x0 - P, a.W, in);
#pragma unroll
    for (int kx = 0; kx < K; ++kx) {
      A w[V];
#pragma unroll
      for (int j = 0; j < V; ++j) w[j] = taps[ky * K + kx][cl + j];
#pragma unroll
      for (int t = 0; t < STRIP; ++t)
#pragma unroll
        for (int j = 0; j < V; ++j) acc[t][j] = mul_add(w[j], (A)in[t + kx].e[j], acc[t][j]);
    }
  }

  T* yo = static_cast<T*>(a.y) + (int64_t)b * a.y_batch + ((int64_t)y * a.W + x0) * a.y_row + c;
  endless = 0;
#pragma unroll
  for (int i = 0; i < kThreads / 64; ++i) endless |= endless_of[i];
  if (endless) {  // 0 times such a tap is not 0: once more, the columns around the grid left out
#pragma unroll 1
    for (int t = 0; t < STRIP && x0 + t < a.W; ++t) {
      A sum[V];
#pragma unroll
      for (int j = 0; j < V; ++j) sum[j] = a.bias ? (A)static_cast<const T*>(a.bias)[(c + j) % a.Cw] : 0;
#pragma unroll 1
      for (int tap = 0; tap < K * K; ++tap) {
        const int yy = y + tap / K - P, xx = x0 + t + tap % K - P;
        if (yy < 0 || yy >= a.H || xx < 0 || xx >= a.W) continue;
        Piece<T> in;
        in.w = *reinterpret_cast<const u32x4*>(xb + ((int64_t)yy * a.W + xx) * a.x_row);
#pragma unroll
        for (int j = 0; j < V; ++j) sum[j] = mul_add((A)taps[tap][cl + j], (A)in.e[j], sum[j]);
      }
      Piece<T> out;
#pragma unroll
      for (int j = 0; j < V; ++j) out.e[j] = (T)sum[j];
      *reinterpret_cast<u32x4*>(yo + t * a.y_row) = out.w;
    }
    return;
  }
#pragma unroll
  for (int t = 0; t < STRIP; ++t) {
    if (x0 + t < a.W) {
      Piece<T> out;
#pragma unroll
      for (int j = 0; j < V; ++j) out.e[j] = (T)acc[t][j];
      *reinterpret_cast<u32x4*>(yo + t * a.y_row) = out.w;
    }
  }
}

// Weight and bias gradient: partial[chunk][ky][kx][C] = sum over the chunk's strips of g[y, x] * x[y + ky - P,
// x + kx - P], the bias gradient in row K of ky = 0.  One tap row per workgroup (blockIdx.z): K * V accumulators per
// lane, kept over all strips of the chunk, added over the workgroup's strips at the end in a fixed order (fp32: sums of g alone
// and sums over chunks in 64 bits, so that the bias gradient is no further from exact than column sums in a tree).  The K
// workgroups of a chunk fetch the same rows (out of the caches), what bounds it is the latency of a strip's loads.  16-bit types up to
// 5x5: two of a lane's channels are fp32 at a time, so that three waves fit a SIMD (all eight: 173 VGPRs at 5x5, two waves), and the
// grid is the three workgroups a CU that run at once.  bf16: 64 x 28x28 x 256, 5x5, 46 -> 33 us (51 MB); 64 x 56x56 x 64, 3x3, 29 -> 22 us.
// fp32 has three or four waves as it is and 7x7 of 16 bits two either way: all channels at once and a grid of four workgroups a CU
// (7x7, 64 x 28x28 x 256 bf16 59 us, 65 in parts with three a CU; fp32 77 and 90; 5x5, 64 x 28x28 x 64 fp32 22 and 25).
template <typename T> constexpr bool grad_in_parts(int K) { return sizeof(T) == 2 && K < 7; }
template <typename T, int K, int STRIP>
__global__ __launch_bounds__(kThreads) void grad_kernel(Conv a, const T* __restrict__ g, int64_t g_batch, int64_t g_row,
                                                        float* __restrict__ partial, int strips_per_row, int nstrips) {
  constexpr int V = Lane<T>::kVec, P = K / 2, IN = STRIP + K - 1;
  constexpr int kWaves = kThreads / 64, kAtOnce = grad_in_parts<T>(K) ? 2 : V;
  const int ky = blockIdx.z, c0 = blockIdx.y * kBlockChannels;
  const int lane = threadIdx.x % Lane<T>::kLanes, worker = threadIdx.x / Lane<T>::kLanes;
  const int cl = lane * V, c = c0 + cl;
  using A = Sum<T>;
  float acc[K][V];
  A total[V];  // of g
#pragma unroll
  for (int j = 0; j < V; ++j) {
    total[j] = 0;
#pragma unroll
    for (int k = 0; k < K; ++k) acc[k][j] = 0.f;
  }

  if (c < a.C) {
    const T* xc = static_cast<const T*>(a.x) + c;
    for (int strip = blockIdx.x * Lane<T>::kWorkers + worker; strip < nstrips; strip += gridDim.x * Lane<T>::kWorkers) {
      const int sx = strip % strips_per_row, yb = strip / strips_per_row;
      const int y = yb % a.H, b = yb / a.H;
      const int x0 = sx * STRIP, yy = y + ky - P;
      const bool inside = yy >= 0 && yy < a.H;
      if (!inside && ky != 0) continue;
      Piece<T> gv[STRIP], in[IN];
      load_row<T, STRIP>(g + (int64_t)b * g_batch + (int64_t)y * a.W * g_row + c, g_row, x0, a.W, gv);
      load_row<T, IN>(xc + (int64_t)b * a.x_batch + (int64_t)(inside ? yy : y) * a.W * a.x_row, a.x_row, x0 - P, a.W, in);
      if (kAtOnce == V || ky == 0) {  // (no other workgroup's is kept; the branch costs the kernels without parts registers)
#pragma unroll
        for (int t = 0; t < STRIP; ++t)
#pragma unroll
          for (int j = 0; j < V; ++j) total[j] += (A)gv[t].e[j];
      }
      if (inside) {
#pragma unroll
        for (int j0 = 0; j0 < V; j0 += kAtOnce) {
#pragma unroll
          for (int kx = 0; kx < K; ++kx)
#pragma unroll
            for (int t = 0; t < STRIP; ++t)
#pragma unroll
              for (int j = j0; j < j0 + kAtOnce; ++j) acc[kx][j] = fmaf((float)gv[t].e[j], (float)in[t + kx].e[j], acc[kx][j]);
          if constexpr (kAtOnce < V) __builtin_amdgcn_sched_barrier(0);
        }
      }
    }
  }
  // The products above include zeros around the grid, which is wrong where the other factor is infinite or NaN: a lane whose
  // sums are no numbers adds the products inside the grid again, alone.
  float unbounded = 0.f;
#pragma unroll
  for (int k = 0; k < K; ++k)
#pragma unroll
    for (int j = 0; j < V; ++j) unbounded = fmaf(acc[k][j], 0.f, unbounded);
  if (unbounded != 0.f) {
#pragma unroll
    for (int k = 0; k < K; ++k)
#pragma unroll
      for (int j = 0; j < V; ++j) acc[k][j] = 0.f;
    for (int strip = blockIdx.x * Lane<T>::kWorkers + worker; strip < nstrips; strip += gridDim.x * Lane<T>::kWorkers) {
      const int yb = strip / strips_per_row, y = yb % a.H, b = yb / a.H, yy = y + ky - P;
      if (yy < 0 || yy >= a.H) continue;
      const T* gs = g + (int64_t)b * g_batch + (int64_t)y * a.W * g_row + c;
      const T* xs = static_cast<const T*>(a.x) + (int64_t)b * a.x_batch + (int64_t)yy * a.W * a.x_row + c;
      const int end = min(strip % strips_per_row * STRIP + STRIP, a.W);
#pragma unroll 1
      for (int t = strip % strips_per_row * STRIP; t < end; ++t) {
        Piece<T> gv, in;
        gv.w = *reinterpret_cast<const u32x4*>(gs + t * g_row);
#pragma unroll
        for (int kx = 0; kx < K; ++kx) {
          const int xx = t + kx - P;
          if (xx < 0 || xx >= a.W) continue;
          in.w = *reinterpret_cast<const u32x4*>(xs + xx * a.x_row);
#pragma unroll
          for (int j = 0; j < V; ++j) acc[kx][j] = fmaf((float)gv.e[j], (float)in.e[j], acc[kx][j]);
        }
      }
    }
  }
  // the strips of a wave (lanes of equal channel), then the waves, both in a fixed order
  __shared__ float sums[kWaves][K][kBlockChannels];
  __shared__ A totals[kWaves][kBlockChannels];
  const bool first = (threadIdx.x & 63) < Lane<T>::kLanes;
#pragma unroll
  for (int j = 0; j < V; ++j) {
#pragma unroll
    for (int k = 0; k < K; ++k) {
      float v = acc[k][j];
#pragma unroll
      for (int m = Lane<T>::kLanes; m < 64; m *= 2) v += __shfl_xor(v, m);
      if (first) sums[threadIdx.x / 64][k][cl + j] = v;
    }
#pragma unroll
    for (int m = Lane<T>::kLanes; m < 64; m *= 2) total[j] += __shfl_xor(total[j], m);
    if (first) totals[threadIdx.x / 64][cl + j] = total[j];
  }
  __syncthreads();
  float* out = partial + ((int64_t)blockIdx.x * K + ky) * (K + 1) * a.C;
  for (int i = threadIdx.x; i < (K + 1) * kBlockChannels; i += kThreads) {
    const int k = i / kBlockChannels, j = i % kBlockChannels;
    if (c0 + j < a.C) {
      A v = 0;
#pragma unroll
      for (int w = 0; w < kWaves; ++w) v += k < K ? sums[w][k][j] : totals[w][j];
      out[k * a.C + c0 + j] = (float)v;
    }
  }
}

// dw[cw][tap], db[cw] = the partials summed over the chunks and over the channels that share the filter.  One
// workgroup per (tap or bias, 8 filters); 32 threads share a filter's terms (a few hundred: with eight of them the chain of
// loads took 18 us at 28x28 x 256, 5x5, against 5 us).
template <typename T>
__global__ __launch_bounds__(kThreads) void grad_finish_kernel(const float* __restrict__ partial, int nchunks, int K,
                                                               int C, int Cw, T* __restrict__ dw, T* __restrict__ db) {
  constexpr int kParts = kFinishParts;
  const int row = blockIdx.x;                       // tap ky * K + kx, or K * K for the bias
  const int cw = blockIdx.y * (kThreads / kParts) + threadIdx.x % (kThreads / kParts);
  const int part = threadIdx.x / (kThreads / kParts);
  const int ky = row == K * K ? 0 : row / K, kx = row == K * K ? K : row % K;
  using A = Sum<T>;
  A sum = 0;
  if (cw < Cw) {
    const int groups = C / Cw, terms = nchunks * groups;
#pragma unroll 4
    for (int i = part; i < terms; i += kParts)
      sum += partial[(((int64_t)(i / groups) * K + ky) * (K + 1) + kx) * C + (i % groups) * Cw + cw];
  }
  __shared__ A sums[kParts][kThreads / kParts];
  sums[part][threadIdx.x % (kThreads / kParts)] = sum;
  __syncthreads();
  if (part == 0 && cw < Cw) {
    A v = 0;
    for (int i = 0; i < kParts; ++i) v += sums[i][threadIdx.x];
    if (row == K * K) { if (db) db[cw] = (T)v; }
    else if (dw) dw[(int64_t)cw * K * K + row] = (T)v;
  }
}

// outputs of one lane: the strip length that leaves fewer unused columns in the last strip of a row
int strip_for(int W) { return ((W + 6) / 7) * 7 < ((W + 7) / 8) * 8 ? 7 : 8; }

// workgroups of the gradient kernel along the strips: over all tap rows and channel blocks three per CU where it works in parts, what
// its registers let run at once, else four, and no more than there are strips (each chunk costs K * (K + 1) * C partial sums)
template <typename T> int grad_chunks(const Conv& a, int K) {
  constexpr int workers = Lane<T>::kWorkers;
  const int s = strip_for(a.W);
  const int64_t nstrips = (int64_t)a.B * a.H * ((a.W + s - 1) / s);
  const int64_t share = (int64_t)K * ((a.C + kBlockChannels - 1) / kBlockChannels);
  const int64_t all = grad_in_parts<T>(K) ? 768 : 1024, want = all / share < 1 ? 1 : all / share;
  const int64_t most = (nstrips + workers - 1) / workers;
  return (int)(want < most ? want : most);
}

template <typename T, int K, int STRIP>
void launch(const Conv& a, bool flip, hipStream_t st) {
  const int per_row = (a.W + STRIP - 1) / STRIP, nstrips = a.B * a.H * per_row;
  const dim3 grid((unsigned)((nstrips + Lane<T>::kWorkers - 1) / Lane<T>::kWorkers),
                  (unsigned)((a.C + kBlockChannels - 1) / kBlockChannels));
  conv_kernel<T, K, STRIP><<<grid, dim3(kThreads), 0, st>>>(a, per_row, nstrips, flip ? 1 : 0);
}
template <typename T, int K, int STRIP>
void launch_grad(const Conv& a, const void* g, int64_t g_batch, int64_t g_row, void* dw, void* db, float* partial,
                 hipStream_t st) {
  const int per_row = (a.W + STRIP - 1) / STRIP, nstrips = a.B * a.H * per_row;
  const int chunks = grad_chunks<T>(a, K);
  const dim3 grid((unsigned)chunks, (unsigned)((a.C + kBlockChannels - 1) / kBlockChannels), (unsigned)K);
  grad_kernel<T, K, STRIP><<<grid, dim3(kThreads), 0, st>>>(a, (const T*)g, g_batch, g_row, partial, per_row, nstrips);
  grad_finish_kernel<T><<<dim3((unsigned)(K * K + 1), (unsigned)cdiv64(a.Cw, kThreads / kFinishParts)), dim3(kThreads), 0, st>>>(
      partial, chunks, K, a.C, a.Cw, (T*)dw, (T*)db);
}

template <typename F> void by_shape(int K, int W, F&& f) {
  using std::integral_constant;
  const bool seven = strip_for(W) == 7;
  auto with = [&](auto k) {
    if (seven) f(k, integral_constant<int, 7>());
    else f(k, integral_constant<int, 8>());
  };
  if (K == 3) with(integral_constant<int, 3>());
  else if (K == 5) with(integral_constant<int, 5>());
  else with(integral_constant<int, 7>());
}
template <typename F> void by_type(int dtype, F&& f) {
  if (dtype == kF16) f(_Float16{});
  else if (dtype == kBF16) f(__bf16{});
  else f(float{});
}

}  // namespace

bool supported(int C, int Cw, int K, int dtype) {
  const int vec = dtype == kF32 ? 4 : 8;
  return (K == 3 || K == 5 || K == 7) && C > 0 && Cw > 0 && C % vec == 0 && C % Cw == 0;
}

size_t grad_workspace_bytes(const Conv& a, int K, int dtype) {
  int64_t chunks = 0;
  by_type(dtype, [&](auto t) { chunks = grad_chunks<decltype(t)>(a, K); });
  return sizeof(float) * (size_t)chunks * K * (K + 1) * a.C;
}

void forward(const Conv& a, int K, int dtype, bool flip, hipStream_t st) {
  by_type(dtype, [&](auto t) {
    by_shape(K, a.W, [&](auto k, auto s) { launch<decltype(t), decltype(k)::value, decltype(s)::value>(a, flip, st); });
  });
}

void grad(const Conv& a, const void* g, int64_t g_batch, int64_t g_row, void* dw, void* db, float* partial, int K,
          int dtype, hipStream_t st) {
  by_type(dtype, [&](auto t) {
    by_shape(K, a.W, [&](auto k, auto s) {
      launch_grad<decltype(t), decltype(k)::value, decltype(s)::value>(a, g, g_batch, g_row, dw, db, partial, st);
    });
  });
}

}  // namespace dwconv
}  // namespace fbla
