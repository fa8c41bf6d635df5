// Projections of token rows on the matrix cores, 16-bit types: out = a W^T (+ bias) (+ add), the forward of the blocks'
// nn.Linear layers, and out = a W + a2 W2 (+ add), their input gradients (layers/linfusion.py:26-38,83-103, mlla.py:56,
// focused_la.py:26-27, polaformer.py:24-25).  Up to three products over the same tokens share a launch.
//
// What bounds it: the blocks' projections have 64 to 1280 channels on either side and 1e2 to 2e5 tokens, a few steps of the
// contraction per tile, so that a tile is mostly its first loads and its stores: HBM for many tokens, latency for few.
// Tile: TM tokens x TN outputs by four waves (2 x 2), steps of 64 channels of the contraction; both operands arrive flat (16
// bytes per lane), two steps ahead in registers, and go through two LDS buffers, one barrier a step.  W is the A operand of
// the matrix instruction, so that a lane owns 16 neighbouring outputs of one token (the rows of W are permuted on the way
// into LDS, or by the transposing read where the contraction runs over W's rows); results leave through LDS as whole rows.
// Sums are fp32 and rounded once, bias, `add` and the second product included.
//
// GPU us in a captured graph, four sets of rows in turn, the library / here (bf16, with bias; in brackets the input gradient): 200704
// x 64 -> 128 28.0 / 25.3 (54.3 / 19.3), 50176 x 256 -> 512 41.1 / 38.5 (25.7 / 31.8), -> 256 15.8 / 20.3 (17.6 / 19.6), 3136 x 256 -> 512
// 6.5 / 5.8 (7.6 / 5.4), 1024 x 640 -> 640 6.3 / 6.3 (7.3 / 5.9), 8192 x 640 -> 640 14.4 / 16.8 (17.6 / 16.3), three of them in one launch
// 42.6 / 37.1.  The blocks keep the library's GEMM where it is the faster one and long
// enough to hide its host time (`projects` in fbla_torch.cpp has the lines and both sides of each): a launch here costs the host 4 us, a GEMM call of
// torch 17, and launches and passes that go into one here pay back what the library is faster at by itself.  A first form with
// branches around its loads waited for every step's rows (and looped over lanes for descriptors the compiler could not see to
// be uniform): 15 % more throughout.  Blocks: LinFusion forward 8192 x 640 243 -> 142 us (with norm_leaky below, residual sums in
// the products), MLLA step 64 x 56x56 x 64 414 -> 371, PolaFormer step 64 x 28x28 x 256 781 -> 750.
#include <hip/hip_runtime.h>


#include "fbla_mfma_shared.h"

namespace fbla {
namespace gemm {

namespace {

constexpr int kThreads = 256;
constexpr int kBufferFlags = 0x00020000;  // raw buffer, 32-bit words, range checked
constexpr int kPast = 1 << 30;             // a lane offset past every buffer
constexpr int kStep = 64;  // channels of the contraction per step: 128 bytes of a row

typedef uint32_t u32x4 __attribute__((ext_vector_type(4)));
typedef uint32_t u32x2 __attribute__((ext_vector_type(2)));
typedef short i16x4 __attribute__((ext_vector_type(4)));
typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
typedef _Float16 f16x8 __attribute__((ext_vector_type(8)));
typedef float f32x8 __attribute__((ext_vector_type(8)));
using mfma::f32x16;

template <typename T> struct Vec;
template <> struct Vec<__bf16> { typedef bf16x8 type; };
template <> struct Vec<_Float16> { typedef f16x8 type; };

__device__ __forceinline__ f32x16 mma(bf16x8 a, bf16x8 b, f32x16 c) { return __builtin_amdgcn_mfma_f32_32x32x16_bf16(a, b, c, 0, 0, 0); }
__device__ __forceinline__ f32x16 mma(f16x8 a, f16x8 b, f32x16 c) { return __builtin_amdgcn_mfma_f32_32x32x16_f16(a, b, c, 0, 0, 0); }

__device__ __forceinline__ u32x2 transposed_read(const unsigned char* at) {
  typedef i16x4 __attribute__((address_space(3))) * lds_ptr;
  return __builtin_bit_cast(u32x2, __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_ptr)(at)));
}

struct Jobs {
  Job job[kMostJobs];
  int first_tile[kMostJobs + 1];  // in units of output tiles, over all jobs
  int count;
  int64_t tokens;
};

// Place of 16-byte piece `ch` of row `row` in a tile of the contraction's rows (TN outputs wide): four consecutive rows and the
// pieces c, c + 2 that one transposing read touches fall into different banks.
template <int TN> __device__ __forceinline__ int place_rows(int row, int ch) {
  if constexpr (TN == 128) return row * 256 + ((ch ^ ((row & 1) | ((row & 2) << 1))) << 4);
  else return row * 128 + ((ch ^ ((row & 2) << 1)) << 4);
}

template <typename T, int TM, int TN, bool ROWS, bool TWO>
__global__ __launch_bounds__(kThreads, 2) void project_kernel(Jobs jobs) {
  using V = typename Vec<T>::type;
  constexpr int kABytes = TM * kStep * 2, kWBytes = TN * kStep * 2, kBuf = kABytes + kWBytes;
  constexpr int kAPieces = kABytes / 16 / kThreads, kWPieces = kWBytes / 16 / kThreads;  // per thread and step
  constexpr int MB = TM / 64, NB = TN / 64;                                              // 32 x 32 blocks of a wave
  constexpr int kOutRow = TN * 2 + 16;  // (16 bytes apart from a multiple of the banks)
  __shared__ __attribute__((aligned(16))) unsigned char smem[2 * kBuf > TM * kOutRow ? 2 * kBuf : TM * kOutRow];

  const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int wm = wave >> 1, wn = wave & 1, kb = lane >> 5;

  struct Source {
    const T *a, *w;
    int a_row, w_row, K, a_bytes, w_bytes;  // bytes to the end of the tile's last row, and of W's last row
  };
  // The output tiles of a block of tokens read the same rows: they run on one XCD (workgroup i is on XCD i % 8).  Blocks beyond
  // the last multiple of eight keep the plain order.  (One round of workgroups that walk the tiles, the next one's first rows
  // requested before the results leave, was slower throughout: 50176 x 256 -> 2 x 512 57.4 us against 48.8, spilling at two
  // workgroups a CU.)
  const int tiles = jobs.first_tile[jobs.count], blocks = (int)((jobs.tokens + TM - 1) / TM), i = blockIdx.x;
  const int together = blocks / 8 * 8 * tiles;
  const int block = i < together ? i / (8 * tiles) * 8 + i % 8 : i / tiles;
  const int tile = i < together ? i / 8 % tiles : i % tiles;
  int j = 0;
  if (jobs.count > 1 && tile >= jobs.first_tile[1]) j = 1;
  if (jobs.count > 2 && tile >= jobs.first_tile[2]) j = 2;
  const Job& job = jobs.job[j];
  const int n0 = (tile - jobs.first_tile[j]) * TN, N = job.N;
  const int64_t t0 = (int64_t)block * TM;
  const int rows = (int)min((int64_t)TM, jobs.tokens - t0);
  const int steps0 = (job.K[0] + kStep - 1) / kStep, steps = steps0 + (TWO ? (job.K[1] + kStep - 1) / kStep : 0);
  auto source = [&](int seg) {
    Source r;
    r.K = job.K[seg];
    r.a_row = (int)job.a_row[seg] * 2;
    r.w_row = (ROWS ? N : r.K) * 2;
    r.a = (const T*)job.a[seg] + t0 * job.a_row[seg];
    r.w = (const T*)job.w[seg] + (ROWS ? (int64_t)n0 : (int64_t)n0 * r.K);
    r.a_bytes = (rows - 1) * r.a_row + r.K * 2;
    r.w_bytes = ROWS ? (r.K * N - n0) * 2 : min(TN, N - n0) * r.w_row;
    return r;
  };
  // (a job of one product next to others of two: what its last loads ask for beyond its steps is the first product's again)
  const Source first = source(0), other = source(TWO && job.K[1] ? 1 : 0);
  // The steps of both products, one after the other.  Loads are buffer loads without a branch around them (so that a wait for one
  // step's rows leaves the next step's in flight).  Each step's buffers begin at its first channels (or W's first row) and end with
  // the rows, so that it is the lanes' own offsets that meet the end: a scalar offset past a buffer's bytes is not sure to be seen
  // by the bounds check.  What lies past the last token, past W's last row, past the rows' channels or past the last step comes back
  // as zero.
  struct Regs {
    u32x4 a[kAPieces], w[kWPieces];
  };
  auto fetch = [&](Regs& r, int s) {
    const bool second = TWO && s >= steps0;
    const Source from = second ? other : first;
    const int k0 = (second ? s - steps0 : s) * kStep;
    const __amdgpu_buffer_rsrc_t a = __builtin_amdgcn_make_buffer_rsrc((void*)(from.a + k0), 0, max(from.a_bytes - k0 * 2, 0), kBufferFlags);
    const __amdgpu_buffer_rsrc_t w = __builtin_amdgcn_make_buffer_rsrc((void*)(from.w + (ROWS ? (int64_t)k0 * N : k0)), 0,
                                                                       max(from.w_bytes - (ROWS ? k0 * from.w_row : k0 * 2), 0), kBufferFlags);
    const int past = k0 + (tid & 7) * 8 >= from.K ? kPast : 0;
#pragma unroll
    for (int p = 0; p < kAPieces; ++p) {
      const int q = tid + kThreads * p;
      r.a[p] = __builtin_amdgcn_raw_buffer_load_b128(a, ((q >> 3) * from.a_row + (q & 7) * 16) | past, 0, 0);
    }
#pragma unroll
    for (int p = 0; p < kWPieces; ++p) {
      const int q = tid + kThreads * p;
      if constexpr (ROWS) r.w[p] = __builtin_amdgcn_raw_buffer_load_b128(w, q / (TN / 8) * from.w_row + q % (TN / 8) * 16, 0, 0);
      else r.w[p] = __builtin_amdgcn_raw_buffer_load_b128(w, ((q >> 3) * from.w_row + (q & 7) * 16) | past, 0, 0);
    }
  };
  auto stash = [&](const Regs& r, unsigned char* at) {
    unsigned char* wt = at + kABytes;
#pragma unroll
    for (int p = 0; p < kAPieces; ++p) {
      const int q = tid + kThreads * p;
      *reinterpret_cast<u32x4*>(at + mfma::swz<128>(q >> 3, q & 7)) = r.a[p];
    }
#pragma unroll
    for (int p = 0; p < kWPieces; ++p) {
      const int q = tid + kThreads * p;
      if constexpr (ROWS) {
        *reinterpret_cast<u32x4*>(wt + place_rows<TN>(q / (TN / 8), q % (TN / 8))) = r.w[p];
      } else {
        // output 16 b + 4 g + j of 32 goes to row 8 g + 4 b + j
        const int n = q >> 3, row = (n & ~31) | ((n & 12) << 1) | ((n & 16) >> 2) | (n & 3);
        *reinterpret_cast<u32x4*>(wt + mfma::swz<128>(row, q & 7)) = r.w[p];
      }
    }
  };
  int woff[NB][2];  // ROWS: this lane's two transposing reads
  if constexpr (ROWS) {
    const int g = lane >> 4, s = lane & 15, q = s & 3;
#pragma unroll
    for (int b = 0; b < NB; ++b)
#pragma unroll
      for (int h = 0; h < 2; ++h)
        woff[b][h] = place_rows<TN>(8 * (g >> 1) + 4 * h + (s >> 2), 4 * (wn * NB + b) + 2 * (q & 1) + (g & 1)) + 8 * (q >> 1);
  }
  f32x16 acc[MB][NB];
  struct Fragments {
    V x[MB], w[NB];
  };
  auto fragments = [&](Fragments& f, const unsigned char* at, int ks) {
    const unsigned char* wt = at + kABytes;
#pragma unroll
    for (int b = 0; b < NB; ++b) {
      if constexpr (ROWS) {  // (16 rows further on the swizzle is the same)
        const u32x2 lo = transposed_read(wt + ks * 16 * TN * 2 + woff[b][0]), hi = transposed_read(wt + ks * 16 * TN * 2 + woff[b][1]);
        f.w[b] = __builtin_bit_cast(V, u32x4{lo[0], lo[1], hi[0], hi[1]});
      } else {
        f.w[b] = __builtin_bit_cast(V, *reinterpret_cast<const u32x4*>(wt + mfma::swz<128>(32 * (wn * NB + b) + (lane & 31), 2 * ks + kb)));
      }
    }
#pragma unroll
    for (int a = 0; a < MB; ++a)
      f.x[a] = __builtin_bit_cast(V, *reinterpret_cast<const u32x4*>(at + mfma::swz<128>(32 * (wm * MB + a) + (lane & 31), 2 * ks + kb)));
  };
  auto multiply = [&](const unsigned char* at) {  // the next fragments are requested before the products of the ones at hand
    Fragments f[2];
    fragments(f[0], at, 0);
#pragma unroll
    for (int ks = 0; ks < kStep / 16; ++ks) {
      if (ks + 1 < kStep / 16) fragments(f[(ks + 1) & 1], at, ks + 1);
#pragma unroll
      for (int a = 0; a < MB; ++a)
#pragma unroll
        for (int b = 0; b < NB; ++b) acc[a][b] = mma(f[ks & 1].w[b], f[ks & 1].x[a], acc[a][b]);
      __builtin_amdgcn_sched_barrier(0);
    }
  };

  Regs r0, r1;
  fetch(r0, 0);
  fetch(r1, 1);
  V bias[NB][2];  // this lane's outputs'
#pragma unroll
  for (int b = 0; b < NB; ++b)
#pragma unroll
    for (int h = 0; h < 2; ++h) {
      const int n = n0 + 32 * (wn * NB + b) + 16 * kb + 8 * h;
      bias[b][h] = job.bias ? *reinterpret_cast<const V*>((const T*)job.bias + (n < N ? n : 0)) : V{};
    }
#pragma unroll
  for (int a = 0; a < MB; ++a)
#pragma unroll
    for (int b = 0; b < NB; ++b)
#pragma unroll
      for (int r = 0; r < 16; ++r) acc[a][b][r] = 0.f;
  // step s is in LDS buffer s % 2 while s + 1 and s + 2 are in registers or on their way there
  for (int s = 0; s + 1 < steps; s += 2) {
    stash(r0, smem);
    fetch(r0, s + 2);
    __syncthreads();  // (every wave is done with the step before, whose buffer is written next)
    multiply(smem);
    stash(r1, smem + kBuf);
    fetch(r1, s + 3);
    __syncthreads();
    multiply(smem + kBuf);
  }
  if (steps & 1) {
    stash(r0, smem);
    __syncthreads();
    multiply(smem);
  }

  // ---- out: a lane's 16 neighbouring outputs of a token, rounded, to LDS; whole rows from there
  __syncthreads();
#pragma unroll
  for (int a = 0; a < MB; ++a) {
    const int row = 32 * (wm * MB + a) + (lane & 31);
#pragma unroll
    for (int b = 0; b < NB; ++b) {
      const int col = 32 * (wn * NB + b) + 16 * kb;
#pragma unroll
      for (int h = 0; h < 2; ++h) {
        const int n = n0 + col + 8 * h;
        f32x8 v;
#pragma unroll
        for (int e = 0; e < 8; ++e) v[e] = acc[a][b][8 * h + e];
        v += __builtin_convertvector(bias[b][h], f32x8);
        if (job.add) {
          const bool has = n < N && row < rows;
          const V x = *reinterpret_cast<const V*>((const T*)job.add + (has ? (t0 + row) * job.add_row + n : 0));
          v += __builtin_convertvector(x, f32x8);
        }
        *reinterpret_cast<V*>(smem + row * kOutRow + (col + 8 * h) * 2) = __builtin_convertvector(v, V);
      }
    }
  }
  __syncthreads();
  constexpr int kRowPieces = TN / 8;
#pragma unroll
  for (int p = 0; p < TM * kRowPieces / kThreads; ++p) {
    const int q = tid + kThreads * p, row = q / kRowPieces, ch = q % kRowPieces;
    if (row < rows && n0 + 8 * ch < N)
      *reinterpret_cast<u32x4*>((T*)job.out + (t0 + row) * job.out_row + n0 + 8 * ch) =
          *reinterpret_cast<const u32x4*>(smem + row * kOutRow + ch * 16);
  }
}

template <typename T, int TM, int TN, bool ROWS>
void launch(const Job* job, int count, int64_t tokens, hipStream_t st) {
  Jobs jobs{};
  jobs.count = count;
  jobs.tokens = tokens;
  bool two = false;
  for (int j = 0; j < count; ++j) {
    jobs.job[j] = job[j];
    jobs.first_tile[j + 1] = jobs.first_tile[j] + (job[j].N + TN - 1) / TN;
    two = two || job[j].K[1] > 0;
  }
  const dim3 grid((unsigned)(cdiv64(tokens, TM) * jobs.first_tile[count])), block(kThreads);
  if (two) project_kernel<T, TM, TN, ROWS, true><<<grid, block, 0, st>>>(jobs);
  else project_kernel<T, TM, TN, ROWS, false><<<grid, block, 0, st>>>(jobs);
}

// By the number of 128 x 128 tiles: too few for the CUs are cut to 64 x 64; large tiles need enough of them and of steps to
// outweigh three workgroups a CU of 128 x 64.  us with 64 x 64 / 128 x 64 / 128 x 128, forward (bf16): 392 x 64 -> 128 3.8 / 4.6 / 4.6, 1024 x
// 640 -> 3 x 640 (120 tiles) 8.5 / 8.6 / 11.3, 1024 x 1280 -> 3 x 1280 (240) 26.6 / 20.7 / 20.7, 8192 x 640 -> 640 (320) 14.6 / 14.5 / 16.3,
// -> 3 x 640 (960) 36.4 / 32.9 / 30.3, 50176 x 256 -> 256 (784) 17.2 / 16.8 / 17.5, -> 2 x 512 (3136) 61 / 51.8 / 48.8, 200704 x 64 -> 128
// (1568) 18.9 / 16.9 / 17.6.
template <typename T, bool ROWS> void choose(const Job* job, int count, int64_t tokens, hipStream_t st) {
  int64_t wide = 0;
  int least_k = 1 << 30;
  for (int j = 0; j < count; ++j) {
    wide += (job[j].N + 127) / 128;
    least_k = job[j].K[0] < least_k ? job[j].K[0] : least_k;
  }
  const int64_t tiles = cdiv64(tokens, 128) * wide;
  if (tiles < 200) launch<T, 64, 64, ROWS>(job, count, tokens, st);
  else if (tiles < 900 || least_k < 256) launch<T, 128, 64, ROWS>(job, count, tokens, st);
  else launch<T, 128, 128, ROWS>(job, count, tokens, st);
}

// LayerNorm over the channels of a row and LeakyReLU (layers/linfusion.py:26-38), both paths of the block in one launch: a wave
// holds a row (C channels of 16-byte pieces, PER a lane), mean and variance from the registers, fp32 throughout and rounded
// once.  mean and rstd (fp32, or null) are what torch's LayerNorm saves.  2 x 8192 x 640 fp16, 42 MB:
// 12.4 us (3.4 TB/s); torch's norms and activations took 41.
template <typename T, int PER>
__global__ __launch_bounds__(kThreads) void norm_leaky_kernel(NormJob j0, NormJob j1, int64_t tokens, int C, int wgs) {
  using V = typename Vec<T>::type;
  const bool second = (int)blockIdx.x >= wgs;
  const NormJob& j = second ? j1 : j0;
  const int lane = threadIdx.x & 63;
  const int64_t t = (int64_t)(second ? blockIdx.x - wgs : blockIdx.x) * (kThreads / 64) + (threadIdx.x >> 6);
  if (t >= tokens) return;
  const int pieces = C / 8;
  const T* x = (const T*)j.x + t * C;
  f32x8 v[PER];
#pragma unroll
  for (int i = 0; i < PER; ++i) {
    const int ch = lane + 64 * i;
    const V e = *reinterpret_cast<const V*>(x + (ch < pieces ? 8 * ch : 0));
    v[i] = __builtin_convertvector(e, f32x8);
  }
  auto sum_of = [&](auto term) {
    float sum = 0.f;
#pragma unroll
    for (int i = 0; i < PER; ++i)
#pragma unroll
      for (int e = 0; e < 8; ++e) sum += lane + 64 * i < pieces ? term(v[i][e]) : 0.f;
#pragma unroll
    for (int m = 1; m < 64; m *= 2) sum += __shfl_xor(sum, m);
    return sum;
  };
  const float mean = sum_of([](float a) { return a; }) / (float)C;
  const float var = sum_of([&](float a) { return (a - mean) * (a - mean); }) / (float)C;
  const float rstd = 1.f / sqrtf(var + j.eps);
#pragma unroll
  for (int i = 0; i < PER; ++i) {
    const int ch = lane + 64 * i;
    if (ch >= pieces) continue;
    f32x8 y;
#pragma unroll
    for (int e = 0; e < 8; ++e) y[e] = (v[i][e] - mean) * rstd;
    if (j.weight) y *= __builtin_convertvector(*reinterpret_cast<const V*>((const T*)j.weight + 8 * ch), f32x8);
    if (j.bias) y += __builtin_convertvector(*reinterpret_cast<const V*>((const T*)j.bias + 8 * ch), f32x8);
#pragma unroll
    for (int e = 0; e < 8; ++e) y[e] = y[e] > 0.f ? y[e] : y[e] * j.slope;
    *reinterpret_cast<V*>((T*)j.out + t * C + 8 * ch) = __builtin_convertvector(y, V);
  }
  if (lane == 0 && j.mean) {
    j.mean[t] = mean;
    j.rstd[t] = rstd;
  }
}

template <typename T> void launch_norm(const NormJob* jobs, int count, int64_t tokens, int C, hipStream_t st) {
  const int wgs = (int)cdiv64(tokens, kThreads / 64);
  const dim3 grid((unsigned)(wgs * count)), block(kThreads);
  const NormJob &a = jobs[0], &b = jobs[count - 1];
  if (C <= 512) norm_leaky_kernel<T, 1><<<grid, block, 0, st>>>(a, b, tokens, C, wgs);
  else if (C <= 1024) norm_leaky_kernel<T, 2><<<grid, block, 0, st>>>(a, b, tokens, C, wgs);
  else norm_leaky_kernel<T, 4><<<grid, block, 0, st>>>(a, b, tokens, C, wgs);
}

}  // namespace

void norm_leaky(const NormJob* jobs, int count, int64_t tokens, int C, int dtype, hipStream_t st) {
  if (dtype == kF16) launch_norm<_Float16>(jobs, count, tokens, C, st);
  else launch_norm<__bf16>(jobs, count, tokens, C, st);
}

void project(const Job* jobs, int count, int64_t tokens, bool rows_of_w, int dtype, hipStream_t st) {
  if (dtype == kF16) {
    if (rows_of_w) choose<_Float16, true>(jobs, count, tokens, st);
    else choose<_Float16, false>(jobs, count, tokens, st);
  } else {
    if (rows_of_w) choose<__bf16, true>(jobs, count, tokens, st);
    else choose<__bf16, false>(jobs, count, tokens, st);
  }
}

}  // namespace gemm
}  // namespace fbla
