/*
 * flash_bla_hip.h -- C ABI of libfbla_hip.so: bidirectional (non-causal) linear
 * attention for AMD gfx950 (MI355X).
 *
 * The reference (fla-org/flash-bidirectional-linear-attention, `flash_bla`) has
 * no native layer: its operators are torch.autograd.Function classes that launch
 * Triton kernels.  Each entry point below replaces the kernel launches made by
 * one of those Functions; the Python operator layer keeps the reference's
 * signatures and binds these symbols with ctypes.
 *
 * Conventions
 *   - every pointer is a DEVICE pointer unless stated otherwise; the library
 *     never allocates, frees or retains device memory: outputs and the workspace
 *     are provided by the caller (size from the *_workspace_bytes queries);
 *   - work is enqueued on `stream` (a hipStream_t passed as void*); no call
 *     synchronises the device;
 *   - return value 0 = success, negative = error (fbla_last_error() gives the
 *     text for the calling thread); no C++ exception crosses the boundary;
 *   - dense tensors are contiguous [B,H,L,D]; packed tensors are contiguous
 *     [T_total,H,D] with int32 cu_seqlens[N+1] on the device;
 *   - the state tensors s [B*H,DK,DV] (or [N*H,DK,DV]) and km [..,DK] are fp32.
 *     s already includes `scale`; km is the mean key.  Forward writes them,
 *     backward reads them (the reference saves the same two tensors in its
 *     autograd context: linear_attn/fused.py:395);
 *   - reductions over tokens are two-stage and fixed-order: results are
 *     bit-identical from run to run.
 */
#ifndef FLASH_BLA_HIP_H
#define FLASH_BLA_HIP_H

#include <stddef.h>
#include <stdint.h>

#ifdef __cplusplus
extern "C" {
#endif

/* element type of q/k/v/o and of the gradients */
#define FBLA_F16 0
#define FBLA_BF16 1
#define FBLA_F32 2

/* flags */
#define FBLA_NORMALIZE 1     /* o = (q S)/(q.km + eps); clear = simple_la (no denominator) */
#define FBLA_DECOUPLED 2     /* numerator from q_rope/k_rope, denominator from q/k */
#define FBLA_DEFAULT_SCALE 4 /* packed layout only: scale = 1/len_i per sequence */
#define FBLA_ELU1_QK 8       /* q and k are given BEFORE the callers' feature map
                              * phi(x) = elu(x) + 1 (layers/linfusion.py:88-89, layers/mlla.py:74-75) and the
                              * kernels apply it as they load them; fp16 / bf16, DK = DV = 64, not decoupled
                              * (FBLA_ERR_UNSUPPORTED otherwise); the backward entry points take it together
                              * with FBLA_ELU1_GRAD only */
#define FBLA_ELU1_GRAD 16    /* backward entry points only: q and k are the MAPPED tensors phi(x) = elu(x) + 1 (what
                              * the forward consumed and saved) and dq, dk are wanted with respect to x: the
                              * kernels multiply them by phi'(x) = min(phi(x), 1) as they write them, which
                              * replaces the autograd of `F.elu(x) + 1.0` (two elementwise launches per call).
                              * Together with FBLA_ELU1_QK, q and k are given before the map here as well and the
                              * backward kernels map them on load (no mapped copies exist anywhere).
                              * fp16 / bf16, DK = DV = 64, not decoupled (FBLA_ERR_UNSUPPORTED otherwise) */

/* error codes */
#define FBLA_OK 0
#define FBLA_ERR_BAD_ARG (-1)
#define FBLA_ERR_UNSUPPORTED (-2)
#define FBLA_ERR_WORKSPACE (-3)
#define FBLA_ERR_LAUNCH (-4)

/* Library version (major*10000 + minor*100 + patch). */
int fbla_version(void);

/* Profiling aid with no counterpart in the reference: restrict the entry points
 * called from this thread to a subset of their kernels so that one kernel can be
 * timed in isolation (bit 0 forward partial state, 1 forward state reduce,
 * 2 forward output, 3 backward pass A, 4 backward reduce, 5 backward pass B).
 * 0 restores the default (all kernels).  Skipped kernels leave their outputs
 * untouched, so results are only meaningful with the default mask.  Ignored unless
 * the process was started with FBLA_ALLOW_PHASE_MASK=1 in its environment. */
void fbla_set_phase_mask(unsigned mask);

/* Message of the last error raised on the calling thread ("" if none). */
const char* fbla_last_error(void);

/* Workspace (bytes) needed by fbla_la_fwd (pass=0) / fbla_la_bwd (pass=1) for a
 * dense problem.  Replaces the torch.empty temporaries of
 * linear_attn/fused.py:362-363,422-423 (which grow with L/32; ours do not). */
size_t fbla_la_workspace_bytes(int pass, int64_t B, int64_t H, int64_t L, int DK, int DV,
                               int dtype, int flags);

/* Dense forward.  Replaces the launches in
 *   LinearAttnFunction.forward        flash_bla/ops/linear_attn/fused.py:352-398
 *   SimpleLinearAttnFunction.forward  flash_bla/ops/simple_la/fused.py:495-535   (flags without FBLA_NORMALIZE)
 *   DecoupledLAFunction.forward       flash_bla/ops/linear_attn/decoupled.py:413-460 (FBLA_DECOUPLED)
 * q,k,(q_rope,k_rope): [B,H,L,DK]; v,o: [B,H,L,DV]; q_rope/k_rope NULL unless decoupled. */
int fbla_la_fwd(const void* q, const void* k, const void* v, const void* q_rope,
                const void* k_rope, void* o, float* s, float* km, void* workspace,
                size_t workspace_bytes, int64_t B, int64_t H, int64_t L, int DK, int DV, int dtype,
                int flags, float scale, float eps, void* stream);

/* Dense backward.  Replaces the launches in
 *   LinearAttnFunction.backward        flash_bla/ops/linear_attn/fused.py:400-453
 *   SimpleLinearAttnFunction.backward  flash_bla/ops/simple_la/fused.py:537-626
 *   DecoupledLAFunction.backward       flash_bla/ops/linear_attn/decoupled.py:462-509
 * `o` is not an input: o.dO is recomputed from q and s.  dq_rope/dk_rope are
 * written only when decoupled (then dq/dk receive the denominator gradients). */
int fbla_la_bwd(const void* q, const void* k, const void* v, const void* q_rope,
                const void* k_rope, const void* dout, const float* s, const float* km, void* dq,
                void* dk, void* dv, void* dq_rope, void* dk_rope, void* workspace,
                size_t workspace_bytes, int64_t B, int64_t H, int64_t L, int DK, int DV, int dtype,
                int flags, float scale, float eps, void* stream);

/* Dense forward that allocates nothing.  No counterpart in the reference: it is for callers
 * that cannot allocate device memory (code under HIP graph capture, tight serving loops,
 * harnesses that forbid hipMalloc) and have no workspace to hand over.  Same arguments,
 * arithmetic and results as fbla_la_fwd, but the workspace is a fixed array of
 * FBLA_STATIC_SCRATCH_BYTES inside the library's device image (each GPU the library runs on
 * holds one copy until the process ends).  A problem whose fbla_la_workspace_bytes(0, ...)
 * exceeds that returns FBLA_ERR_WORKSPACE.  The call makes no hipMalloc / hipFree and no
 * allocating library call.  All calls on one GPU share the array: calls that overlap on one
 * GPU (two streams, two threads) race; serialise them or use fbla_la_fwd.  The first call on a
 * device looks up the array's address (hipGetSymbolAddress, which may load the code object) and
 * sets the kernels' LDS attributes: make one eager call per device and problem shape before
 * recording calls into a HIP graph. */
#define FBLA_STATIC_SCRATCH_BYTES (16u << 20)
size_t fbla_static_scratch_bytes(void);
int fbla_la_fwd_static(const void* q, const void* k, const void* v, const void* q_rope,
                       const void* k_rope, void* o, float* s, float* km, int64_t B, int64_t H,
                       int64_t L, int DK, int DV, int dtype, int flags, float scale, float eps,
                       void* stream);

/* Two queries on shared keys and values, dense, with the denominator.  Replaces the two operator
 * calls of PolaLinearAttention.forward (flash_bla/layers/polaformer.py:89-90:
 *   x_sim = linear_attention(q_sim, k, v1),  x_opp = linear_attention(q_opp, k, v2)
 * with v1 | v2 the two halves of the value channels), which read k twice forward and twice
 * backward and leave the sum of the two dk to autograd.  Here
 *   S = scale * K^T [v1 | v2]  (one pass over k and v),  km = mean k,
 *   o1 = (q1 S[:, :DV/2]) / (q1 . km + eps),  o2 = (q2 S[:, DV/2:]) / (q2 . km + eps),
 * and the backward reads k and v once and writes dk = dk1 + dk2 once.
 * q1, q2, dq1, dq2, k, dk: [B,H,L,DK]; v, dv: [B,H,L,DV]; o1, o2, dout1, dout2: [B,H,L,DV/2];
 * s: [B,H,DK,DV], km: [B,H,DK] fp32.  fp16 / bf16, DK and DV/2 multiples of 8 up to 128 (the
 * workspace query returns 0 for anything else, the calls FBLA_ERR_UNSUPPORTED). */
size_t fbla_la_pair_workspace_bytes(int pass, int64_t B, int64_t H, int64_t L, int DK, int DV, int dtype);
int fbla_la_pair_fwd(const void* q1, const void* q2, const void* k, const void* v, void* o1, void* o2,
                     float* s, float* km, void* workspace, size_t workspace_bytes, int64_t B, int64_t H,
                     int64_t L, int DK, int DV, int dtype, float scale, float eps, void* stream);
int fbla_la_pair_bwd(const void* q1, const void* q2, const void* k, const void* v, const void* dout1,
                     const void* dout2, const float* s, const float* km, void* dq1, void* dq2, void* dk,
                     void* dv, void* workspace, size_t workspace_bytes, int64_t B, int64_t H, int64_t L,
                     int DK, int DV, int dtype, float scale, float eps, void* stream);

/* Dense problems with Lk key / value tokens and Lq query tokens per (batch, head), Lk != Lq:
 * q, dq: [B,H,Lq,DK]; k, dk: [B,H,Lk,DK]; v, dv: [B,H,Lk,DV]; o, dout: [B,H,Lq,DV]; km is the mean
 * over the Lk keys.  The reference has no counterpart: its dense kernels take one length from q
 * (linear_attn/fused.py:355) and read k, v out of bounds when the PVT-style blocks
 * (layers/focused_la.py:55,73-75, layers/polaformer.py) shorten the keys with sr_ratio > 1.
 * Flags as for fbla_la_fwd without FBLA_DECOUPLED (the decoupled operator has the pair of entry
 * points below); every dtype and head dim of fbla_la_fwd.  fbla_la_cross_workspace_bytes takes
 * FBLA_DECOUPLED in `flags` for the decoupled pair. */
size_t fbla_la_cross_workspace_bytes(int pass, int64_t B, int64_t H, int64_t Lq, int64_t Lk, int DK,
                                     int DV, int dtype, int flags);
int fbla_la_cross_fwd(const void* q, const void* k, const void* v, void* o, float* s, float* km,
                      void* workspace, size_t workspace_bytes, int64_t B, int64_t H, int64_t Lq,
                      int64_t Lk, int DK, int DV, int dtype, int flags, float scale, float eps,
                      void* stream);
int fbla_la_cross_bwd(const void* q, const void* k, const void* v, const void* dout, const float* s,
                      const float* km, void* dq, void* dk, void* dv, void* workspace,
                      size_t workspace_bytes, int64_t B, int64_t H, int64_t Lq, int64_t Lk, int DK,
                      int DV, int dtype, int flags, float scale, float eps, void* stream);

/* The decoupled operator with Lk != Lq: q, q_rope, dq, dq_rope: [B,H,Lq,DK]; k, k_rope, dk, dk_rope:
 * [B,H,Lk,DK]; v, dv: [B,H,Lk,DV]; o, dout: [B,H,Lq,DV].  No counterpart in the reference
 * (linear_attn/decoupled.py:413-509 takes one length from q).  Workspace: fbla_la_cross_workspace_bytes
 * with flags = FBLA_NORMALIZE | FBLA_DECOUPLED. */
int fbla_decoupled_cross_fwd(const void* q, const void* k, const void* q_rope, const void* k_rope,
                             const void* v, void* o, float* s, float* km, void* workspace,
                             size_t workspace_bytes, int64_t B, int64_t H, int64_t Lq, int64_t Lk, int DK,
                             int DV, int dtype, float scale, float eps, void* stream);
int fbla_decoupled_cross_bwd(const void* q, const void* k, const void* q_rope, const void* k_rope,
                             const void* v, const void* dout, const float* s, const float* km, void* dq,
                             void* dk, void* dq_rope, void* dk_rope, void* dv, void* workspace,
                             size_t workspace_bytes, int64_t B, int64_t H, int64_t Lq, int64_t Lk, int DK,
                             int DV, int dtype, float scale, float eps, void* stream);

/* Workspace for the packed (variable-length) entry points. */
size_t fbla_varlen_workspace_bytes(int pass, int64_t total_tokens, int64_t N, int64_t H,
                                   int64_t max_seqlen, int DK, int DV, int dtype, int flags);

/* Packed forward.  Replaces VarlenLinearAttnFunction.forward
 * (flash_bla/ops/linear_attn/varlen.py:339-422).  max_seqlen is an upper bound on
 * the sequence lengths and only sizes the launch; any value >= the true maximum
 * gives the same result (tests/ops/test_varlen_linear_attn.py:45-55).  With
 * FBLA_DEFAULT_SCALE each sequence uses 1/len_i (varlen.py:66) and `scale` is ignored.
 * s: [N*H,DK,DV], km: [N*H,DK] fp32. */
int fbla_varlen_fwd(const void* q, const void* k, const void* v, const int32_t* cu_seqlens,
                    void* o, float* s, float* km, void* workspace, size_t workspace_bytes,
                    int64_t total_tokens, int64_t N, int64_t H, int64_t max_seqlen, int DK, int DV,
                    int dtype, int flags, float scale, float eps, void* stream);

/* Packed backward.  Replaces VarlenLinearAttnFunction.backward (varlen.py:426-505). */
int fbla_varlen_bwd(const void* q, const void* k, const void* v, const int32_t* cu_seqlens,
                    const void* dout, const float* s, const float* km, void* dq, void* dk, void* dv,
                    void* workspace, size_t workspace_bytes, int64_t total_tokens, int64_t N,
                    int64_t H, int64_t max_seqlen, int DK, int DV, int dtype, int flags,
                    float scale, float eps, void* stream);

/* ---- piecewise (PISA) attention, forward only --------------------------------
 * Tensors are contiguous [BH, T, K] / [BH, T, V] (batch and heads flattened). */

/* Workspace of fbla_chunk_reduce (with_norm != 0 when h_norm is requested). */
size_t fbla_chunk_reduce_workspace_bytes(int64_t BH, int64_t T, int K, int V, int chunk, int dtype,
                                         int with_norm);

/* Block statistics of the linear branch.  Replaces fused_chunk_reduce /
 * fused_chunk_reduce_kernel (flash_bla/ops/piecewise_attn/kernel.py:89-128,152-176).
 * With NT = ceil(T/chunk): qc, kc [BH,NT,K] = chunk means of q, k; vc [BH,NT,V] = chunk
 * sums of v; h [BH,K,V] = sum_c (K_c - kc_c)^T V_c; h_norm [BH,NT] (optional, may be
 * NULL) = p-norm of each chunk's (K_c - kc_c)^T V_c (kernel.py:172-174).  All outputs
 * are fp32 (the reference stores them in the input dtype). */
int fbla_chunk_reduce(const void* q, const void* k, const void* v, float* qc, float* kc, float* vc,
                      float* h, float* h_norm, void* workspace, size_t workspace_bytes, int64_t BH,
                      int64_t T, int K, int V, int chunk, float p_norm, int dtype, void* stream);

/* Block selection.  Replaces the score matrix and torch.topk of the wrapper
 * (flash_bla/ops/piecewise_attn/kernel.py:304-318): for every query block the NS key blocks
 * with the largest qc . kc * scale (+ log(bias + 1e-5) when bias [BH,NT], the h_norm output
 * of fbla_chunk_reduce, is given; kernel.py:314-315 applies a softmax on top, which does not
 * change the order).  qc, kc: fp32 [BH,NT,K] from fbla_chunk_reduce; indices: int32
 * [BH,NT,NS], written in ascending block order (torch.topk orders by score; the attention
 * result does not depend on the order); ties at the threshold go to the lower block index.
 * K in [1,128]; the scores of 16 query blocks against all NT key blocks must fit LDS
 * (NT up to about 2000). */
int fbla_select_blocks(const float* qc, const float* kc, const float* bias, int32_t* indices,
                       int64_t BH, int64_t NT, int K, int NS, float scale, void* stream);

/* Workspace of fbla_piecewise_fwd; 0 when the shape is not supported (a head dim above 128, or so
 * many blocks that their selection flags do not fit LDS). */
size_t fbla_piecewise_workspace_bytes(int64_t BH, int64_t T, int K, int V, int block, int dtype);

/* Piecewise attention forward.  Replaces piecewise_sparse_attention_fwd_kernel
 * (kernel.py:189-292): exact softmax attention over the NS selected key blocks of every
 * query block of `block` tokens (indices: int32 [BH, NT, NS], NT = ceil(T / block)), the
 * remaining blocks through their mean key / value sum (zeroth order) and h (first order).
 * kc, vc, h are the fp32 outputs of fbla_chunk_reduce with chunk = block.  fp16 / bf16 with
 * block = 16, 32 or a multiple of 64 run on the MFMA kernel (K, V other than 64 / 128 through
 * zero-widened copies in the workspace); other block sizes and fp32 inputs run on a shape-generic
 * fp32 kernel (same results to rounding, one to two orders of magnitude slower, no workspace
 * used).  The reference takes the same domain through BK = min(128, next_pow2(K))
 * (kernel.py:296-308). */
int fbla_piecewise_fwd(const void* q, const void* k, const void* v, const float* kc, const float* vc,
                       const float* h, const int32_t* indices, void* o, void* workspace,
                       size_t workspace_bytes, int64_t BH, int64_t T, int K, int V, int block, int NS,
                       float scale, int dtype, void* stream);

/* The feature map of the reference's blocks, phi(x) = elu(x) + 1, for the queries and the
 * keys in one launch.  Replaces the two elementwise torch kernels per tensor of
 * flash_bla/layers/linfusion.py:88-89, mlla.py:74-75 and rala.py:52-53 (`F.elu(x) + 1.0`), with
 * torch's rounding (elu in fp32 rounded to the element type, then + 1 rounded again).
 * x0/y0 hold n0 elements, x1/y1 n1 (either count may be 0); y may alias x.  Any dtype of the
 * FBLA_* element types; pointers 16-byte aligned. */
int fbla_elu1_fwd(const void* x0, void* y0, int64_t n0, const void* x1, void* y1, int64_t n1, int dtype,
                  void* stream);

/* Its derivative: dx = dy * (x > 0 ? 1 : exp(x)), what autograd computes for `F.elu(x) + 1.0`. */
int fbla_elu1_bwd(const void* x, const void* dy, void* dx, int64_t n, int dtype, void* stream);

/* Depth-wise convolution of token rows on an H x W grid ("same" padding, stride 1): y[b, t, c] = bias[c % Cw] +
 * sum over the K x K taps of w[c % Cw][tap] * x[b, neighbour of t, c], zero outside the grid.  Replaces the blocks'
 * nn.Conv2d on a transposed view of the tokens (flash_bla/layers/mlla.py:92, rala.py:58, focused_la.py:88-93,
 * polaformer.py:97-101), which reads and writes the tokens where they are.  Token t of batch b is the C elements at
 * x + b * x_batch + t * x_row (strides in elements: whole 16-byte pieces, at least C; likewise y and g); w [Cw, K, K] and
 * bias [Cw] (or NULL) have the element type of x.  x, y and g hold B batches of H * W tokens (the batches of y may not
 * overlap).  K is 3, 5 or 7, C a multiple of Cw and of 8 (16-bit) or 4 (fp32).
 * flip != 0 applies the taps in reverse order: with the output's gradient as x and no bias, the gradient of x. */
int fbla_dwconv_fwd(const void* x, int64_t x_batch, int64_t x_row, const void* w, const void* bias, void* y,
                    int64_t y_batch, int64_t y_row, int64_t B, int64_t H, int64_t W, int C, int Cw, int K, int flip,
                    int dtype, void* stream);

/* Gradients of the filters: dw [Cw, K, K] and db [Cw] (either may be NULL) from x and the output's gradient g, summed
 * in fp32 in a fixed order and rounded once.  workspace: fbla_dwconv_grad_workspace_bytes bytes of device memory. */
size_t fbla_dwconv_grad_workspace_bytes(int64_t B, int64_t H, int64_t W, int C, int Cw, int K, int dtype);
int fbla_dwconv_grad(const void* x, int64_t x_batch, int64_t x_row, const void* g, int64_t g_batch, int64_t g_row,
                     void* dw, void* db, void* workspace, size_t workspace_bytes, int64_t B, int64_t H, int64_t W,
                     int C, int Cw, int K, int dtype, void* stream);

/* Gradients of a projection y = x W^T + b over token rows: dw [M, N] = sum over the tokens of g[t]^T x[t], db [M] (or NULL) =
 * the sum of g, in fp32 in a fixed order, rounded once.  What autograd computes for the blocks' nn.Linear layers
 * (flash_bla/layers/mlla.py:56, rala.py:31, focused_la.py:26-27, polaformer.py:24-25).  g: rows of M elements g_row
 * apart, x: rows of N elements x_row apart (whole 16-byte pieces); M and N multiples of 8 (16-bit) or 4 (fp32).
 * workspace: fbla_linear_wgrad_workspace_bytes bytes of device memory. */
size_t fbla_linear_wgrad_workspace_bytes(int64_t tokens, int M, int N, int dtype);
int fbla_linear_wgrad(const void* g, int64_t g_row, const void* x, int64_t x_row, void* dw, void* db, void* workspace,
                      size_t workspace_bytes, int64_t tokens, int M, int N, int dtype, void* stream);

/* Up to three projections of the same number of token rows in one launch (fp16 / bf16): out [tokens, N] = a W + a2 W2 + bias +
 * add, in fp32, rounded once.  rows_of_w = 0: w is [N, K] (nn.Linear's forward, a w^T; flash_bla/layers/mlla.py:56,
 * linfusion.py:26-38,83-103, rala.py:31, focused_la.py:26-27, polaformer.py:24-25); 1: w is [K, N] (its input gradient).  a2
 * (with w2 of K2 channels), bias [N] and add (rows) may be NULL.  Rows of a, a2, add and out lie a_row, .. elements apart
 * (whole 16-byte pieces, at least their channels); w without gaps; N and K multiples of 8; 16-byte aligned pointers.  out may
 * be add. */
typedef struct {
  const void* a;
  int64_t a_row;
  const void* w;
  const void* a2;
  int64_t a2_row;
  const void* w2;
  const void* bias;
  const void* add;
  int64_t add_row;
  void* out;
  int64_t out_row;
  int32_t N, K, K2;
} fbla_projection;
int fbla_project(const fbla_projection* jobs, int count, int64_t tokens, int rows_of_w, int dtype, void* stream);

/* LayerNorm over the C channels of contiguous rows and LeakyReLU (flash_bla/layers/linfusion.py:26-38), one or two sets of rows
 * in one launch, in fp32 and rounded once.  weight and bias [C] may be NULL; mean and rstd (fp32 [tokens], for a backward) may
 * both be NULL.  fp16 / bf16, C a multiple of 8 up to 2048. */
typedef struct {
  const void *x, *weight, *bias;
  void* out;
  float *mean, *rstd;
  float eps, slope;
} fbla_norm;
int fbla_norm_leaky(const fbla_norm* jobs, int count, int64_t tokens, int C, int dtype, void* stream);

/* What the vision blocks do between their projections and the attention operators.  Rows are [B, N, C], C = heads * d,
 * joint projections [B, N, 2 C], heads [B, heads, N, width]; contiguous, one element type, d in whole 16-byte pieces.
 *
 * Polarity features (flash_bla/layers/polaformer.py:63-84): with y = q / scale of qg's first half (the second half is the
 * gate and is not read) or (k + pe) / scale of kv's first half, pos = relu(y)^power and neg = relu(-y)^power;
 * q_same = pos | neg, q_opp = neg | pos, k_both = pos | neg as heads of 2 d, v_heads = kv's second half as heads of d.
 * pe [Nk, C], scale [C], power [heads, d] (at least 1).  The backward takes the gradients of the four outputs, of the
 * values as rows (dv_rows [B, Nk, C], added to dv) and of the gate as rows (dgate, copied into dqg). */
int fbla_polarity_fwd(const void* qg, const void* kv, const void* pe, const void* scale, const void* power, void* q_same,
                      void* q_opp, void* k_both, void* v_heads, int64_t B, int64_t N, int64_t Nk, int heads, int d, int dtype,
                      void* stream);
size_t fbla_polarity_bwd_workspace_bytes(int64_t B, int64_t N, int64_t Nk, int heads, int d, int dtype);
int fbla_polarity_bwd(const void* qg, const void* kv, const void* pe, const void* scale, const void* power,
                      const void* dq_same, const void* dq_opp, const void* dk_both, const void* dv_heads, const void* dv_rows,
                      const void* dgate, void* dqg, void* dkv, void* dpe, void* dscale, void* dpower, void* workspace,
                      size_t workspace_bytes, int64_t B, int64_t N, int64_t Nk, int heads, int d, int dtype, void* stream);

/* Rotary features (flash_bla/layers/mlla.py:74-81): q, k = elu(x) + 1 of the halves of qk, q_rot, k_rot = their channel
 * pairs turned by rot (fp32 [N, rot_channels / 2, 2]: cos, sin; channel c uses entry c % rot_channels), v = x, all as heads.
 * The backward adds dv_rows [B, N, C] to the values' gradient. */
int fbla_rotary_fwd(const void* qk, const void* x, const float* rot, int rot_channels, void* q, void* k, void* q_rot,
                    void* k_rot, void* v, int64_t B, int64_t N, int heads, int d, int dtype, void* stream);
int fbla_rotary_bwd(const void* qk, const float* rot, int rot_channels, const void* dq, const void* dk, const void* dq_rot,
                    const void* dk_rot, const void* dv, const void* dv_rows, void* dqk, void* dx, int64_t B, int64_t N,
                    int heads, int d, int dtype, void* stream);

/* Heads back to rows: out = (heads + local) * gate (flash_bla/layers/polaformer.py:92-104; without a gate mlla.py:88-92).
 * o2 not NULL: the channels of a head are the halves o | o2 of d / 2 each (whole 16-byte pieces).  gate: rows gate_row
 * elements apart, or NULL; then the backward writes d_o alone (dlocal is dout). */
int fbla_merge_fwd(const void* o, const void* o2, const void* local, const void* gate, int64_t gate_row, void* out, int64_t B,
                   int64_t N, int heads, int d, int dtype, void* stream);
int fbla_merge_bwd(const void* dout, const void* o, const void* o2, const void* local, const void* gate, int64_t gate_row,
                   void* d_o, void* d_o2, void* dlocal, void* dgate, int64_t B, int64_t N, int heads, int d, int dtype,
                   void* stream);

/* Linear interpolation of token rows from `from` to `to` tokens, the corners not aligned: what
 * F.interpolate(mode='linear', size=to) gives for the transposed rows (flash_bla/layers/focused_la.py:88-91,
 * polaformer.py:95-98).  x: token t of batch b is the C elements at x + b * x_batch + t * x_row (whole 16-byte pieces, at
 * least C); y and g [B, to, C], dx [B, from, C] contiguous; from * to below 2^28, C in whole 16-byte pieces. */
int fbla_interpolate_fwd(const void* x, int64_t x_batch, int64_t x_row, void* y, int64_t B, int64_t from, int64_t to, int C,
                         int dtype, void* stream);
int fbla_interpolate_bwd(const void* g, void* dx, int64_t B, int64_t from, int64_t to, int C, int dtype, void* stream);

/* Focused features (flash_bla/layers/focused_la.py:56-74, focusing factor 3): with t = (relu(x) + 1e-6) / scale of q
 * [B, N, C] or of kv's first half plus pe, the feature t^3 |t| / |t^3| (lengths over the C channels) as heads of d, and kv's
 * second half as heads v_out.  C in whole
 * 16-byte pieces, at most 2048 (16-bit) or 1024 (fp32).  The backward adds dv_rows [B, Nk, C] to the values' gradient. */
int fbla_focus_fwd(const void* q, const void* kv, const void* pe, const void* scale, void* q_out, void* k_out, void* v_out,
                   int64_t B, int64_t N, int64_t Nk, int heads, int d, int dtype, void* stream);
size_t fbla_focus_bwd_workspace_bytes(int64_t B, int64_t N, int64_t Nk, int heads, int d, int dtype);
int fbla_focus_bwd(const void* q, const void* kv, const void* pe, const void* scale, const void* dq_heads,
                   const void* dk_heads, const void* dv_heads, const void* dv_rows, void* dq, void* dkv, void* dpe,
                   void* dscale, void* workspace, size_t workspace_bytes, int64_t B, int64_t N, int64_t Nk, int heads, int d,
                   int dtype, void* stream);

/* The attention of two vision blocks on their projections' rows, heads of 32 channels, fp16 / bf16 (C = 32 * heads): with
 * features, state, output, merge and gate of flash_bla/layers/polaformer.py:63-104 (kind 0: polarity features of q and k, values v,
 * local values, gate; pe [Nk, C], scale [C] and power [C] the parameters: over softplus(scale), to 1 + alpha sigmoid(power),
 * alpha >= 0) or flash_bla/layers/mlla.py:74-92 (kind 1: rotary features of q
 * and k before elu + 1, values v, local values; N = Nk, rot fp32 [N, C / 2, 2]).  Rows of q, k, v, gate, dq, dk, dv, dgate lie
 * *_row elements apart (whole 16-byte pieces, at least C; batches one after the other); local, out, dout, dlocal, dv_more are
 * contiguous rows of C.
 *
 * forward: out = (attention + local) * gate (kind 1: no gate); state_planes (fbla_block_attn_state_elements of the type) and
 * state_km (fp32 [B, heads, 72] or [.., 40]) are written for the backward.  backward_queries: dout -> dq, kind 0 also dgate and
 * dlocal (kind 1: dlocal is dout).  backward_keys, after it with the same workspace: dk, dv = its gradient + dv_more, kind 0 also
 * dpe, dscale, dpower.  workspace: fbla_block_attn_workspace_bytes, any contents before forward and backward_queries. */
typedef struct {
  int32_t kind, dtype, B, N, Nk, heads;
  float eps;
  const void *q, *k, *v, *local, *gate;
  int64_t q_row, k_row, v_row, gate_row;
  const void *pe, *scale, *power;
  float alpha;
  const float* rot;
  void *out, *state_planes;
  float* state_km;
  const void *dout, *dv_more;
  void *dq, *dk, *dv, *dlocal, *dgate;
  int64_t dq_row, dk_row, dv_row, dgate_row;
  void *dpe, *dscale, *dpower;
  void* workspace;
  size_t workspace_bytes;
} fbla_block_attn;
size_t fbla_block_attn_workspace_bytes(int kind, int64_t B, int64_t N, int64_t Nk, int heads);
size_t fbla_block_attn_state_elements(int kind, int64_t B, int heads);
int fbla_block_attn_forward(const fbla_block_attn* a, void* stream);
int fbla_block_attn_backward_queries(const fbla_block_attn* a, void* stream);
int fbla_block_attn_backward_keys(const fbla_block_attn* a, void* stream);

/* Weighted and turned heads (flash_bla/layers/rala.py:60-69): k_out = k * weight, q_rot and k_rot = the channel pairs of q and
 * of k_out (before its rounding) turned by rot (fp32 [N, d / 2, 2]: cos, sin).  All heads are [B, heads, N, d], weight
 * [B, heads, N]; d a power of two of at most 64 16-byte pieces.  The backward gives the gradients through these outputs
 * alone (dq: through q_rot). */
int fbla_turn_fwd(const void* q, const void* k, const void* weight, const float* rot, void* k_out, void* q_rot, void* k_rot,
                  int64_t B, int64_t N, int heads, int d, int dtype, void* stream);
int fbla_turn_bwd(const void* k, const void* weight, const float* rot, const void* dk_out, const void* dq_rot,
                  const void* dk_rot, void* dq, void* dk, void* dweight, int64_t B, int64_t N, int heads, int d, int dtype,
                  void* stream);

#ifdef __cplusplus
}
#endif
#endif /* FLASH_BLA_HIP_H */
