// Host path of the Python operators: one call from Python per direction of an operator or a block, which allocates the
// outputs through torch, enqueues the launches of libfbla_hip.so on torch's current stream and returns.  No arithmetic
// happens here, nothing is kept between calls but the library's entry points.
//
// Why native: a call of six to twenty short kernels is bound by the host that issues it.  Through Python and ctypes an
// operator's forward and its backward took 14 us each to issue (8.5 here), a block's training step 300 to 1100 us
// (layers/_whole.py).
#include <ATen/hip/impl/HIPStreamMasqueradingAsCUDA.h>
#include <dlfcn.h>
#include <torch/csrc/Exceptions.h>
#include <torch/extension.h>

#include <algorithm>
#include <array>
#include <string>
#include <variant>
#include <vector>

#include "../../include/flash_bla_hip.h"

namespace {

namespace py = pybind11;
using at::Tensor;
using Maybe = std::optional<Tensor>;

// ---- the library's entry points -----------------------------------------------------------------------------------
#define FBLA_ENTRY_POINTS(X)                                                                                           \
  X(fbla_last_error) X(fbla_la_workspace_bytes) X(fbla_la_fwd) X(fbla_la_bwd) X(fbla_la_pair_workspace_bytes)          \
  X(fbla_la_pair_fwd) X(fbla_la_pair_bwd) X(fbla_la_cross_workspace_bytes) X(fbla_la_cross_fwd) X(fbla_la_cross_bwd)   \
  X(fbla_decoupled_cross_fwd) X(fbla_decoupled_cross_bwd) X(fbla_varlen_workspace_bytes) X(fbla_varlen_fwd)            \
  X(fbla_varlen_bwd) X(fbla_chunk_reduce_workspace_bytes) X(fbla_chunk_reduce) X(fbla_select_blocks)                   \
  X(fbla_piecewise_workspace_bytes) X(fbla_piecewise_fwd) X(fbla_elu1_fwd) X(fbla_elu1_bwd) X(fbla_dwconv_fwd)         \
  X(fbla_dwconv_grad_workspace_bytes) X(fbla_dwconv_grad) X(fbla_linear_wgrad_workspace_bytes) X(fbla_linear_wgrad)    \
  X(fbla_polarity_fwd) X(fbla_polarity_bwd_workspace_bytes) X(fbla_polarity_bwd) X(fbla_rotary_fwd) X(fbla_rotary_bwd) \
  X(fbla_merge_fwd) X(fbla_merge_bwd) X(fbla_turn_fwd) X(fbla_turn_bwd) X(fbla_focus_fwd)                              \
  X(fbla_focus_bwd_workspace_bytes) X(fbla_focus_bwd) X(fbla_interpolate_fwd) X(fbla_interpolate_bwd)                   \
  X(fbla_project) X(fbla_norm_leaky) X(fbla_block_attn_workspace_bytes) X(fbla_block_attn_state_elements)              \
  X(fbla_block_attn_forward) X(fbla_block_attn_backward_queries) X(fbla_block_attn_backward_keys)

struct Api {
#define FBLA_MEMBER(f) decltype(&::f) f = nullptr;
  FBLA_ENTRY_POINTS(FBLA_MEMBER)
#undef FBLA_MEMBER
};
Api api;

void load(const std::string& path) {
  void* lib = dlopen(path.c_str(), RTLD_NOW | RTLD_LOCAL);
  if (!lib) throw std::runtime_error("flash_bla: " + std::string(dlerror()));
  Api found;
  const char* missing = nullptr;
#define FBLA_FIND(f)                                                 \
  found.f = reinterpret_cast<decltype(&::f)>(dlsym(lib, #f));        \
  if (!found.f) missing = #f;
  FBLA_ENTRY_POINTS(FBLA_FIND)
#undef FBLA_FIND
  if (missing) throw std::runtime_error("flash_bla: " + path + " does not export " + missing);
  api = found;
}

void check(int rc, const char* what) {
  if (rc == 0) return;
  const std::string msg = std::string(what) + " failed (" + std::to_string(rc) + "): " + api.fbla_last_error();
  if (rc == FBLA_ERR_BAD_ARG || rc == FBLA_ERR_UNSUPPORTED) throw py::value_error(msg);
  throw std::runtime_error(msg);
}

// ---- tensors --------------------------------------------------------------------------------------------------------
Tensor given(const Maybe& t) { return t ? *t : Tensor(); }
void* ptr(const Tensor& t) { return t.defined() ? t.data_ptr() : nullptr; }
float* f32(const Tensor& t) { return static_cast<float*>(ptr(t)); }
bool off_piece(const Tensor& t) { return reinterpret_cast<uintptr_t>(t.data_ptr()) % 16 != 0; }

int code_of(const Tensor& t) {
  switch (t.scalar_type()) {
    case at::kHalf: return FBLA_F16;
    case at::kBFloat16: return FBLA_BF16;
    case at::kFloat: return FBLA_F32;
    default: throw py::type_error("q, k, and v must have dtype float16, bfloat16, or float32");
  }
}

void require_gpu(std::initializer_list<Tensor> tensors) {
  for (const Tensor& t : tensors)
    if (t.defined() && !t.is_cuda())
      throw py::value_error("flash_bla HIP operators need GPU tensors (got a CPU tensor); use the naive_* functions for CPU math");
}

// The tensor in contiguous memory on a 16-byte boundary, which the kernels' pieces need; a copy where it is not.
Tensor whole(const Tensor& t) {
  if (!t.defined()) return t;
  Tensor c = t.contiguous();
  return off_piece(c) ? c.clone(at::MemoryFormat::Contiguous) : c;
}
Tensor whole(const Maybe& t) { return t ? whole(*t) : Tensor(); }

// Token rows [B, N, C] that the kernels read in place: channels adjacent, rows and batches whole 16-byte pieces apart; a
// copy of anything else.
Tensor rows(const Tensor& t) {
  const int64_t piece = 16 / t.element_size(), C = t.size(2);
  if (t.stride(2) != 1 || t.stride(0) % piece || t.stride(1) % piece || t.stride(1) < C || t.stride(0) < C || off_piece(t))
    return t.clone(at::MemoryFormat::Contiguous);
  return t;
}
// The same with the batches' rows at one distance throughout.
Tensor rows_of_batches(const Tensor& t) {
  if (!t.defined()) return t;
  Tensor r = rows(t);
  return r.stride(0) != r.stride(1) * r.size(1) ? r.clone(at::MemoryFormat::Contiguous) : r;
}
// t [..., C] as rows [tokens, C] at a distance of whole pieces.
Tensor token_rows(const Tensor& t) {
  Tensor r = t.reshape({-1, t.size(-1)});
  if (r.stride(1) != 1 || r.stride(0) * r.element_size() % 16 || r.stride(0) < r.size(1) || off_piece(r))
    return r.clone(at::MemoryFormat::Contiguous);
  return r;
}

Tensor like(const Tensor& t, at::IntArrayRef shape) { return at::empty(shape, t.options().memory_format(std::nullopt)); }
Tensor like(const Tensor& t) { return at::empty(t.sizes(), t.options()); }
Tensor like_f32(const Tensor& t, at::IntArrayRef shape) { return at::empty(shape, t.options().dtype(at::kFloat)); }
Tensor scratch(size_t bytes, const Tensor& like) {
  return at::empty({std::max<int64_t>((int64_t)bytes, 1)}, like.options().dtype(at::kByte));
}

// A number that sizes are divided by (in C++ a division by zero ends the process).
void check_positive(const char* what, int64_t n) {
  if (n < 1) throw py::value_error(std::string(what) + " must be positive, got " + std::to_string(n));
}

// Makes the tensor's device the current one and holds torch's current stream there.
struct On {
  c10::DeviceGuard guard;
  void* stream;
  explicit On(const Tensor& t)
      : guard(t.device()), stream(at::hip::getCurrentHIPStreamMasqueradingAsCUDA(t.get_device()).stream()) {}
};

// ---- operators --------------------------------------------------------------------------------------------------------
struct Attended {
  Tensor o, s, km;
};

// q [B,H,L,DK], k [B,H,Lk,DK], v [B,H,Lk,DV], with the decoupled operator also their rotary rows; contiguous
Attended la_fwd(const Tensor& q_, const Tensor& k_, const Tensor& v_, const Tensor& qr_, const Tensor& kr_, double scale, double eps,
                int flags) {
  require_gpu({q_, k_, v_, qr_, kr_});
  const Tensor q = whole(q_), k = whole(k_), v = whole(v_), qr = whole(qr_), kr = whole(kr_);
  const int64_t B = q.size(0), H = q.size(1), T = q.size(2), Tk = k.size(2);
  const int DK = q.size(3), DV = v.size(3), code = code_of(q);
  Attended r{like(v, {B, H, T, DV}), like_f32(q, {B, H, DK, DV}), like_f32(q, {B, H, DK})};
  const On on(q);
  const bool decoupled = flags & FBLA_DECOUPLED;
  const size_t need = Tk == T ? api.fbla_la_workspace_bytes(0, B, H, T, DK, DV, code, flags)
                              : api.fbla_la_cross_workspace_bytes(0, B, H, T, Tk, DK, DV, code, flags);
  const Tensor ws = scratch(need, q);
  const size_t bytes = ws.numel();
  if (Tk == T)
    check(api.fbla_la_fwd(ptr(q), ptr(k), ptr(v), ptr(qr), ptr(kr), ptr(r.o), f32(r.s), f32(r.km), ptr(ws), bytes, B, H, T, DK, DV,
                          code, flags, scale, eps, on.stream), "fbla_la_fwd");
  else if (decoupled)
    check(api.fbla_decoupled_cross_fwd(ptr(q), ptr(k), ptr(qr), ptr(kr), ptr(v), ptr(r.o), f32(r.s), f32(r.km), ptr(ws), bytes, B, H, T,
                                       Tk, DK, DV, code, scale, eps, on.stream), "fbla_decoupled_cross_fwd");
  else
    check(api.fbla_la_cross_fwd(ptr(q), ptr(k), ptr(v), ptr(r.o), f32(r.s), f32(r.km), ptr(ws), bytes, B, H, T, Tk, DK, DV, code, flags,
                                scale, eps, on.stream), "fbla_la_cross_fwd");
  return r;
}

struct AttendedGrads {
  Tensor q, k, v, q_rope, k_rope;
};

AttendedGrads la_bwd(const Tensor& q_, const Tensor& k_, const Tensor& v_, const Tensor& qr_, const Tensor& kr_, const Tensor& do_,
                     const Tensor& s_, const Tensor& km_, double scale, double eps, int flags) {
  require_gpu({q_, k_, v_, do_});
  const Tensor q = whole(q_), k = whole(k_), v = whole(v_), qr = whole(qr_), kr = whole(kr_), g = whole(do_), s = whole(s_),
               km = whole(km_);
  const int64_t B = q.size(0), H = q.size(1), T = q.size(2), Tk = k.size(2);
  const int DK = q.size(3), DV = v.size(3), code = code_of(q);
  const bool decoupled = flags & FBLA_DECOUPLED;
  AttendedGrads d{like(q), like(k), like(v), decoupled ? like(qr) : Tensor(), decoupled ? like(kr) : Tensor()};
  const On on(q);
  const size_t need = Tk == T ? api.fbla_la_workspace_bytes(1, B, H, T, DK, DV, code, flags)
                              : api.fbla_la_cross_workspace_bytes(1, B, H, T, Tk, DK, DV, code, flags);
  const Tensor ws = scratch(need, q);
  const size_t bytes = ws.numel();
  if (Tk == T)
    check(api.fbla_la_bwd(ptr(q), ptr(k), ptr(v), ptr(qr), ptr(kr), ptr(g), f32(s), f32(km), ptr(d.q), ptr(d.k), ptr(d.v), ptr(d.q_rope),
                          ptr(d.k_rope), ptr(ws), bytes, B, H, T, DK, DV, code, flags, scale, eps, on.stream), "fbla_la_bwd");
  else if (decoupled)
    check(api.fbla_decoupled_cross_bwd(ptr(q), ptr(k), ptr(qr), ptr(kr), ptr(v), ptr(g), f32(s), f32(km), ptr(d.q), ptr(d.k),
                                       ptr(d.q_rope), ptr(d.k_rope), ptr(d.v), ptr(ws), bytes, B, H, T, Tk, DK, DV, code, scale, eps,
                                       on.stream), "fbla_decoupled_cross_bwd");
  else
    check(api.fbla_la_cross_bwd(ptr(q), ptr(k), ptr(v), ptr(g), f32(s), f32(km), ptr(d.q), ptr(d.k), ptr(d.v), ptr(ws), bytes, B, H, T,
                                Tk, DK, DV, code, flags, scale, eps, on.stream), "fbla_la_cross_bwd");
  return d;
}

bool pair_supported(const Tensor& q, const Tensor& v) {
  return q.is_cuda() && (q.scalar_type() == at::kHalf || q.scalar_type() == at::kBFloat16) &&
         api.fbla_la_pair_workspace_bytes(0, q.size(0), q.size(1), q.size(2), q.size(3), v.size(3), code_of(q)) != 0;
}

struct Paired {
  Tensor o1, o2, s, km;
};

Paired pair_fwd(const Tensor& q1_, const Tensor& q2_, const Tensor& k_, const Tensor& v_, double scale, double eps) {
  require_gpu({q1_, q2_, k_, v_});
  const Tensor q1 = whole(q1_), q2 = whole(q2_), k = whole(k_), v = whole(v_);
  const int64_t B = q1.size(0), H = q1.size(1), T = q1.size(2);
  const int DK = q1.size(3), DV = v.size(3), code = code_of(q1);
  Paired r{like(v, {B, H, T, DV / 2}), like(v, {B, H, T, DV / 2}), like_f32(q1, {B, H, DK, DV}), like_f32(q1, {B, H, DK})};
  const On on(q1);
  const Tensor ws = scratch(api.fbla_la_pair_workspace_bytes(0, B, H, T, DK, DV, code), q1);
  check(api.fbla_la_pair_fwd(ptr(q1), ptr(q2), ptr(k), ptr(v), ptr(r.o1), ptr(r.o2), f32(r.s), f32(r.km), ptr(ws), ws.numel(), B, H, T,
                             DK, DV, code, scale, eps, on.stream), "fbla_la_pair_fwd");
  return r;
}

struct PairedGrads {
  Tensor q1, q2, k, v;
};

PairedGrads pair_bwd(const Tensor& q1_, const Tensor& q2_, const Tensor& k_, const Tensor& v_, const Tensor& do1_, const Tensor& do2_,
                     const Tensor& s_, const Tensor& km_, double scale, double eps) {
  require_gpu({q1_, q2_, k_, v_, do1_, do2_});
  const Tensor q1 = whole(q1_), q2 = whole(q2_), k = whole(k_), v = whole(v_), g1 = whole(do1_), g2 = whole(do2_), s = whole(s_),
               km = whole(km_);
  const int64_t B = q1.size(0), H = q1.size(1), T = q1.size(2);
  const int DK = q1.size(3), DV = v.size(3), code = code_of(q1);
  PairedGrads d{like(q1), like(q2), like(k), like(v)};
  const On on(q1);
  const Tensor ws = scratch(api.fbla_la_pair_workspace_bytes(1, B, H, T, DK, DV, code), q1);
  check(api.fbla_la_pair_bwd(ptr(q1), ptr(q2), ptr(k), ptr(v), ptr(g1), ptr(g2), f32(s), f32(km), ptr(d.q1), ptr(d.q2), ptr(d.k), ptr(d.v),
                             ptr(ws), ws.numel(), B, H, T, DK, DV, code, scale, eps, on.stream), "fbla_la_pair_bwd");
  return d;
}

// packed q, k [T,H,DK], v [T,H,DV], int32 cu [N + 1]
Attended varlen_fwd(const Tensor& q_, const Tensor& k_, const Tensor& v_, const Tensor& cu_, int64_t longest, std::optional<double> scale,
                    double eps, int extra) {
  require_gpu({q_, k_, v_, cu_});
  const Tensor q = whole(q_), k = whole(k_), v = whole(v_), cu = whole(cu_);
  const int64_t T = q.size(0), H = q.size(1), N = cu.numel() - 1;
  const int DK = q.size(2), DV = v.size(2), code = code_of(q);
  const int flags = FBLA_NORMALIZE | (scale ? 0 : FBLA_DEFAULT_SCALE) | extra;
  Attended r{like(v), like_f32(q, {N, H, DK, DV}), like_f32(q, {N, H, DK})};
  const On on(q);
  const Tensor ws = scratch(api.fbla_varlen_workspace_bytes(0, T, N, H, longest, DK, DV, code, flags), q);
  check(api.fbla_varlen_fwd(ptr(q), ptr(k), ptr(v), static_cast<const int32_t*>(ptr(cu)), ptr(r.o), f32(r.s), f32(r.km), ptr(ws),
                            ws.numel(), T, N, H, longest, DK, DV, code, flags, scale.value_or(0.0), eps, on.stream), "fbla_varlen_fwd");
  return r;
}

std::tuple<Tensor, Tensor, Tensor> varlen_bwd(const Tensor& q_, const Tensor& k_, const Tensor& v_, const Tensor& cu_, int64_t longest,
                                              const Tensor& do_, const Tensor& s_, const Tensor& km_, std::optional<double> scale,
                                              double eps, int extra) {
  require_gpu({q_, k_, v_, do_, cu_});
  const Tensor q = whole(q_), k = whole(k_), v = whole(v_), cu = whole(cu_), g = whole(do_), s = whole(s_), km = whole(km_);
  const int64_t T = q.size(0), H = q.size(1), N = cu.numel() - 1;
  const int DK = q.size(2), DV = v.size(2), code = code_of(q);
  const int flags = FBLA_NORMALIZE | (scale ? 0 : FBLA_DEFAULT_SCALE) | extra;
  Tensor dq = like(q), dk = like(k), dv = like(v);
  const On on(q);
  const Tensor ws = scratch(api.fbla_varlen_workspace_bytes(1, T, N, H, longest, DK, DV, code, flags), q);
  check(api.fbla_varlen_bwd(ptr(q), ptr(k), ptr(v), static_cast<const int32_t*>(ptr(cu)), ptr(g), f32(s), f32(km), ptr(dq), ptr(dk), ptr(dv),
                            ptr(ws), ws.numel(), T, N, H, longest, DK, DV, code, flags, scale.value_or(0.0), eps, on.stream),
        "fbla_varlen_bwd");
  return {dq, dk, dv};
}

// ---- piecewise attention --------------------------------------------------------------------------------------------
struct Statistics {
  Tensor qc, kc, vc, h, h_norm;
};

Statistics chunk_reduce(const Tensor& q_, const Tensor& k_, const Tensor& v_, int64_t chunk, bool with_norm, double p_norm) {
  check_positive("chunk", chunk);
  require_gpu({q_, k_, v_});
  const Tensor q = whole(q_), k = whole(k_), v = whole(v_);
  const int64_t B = k.size(0), H = k.size(1), T = k.size(2), NT = (T + chunk - 1) / chunk;
  const int K = k.size(3), V = v.size(3), code = code_of(q);
  Statistics r{like_f32(q, {B, H, NT, K}), like_f32(q, {B, H, NT, K}), like_f32(q, {B, H, NT, V}), like_f32(q, {B, H, K, V}),
               with_norm ? like_f32(q, {B, H, NT}) : Tensor()};
  const On on(q);
  const Tensor ws = scratch(api.fbla_chunk_reduce_workspace_bytes(B * H, T, K, V, chunk, code, with_norm), q);
  check(api.fbla_chunk_reduce(ptr(q), ptr(k), ptr(v), f32(r.qc), f32(r.kc), f32(r.vc), f32(r.h), f32(r.h_norm), ptr(ws), ws.numel(), B * H,
                              T, K, V, chunk, p_norm, code, on.stream), "fbla_chunk_reduce");
  return r;
}

Tensor select_blocks(const Tensor& qc_, const Tensor& kc_, const Tensor& bias_, int64_t top, double scale) {
  require_gpu({qc_, kc_, bias_});
  const Tensor qc = whole(qc_), kc = whole(kc_), bias = whole(bias_);
  const int64_t B = qc.size(0), H = qc.size(1), NT = qc.size(2);
  const Tensor index = at::empty({B, H, NT, top}, qc.options().dtype(at::kInt));
  const On on(qc);
  check(api.fbla_select_blocks(f32(qc), f32(kc), f32(bias), static_cast<int32_t*>(ptr(index)), B * H, NT, qc.size(3), top, scale,
                               on.stream), "fbla_select_blocks");
  return index;
}

bool piecewise_supported(const Tensor& q, const Tensor& v, int64_t block) {
  const at::ScalarType t = q.scalar_type();
  return (t == at::kHalf || t == at::kBFloat16 || t == at::kFloat) &&
         api.fbla_piecewise_workspace_bytes(q.size(0) * q.size(1), q.size(2), q.size(3), v.size(3), block, code_of(q)) != 0;
}

Tensor piecewise_fwd(const Tensor& q_, const Tensor& k_, const Tensor& v_, const Tensor& kc_, const Tensor& vc_, const Tensor& h_,
                     const Tensor& index_, int64_t block, double scale) {
  require_gpu({q_, k_, v_, kc_, vc_, h_, index_});
  const Tensor q = whole(q_), k = whole(k_), v = whole(v_), kc = whole(kc_), vc = whole(vc_), h = whole(h_), index = whole(index_);
  const int64_t BH = q.size(0) * q.size(1), T = q.size(2);
  const int K = q.size(3), V = v.size(3), code = code_of(q);
  const Tensor o = like(v);
  const On on(q);
  const Tensor ws = scratch(api.fbla_piecewise_workspace_bytes(BH, T, K, V, block, code), q);
  check(api.fbla_piecewise_fwd(ptr(q), ptr(k), ptr(v), f32(kc), f32(vc), f32(h), static_cast<const int32_t*>(ptr(index)), ptr(o), ptr(ws),
                               ws.numel(), BH, T, K, V, block, index.size(-1), scale, code, on.stream), "fbla_piecewise_fwd");
  return o;
}

// ---- feature map ------------------------------------------------------------------------------------------------------
std::pair<Tensor, Tensor> elu1_fwd(const Tensor& x0_, const Tensor& x1_) {
  require_gpu({x0_, x1_});
  const Tensor x0 = whole(x0_), x1 = whole(x1_);
  if (x1.defined() && (x1.scalar_type() != x0.scalar_type() || x1.device() != x0.device()))
    throw py::value_error("elu1_fwd: both tensors must have the same dtype and device");
  Tensor y0 = like(x0), y1 = x1.defined() ? like(x1) : Tensor();
  const On on(x0);
  check(api.fbla_elu1_fwd(ptr(x0), ptr(y0), x0.numel(), ptr(x1), ptr(y1), x1.defined() ? x1.numel() : 0, code_of(x0), on.stream),
        "fbla_elu1_fwd");
  return {y0, y1};
}

Tensor elu1_bwd(const Tensor& x_, const Tensor& dy_) {
  require_gpu({x_, dy_});
  const Tensor x = whole(x_), dy = whole(dy_);
  const Tensor dx = like(x);
  const On on(x);
  check(api.fbla_elu1_bwd(ptr(x), ptr(dy), ptr(dx), x.numel(), code_of(x), on.stream), "fbla_elu1_bwd");
  return dx;
}

// ---- around the operators ---------------------------------------------------------------------------------------------
void check_grid(const char* what, const Tensor& x, int64_t H, int64_t W) {
  if (x.size(1) != H * W || H < 1)
    throw py::value_error(std::string(what) + ": x must be rows of H * W tokens, got " + std::to_string(x.size(1)) + " for H = " +
                          std::to_string(H) + ", W = " + std::to_string(W));
}

Tensor dwconv_fwd(const Tensor& x_, const Tensor& w_, const Tensor& bias_, int64_t H, int64_t W, bool flip) {
  check_grid("dwconv_fwd", x_, H, W);
  if (w_.scalar_type() != x_.scalar_type() || (bias_.defined() && bias_.scalar_type() != x_.scalar_type()))
    throw py::value_error("dwconv_fwd: x, w and bias must have one dtype");
  require_gpu({x_, w_, bias_});
  const Tensor x = rows(x_), w = w_.contiguous(), bias = bias_.defined() ? bias_.contiguous() : Tensor();
  const int64_t B = x.size(0), N = x.size(1), C = x.size(2);
  const Tensor y = like(x, {B, N, C});
  const On on(x);
  check(api.fbla_dwconv_fwd(ptr(x), x.stride(0), x.stride(1), ptr(w), ptr(bias), ptr(y), N * C, C, B, H, W, C, w.size(0), w.size(-1), flip,
                            code_of(x), on.stream), "fbla_dwconv_fwd");
  return y;
}

std::pair<Tensor, Tensor> dwconv_grad(const Tensor& x_, const Tensor& g_, const Tensor& w, int64_t H, int64_t W, bool with_bias) {
  check_grid("dwconv_grad", x_, H, W);
  if (g_.sizes() != x_.sizes()) throw py::value_error("dwconv_grad: x and g must have one shape");
  if (w.scalar_type() != x_.scalar_type() || g_.scalar_type() != x_.scalar_type())
    throw py::value_error("dwconv_grad: x, g and w must have one dtype");
  require_gpu({x_, g_, w});
  const Tensor x = rows(x_), g = rows(g_);
  const int64_t B = x.size(0), C = x.size(2);
  const int Cw = w.size(0), K = w.size(-1), code = code_of(x);
  Tensor dw = like(w, w.sizes()), db = with_bias ? like(w, {Cw}) : Tensor();
  const On on(x);
  const Tensor ws = scratch(api.fbla_dwconv_grad_workspace_bytes(B, H, W, C, Cw, K, code), x);
  check(api.fbla_dwconv_grad(ptr(x), x.stride(0), x.stride(1), ptr(g), g.stride(0), g.stride(1), ptr(dw), ptr(db), ptr(ws), ws.numel(), B, H,
                             W, C, Cw, K, code, on.stream), "fbla_dwconv_grad");
  return {dw, db};
}

std::pair<Tensor, Tensor> linear_wgrad(const Tensor& g_, const Tensor& x_, bool with_bias) {
  require_gpu({g_, x_});
  const Tensor g = token_rows(g_), x = token_rows(x_);
  const int64_t T = g.size(0), M = g.size(1), N = x.size(1);
  if (x.size(0) != T || g.scalar_type() != x.scalar_type() || g.device() != x.device())
    throw py::value_error("linear_wgrad: g and x must agree in tokens, dtype and device");
  const int code = code_of(x);
  Tensor dw = like(x, {M, N}), db = with_bias ? like(x, {M}) : Tensor();
  const On on(x);
  const Tensor ws = scratch(api.fbla_linear_wgrad_workspace_bytes(T, M, N, code), x);
  check(api.fbla_linear_wgrad(ptr(g), g.stride(0), ptr(x), x.stride(0), ptr(dw), ptr(db), ptr(ws), ws.numel(), T, M, N, code, on.stream),
        "fbla_linear_wgrad");
  return {dw, db};
}

// Projections of rows with one number of tokens, 16-bit types: out = a W^T + bias + add, or (rows_of_w) a W + a2 W2 + add.
struct Projection {
  Tensor a, w, bias, add, a2, w2;
};
std::vector<Tensor> project(const std::vector<Projection>& p, bool rows_of_w) {
  TORCH_CHECK(!p.empty() && p.size() <= 3);
  std::array<fbla_projection, 3> jobs{};
  std::vector<Tensor> keep, out;
  auto ready = [&](const Tensor& t) {
    if (!t.defined()) return t;
    const Tensor r = token_rows(t);
    keep.push_back(r);
    return r;
  };
  int64_t tokens = -1;
  for (size_t i = 0; i < p.size(); ++i) {
    const Tensor a = ready(p[i].a), a2 = ready(p[i].a2), add = ready(p[i].add), w = whole(p[i].w), w2 = whole(p[i].w2),
                 bias = whole(p[i].bias);
    keep.insert(keep.end(), {w, w2, bias});
    const int64_t N = rows_of_w ? w.size(1) : w.size(0), K = rows_of_w ? w.size(0) : w.size(1);
    if (tokens < 0) tokens = a.size(0);
    TORCH_CHECK(a.size(0) == tokens && a.size(1) == K && (!a2.defined() || (a2.size(0) == tokens && a2.size(1) == w2.size(0))) &&
                (!add.defined() || (add.size(0) == tokens && add.size(1) == N)));
    std::vector<int64_t> shape = p[i].a.sizes().vec();
    shape.back() = N;
    out.push_back(like(a, shape));
    jobs[i] = {ptr(a), a.stride(0), ptr(w), ptr(a2), a2.defined() ? a2.stride(0) : 0, ptr(w2), ptr(bias), ptr(add),
               add.defined() ? add.stride(0) : 0, ptr(out[i]), N, (int32_t)N, (int32_t)K, a2.defined() ? (int32_t)a2.size(1) : 0};
  }
  const On on(p[0].a);
  check(api.fbla_project(jobs.data(), p.size(), tokens, rows_of_w, code_of(p[0].a), on.stream), "fbla_project");
  return out;
}

// LeakyReLU of LayerNorm over rows, one or two sets of one shape; mean and rstd as torch's LayerNorm saves them
struct Norm {
  Tensor x, weight, bias;
  double eps, slope;
};
struct Normed {
  Tensor y, mean, rstd;
};
std::vector<Normed> norm_leaky(const std::vector<Norm>& p, bool with_stats) {
  TORCH_CHECK(!p.empty() && p.size() <= 2);
  std::array<fbla_norm, 2> jobs{};
  std::vector<Tensor> keep;
  std::vector<Normed> r;
  const int64_t C = p[0].x.size(-1);
  check_positive("channels", C);
  const int64_t tokens = p[0].x.numel() / C;
  for (size_t i = 0; i < p.size(); ++i) {
    TORCH_CHECK(p[i].x.sizes() == p[0].x.sizes());
    const Tensor x = whole(p[i].x), weight = whole(p[i].weight), bias = whole(p[i].bias);
    keep.insert(keep.end(), {x, weight, bias});
    std::vector<int64_t> shape = x.sizes().vec();
    shape.back() = 1;
    r.push_back({like(x), with_stats ? like_f32(x, shape) : Tensor(), with_stats ? like_f32(x, shape) : Tensor()});
    jobs[i] = {ptr(x), ptr(weight), ptr(bias), ptr(r[i].y), f32(r[i].mean), f32(r[i].rstd), (float)p[i].eps, (float)p[i].slope};
  }
  const On on(p[0].x);
  check(api.fbla_norm_leaky(jobs.data(), p.size(), tokens, C, code_of(p[0].x), on.stream), "fbla_norm_leaky");
  return r;
}

// qg [B,N,2C], kv [B,n,2C], pe [1,n,C], scale [1,1,C], power [1,heads,1,d] -> q_same, q_opp, k_both [B,heads,.,2d], v [B,heads,n,d]
std::array<Tensor, 4> polarity_fwd(const Tensor& qg_, const Tensor& kv_, const Tensor& pe_, const Tensor& scale_, const Tensor& power_,
                                   int64_t heads) {
  check_positive("heads", heads);
  require_gpu({qg_, kv_, pe_, scale_, power_});
  const Tensor qg = whole(qg_), kv = whole(kv_), pe = whole(pe_), scale = whole(scale_), power = whole(power_);
  const int64_t B = qg.size(0), N = qg.size(1), n = kv.size(1), d = qg.size(2) / 2 / heads;
  std::array<Tensor, 4> r{like(qg, {B, heads, N, 2 * d}), like(qg, {B, heads, N, 2 * d}), like(qg, {B, heads, n, 2 * d}),
                          like(qg, {B, heads, n, d})};
  const On on(qg);
  check(api.fbla_polarity_fwd(ptr(qg), ptr(kv), ptr(pe), ptr(scale), ptr(power), ptr(r[0]), ptr(r[1]), ptr(r[2]), ptr(r[3]), B, N, n, heads,
                              d, code_of(qg), on.stream), "fbla_polarity_fwd");
  return r;
}

// gradients of qg, kv, pe, scale and power
std::array<Tensor, 5> polarity_bwd(const Tensor& qg_, const Tensor& kv_, const Tensor& pe_, const Tensor& scale_, const Tensor& power_,
                                   int64_t heads, const Tensor& dq_same, const Tensor& dq_opp, const Tensor& dk_both, const Tensor& dv,
                                   const Tensor& dv_rows, const Tensor& dgate) {
  check_positive("heads", heads);
  require_gpu({qg_, kv_, pe_, scale_, power_, dq_same, dq_opp, dk_both, dv, dv_rows, dgate});
  const Tensor qg = whole(qg_), kv = whole(kv_), pe = whole(pe_), scale = whole(scale_), power = whole(power_);
  const std::array<Tensor, 6> g{whole(dq_same), whole(dq_opp), whole(dk_both), whole(dv), whole(dv_rows), whole(dgate)};
  const int64_t B = qg.size(0), N = qg.size(1), n = kv.size(1), d = qg.size(2) / 2 / heads;
  const int code = code_of(qg);
  std::array<Tensor, 5> r{like(qg), like(kv), like(pe), like(scale), like(power)};
  const On on(qg);
  const Tensor ws = scratch(api.fbla_polarity_bwd_workspace_bytes(B, N, n, heads, d, code), qg);
  check(api.fbla_polarity_bwd(ptr(qg), ptr(kv), ptr(pe), ptr(scale), ptr(power), ptr(g[0]), ptr(g[1]), ptr(g[2]), ptr(g[3]), ptr(g[4]),
                              ptr(g[5]), ptr(r[0]), ptr(r[1]), ptr(r[2]), ptr(r[3]), ptr(r[4]), ptr(ws), ws.numel(), B, N, n, heads, d, code,
                              on.stream), "fbla_polarity_bwd");
  return r;
}

// qk [B,N,2C], x [B,N,C], rotations fp32 [..., pairs, 2] over the N tokens -> q, k, q_rot, k_rot, v [B,heads,N,d]
std::array<Tensor, 5> rotary_fwd(const Tensor& qk_, const Tensor& x_, const Tensor& rotations_, int64_t heads) {
  check_positive("heads", heads);
  require_gpu({qk_, x_, rotations_});
  const Tensor qk = whole(qk_), x = whole(x_), rotations = whole(rotations_);
  const int64_t B = x.size(0), N = x.size(1), d = x.size(2) / heads;
  std::array<Tensor, 5> r;
  for (Tensor& t : r) t = like(x, {B, heads, N, d});
  const On on(x);
  check(api.fbla_rotary_fwd(ptr(qk), ptr(x), f32(rotations), 2 * rotations.size(-2), ptr(r[0]), ptr(r[1]), ptr(r[2]), ptr(r[3]), ptr(r[4]), B,
                            N, heads, d, code_of(x), on.stream), "fbla_rotary_fwd");
  return r;
}

// gradients of qk and x; dv_rows [B,N,C] is added to the values' gradient
std::pair<Tensor, Tensor> rotary_bwd(const Tensor& qk_, const Tensor& rotations_, int64_t heads, const Tensor& dq, const Tensor& dk,
                                     const Tensor& dq_rot, const Tensor& dk_rot, const Tensor& dv, const Tensor& dv_rows) {
  check_positive("heads", heads);
  require_gpu({qk_, rotations_, dq, dk, dq_rot, dk_rot, dv, dv_rows});
  const Tensor qk = whole(qk_), rotations = whole(rotations_);
  const std::array<Tensor, 6> g{whole(dq), whole(dk), whole(dq_rot), whole(dk_rot), whole(dv), whole(dv_rows)};
  const int64_t B = g[5].size(0), N = g[5].size(1), C = g[5].size(2);
  Tensor dqk = like(qk), dx = like(g[5]);
  const On on(qk);
  check(api.fbla_rotary_bwd(ptr(qk), f32(rotations), 2 * rotations.size(-2), ptr(g[0]), ptr(g[1]), ptr(g[2]), ptr(g[3]), ptr(g[4]), ptr(g[5]),
                            ptr(dqk), ptr(dx), B, N, heads, C / heads, code_of(qk), on.stream), "fbla_rotary_bwd");
  return {dqk, dx};
}

// (heads + local) * gate as rows: o [B,heads,N,d], or o and o2 [B,heads,N,d/2] each
Tensor merge_fwd(const Tensor& o_, const Tensor& o2_, const Tensor& local_, const Tensor& gate_) {
  require_gpu({o_, o2_, local_, gate_});
  const Tensor o = whole(o_), o2 = whole(o2_), local = whole(local_), gate = rows_of_batches(gate_);
  const int64_t B = o.size(0), heads = o.size(1), N = o.size(2), d = o2.defined() ? 2 * o.size(3) : o.size(3);
  const Tensor out = like(local);
  const On on(o);
  check(api.fbla_merge_fwd(ptr(o), ptr(o2), ptr(local), ptr(gate), gate.defined() ? gate.stride(1) : 0, ptr(out), B, N, heads, d, code_of(o),
                           on.stream), "fbla_merge_fwd");
  return out;
}

struct MergeGrads {
  Tensor o, o2, local, gate;
};

// without a gate o, o2 and local are not looked at
MergeGrads merge_bwd(const Tensor& dout_, int64_t heads, bool halves, const Tensor& o_, const Tensor& o2_, const Tensor& local_,
                     const Tensor& gate_) {
  check_positive("heads", heads);
  require_gpu({dout_, o_, o2_, local_, gate_});
  const Tensor dout = whole(dout_), o = whole(o_), o2 = whole(o2_), local = whole(local_), gate = rows_of_batches(gate_);
  const int64_t B = dout.size(0), N = dout.size(1), d = dout.size(2) / heads, width = halves ? d / 2 : d;
  MergeGrads r{like(dout, {B, heads, N, width}), halves ? like(dout, {B, heads, N, width}) : Tensor(), dout, Tensor()};
  if (gate.defined()) {
    r.local = like(dout);
    r.gate = like(dout);
  }
  const On on(dout);
  check(api.fbla_merge_bwd(ptr(dout), ptr(o), ptr(o2), ptr(local), ptr(gate), gate.defined() ? gate.stride(1) : 0, ptr(r.o), ptr(r.o2),
                           gate.defined() ? ptr(r.local) : nullptr, ptr(r.gate), B, N, heads, d, code_of(dout), on.stream),
        "fbla_merge_bwd");
  return r;
}

Tensor interpolate_fwd(const Tensor& x_, int64_t tokens) {
  require_gpu({x_});
  const Tensor x = rows(x_);
  const int64_t B = x.size(0), n = x.size(1), C = x.size(2);
  const Tensor y = like(x, {B, tokens, C});
  const On on(x);
  check(api.fbla_interpolate_fwd(ptr(x), x.stride(0), x.stride(1), ptr(y), B, n, tokens, C, code_of(x), on.stream), "fbla_interpolate_fwd");
  return y;
}

Tensor interpolate_bwd(const Tensor& g_, int64_t n) {
  require_gpu({g_});
  const Tensor g = whole(g_);
  const int64_t B = g.size(0), C = g.size(2);
  const Tensor dx = like(g, {B, n, C});
  const On on(g);
  check(api.fbla_interpolate_bwd(ptr(g), ptr(dx), B, n, g.size(1), C, code_of(g), on.stream), "fbla_interpolate_bwd");
  return dx;
}

// q [B,N,C], kv [B,n,2C], pe [1,n,C], scale [1,1,C] -> q, k, v [B,heads,tokens,d]
std::array<Tensor, 3> focus_fwd(const Tensor& q_, const Tensor& kv_, const Tensor& pe_, const Tensor& scale_, int64_t heads) {
  check_positive("heads", heads);
  require_gpu({q_, kv_, pe_, scale_});
  const Tensor q = whole(q_), kv = whole(kv_), pe = whole(pe_), scale = whole(scale_);
  const int64_t B = q.size(0), N = q.size(1), n = kv.size(1), d = q.size(2) / heads;
  std::array<Tensor, 3> r{like(q, {B, heads, N, d}), like(q, {B, heads, n, d}), like(q, {B, heads, n, d})};
  const On on(q);
  check(api.fbla_focus_fwd(ptr(q), ptr(kv), ptr(pe), ptr(scale), ptr(r[0]), ptr(r[1]), ptr(r[2]), B, N, n, heads, d, code_of(q), on.stream),
        "fbla_focus_fwd");
  return r;
}

// gradients of q, kv, pe and scale; dv_rows [B,n,C] is added to the values' gradient
std::array<Tensor, 4> focus_bwd(const Tensor& q_, const Tensor& kv_, const Tensor& pe_, const Tensor& scale_, int64_t heads,
                                const Tensor& dq, const Tensor& dk, const Tensor& dv, const Tensor& dv_rows) {
  check_positive("heads", heads);
  require_gpu({q_, kv_, pe_, scale_, dq, dk, dv, dv_rows});
  const Tensor q = whole(q_), kv = whole(kv_), pe = whole(pe_), scale = whole(scale_);
  const std::array<Tensor, 4> g{whole(dq), whole(dk), whole(dv), whole(dv_rows)};
  const int64_t B = q.size(0), N = q.size(1), n = kv.size(1), d = q.size(2) / heads;
  const int code = code_of(q);
  std::array<Tensor, 4> r{like(q), like(kv), like(pe), like(scale)};
  const On on(q);
  const Tensor ws = scratch(api.fbla_focus_bwd_workspace_bytes(B, N, n, heads, d, code), q);
  check(api.fbla_focus_bwd(ptr(q), ptr(kv), ptr(pe), ptr(scale), ptr(g[0]), ptr(g[1]), ptr(g[2]), ptr(g[3]), ptr(r[0]), ptr(r[1]), ptr(r[2]),
                           ptr(r[3]), ptr(ws), ws.numel(), B, N, n, heads, d, code, on.stream), "fbla_focus_bwd");
  return r;
}

std::array<Tensor, 3> turn_fwd(const Tensor& q_, const Tensor& k_, const Tensor& weight_, const Tensor& rotations_) {
  require_gpu({q_, k_, weight_, rotations_});
  const Tensor q = whole(q_), k = whole(k_), weight = whole(weight_), rotations = whole(rotations_);
  std::array<Tensor, 3> r{like(q), like(q), like(q)};
  const On on(q);
  check(api.fbla_turn_fwd(ptr(q), ptr(k), ptr(weight), f32(rotations), ptr(r[0]), ptr(r[1]), ptr(r[2]), q.size(0), q.size(2), q.size(1),
                          q.size(3), code_of(q), on.stream), "fbla_turn_fwd");
  return r;
}

std::array<Tensor, 3> turn_bwd(const Tensor& k_, const Tensor& weight_, const Tensor& rotations_, const Tensor& dk_out, const Tensor& dq_rot,
                               const Tensor& dk_rot) {
  require_gpu({k_, weight_, rotations_, dk_out, dq_rot, dk_rot});
  const Tensor k = whole(k_), weight = whole(weight_), rotations = whole(rotations_);
  const std::array<Tensor, 3> g{whole(dk_out), whole(dq_rot), whole(dk_rot)};
  std::array<Tensor, 3> r{like(k), like(k), like(weight)};
  const On on(k);
  check(api.fbla_turn_bwd(ptr(k), ptr(weight), f32(rotations), ptr(g[0]), ptr(g[1]), ptr(g[2]), ptr(r[0]), ptr(r[1]), ptr(r[2]), k.size(0),
                          k.size(2), k.size(1), k.size(3), code_of(k), on.stream), "fbla_turn_bwd");
  return r;
}

// ---- blocks ---------------------------------------------------------------------------------------------------------------
// A vision block between its input and its output as one call a direction: what the block's Python steps do one by one, without
// a node of the autograd graph, a Python call and their checks between them.  Projections are `project`'s or torch's GEMMs (the rule
// below); the attention of 16-bit heads of 32 channels runs on the projections' rows (`on_rows`), other heads through the launches
// above.  The gradient of a tensor that two steps read is accumulated by the second step's GEMM instead of a launch of its own (12
// us at 200704 x 64 and 50176 x 256 in bf16).
Tensor flat(const Tensor& t) { return t.reshape({-1, t.size(-1)}); }
// Whether `project` takes products of these rows rather than torch's GEMM: 16-bit types within the entry point's limits
// (fbla_project refuses others), unless the product is large enough for the library's deeper pipeline to count.  A call of the library
// takes the host 17 us, one of ours 4 for up to three products, which small products do not hide.  GPU us of the library / here (bf16,
// with bias, captured graph).  A forward product by itself (`alone`) of whole 256-wide tiles, contractions of 128 and more, over 1.5e9
// multiply-adds and up to 2^24 results is the library's: 50176 x 128 -> 256 13.4 / 16.7, 12544 x 256 -> 512 11.7 / 13.6, 25088 x 256 ->
// 256 11.6 / 13.7, 50176 x 256 -> 256 16.4 / 20.9, x 512 -> 256 22.0 / 30.4, 12544 x 512 -> 512 15.7 / 18.7.  More results: 50176 x 256 ->
// 512 38.3 / 37.1, x 512 -> 512 62.0 / 58.9; fewer products: 8192 x 256 -> 512 8.3 / 8.8, 12544 x 256 -> 256 8.2 / 8.4, 4096 x 512 -> 512
// 9.4 / 8.1; other widths: 12544 x 320 -> 320 11.2 / 9.8, 50176 x 320 -> 640 47.9 / 48.8, 8192 x 640 -> 640 14.9 / 17.4.  Several in a launch,
// an added tensor or a second product pay up to 4e9 where both sides are 512 and more: three of 8192 x 640 -> 640 42.6 / 37.1, of 50176
// x 256 -> 512 109 / 87; one of 4096 x 1280 -> 1280 21.5 / 26.1.
bool projects(const Tensor& x, const Tensor& w, bool alone = false) {
  constexpr int64_t kMostChannels = 1 << 16, kMostWeights = 1 << 29, kLongestRow = 1 << 22;  // of fbla_project
  if (x.element_size() != 2 || w.size(0) > kMostChannels || w.size(1) > kMostChannels || w.numel() > kMostWeights ||
      (x.dim() > 1 && x.stride(-2) > kLongestRow))
    return false;
  const int64_t tokens = x.numel() / x.size(-1);
  const double work = (double)tokens * w.numel();
  if (alone && work > 1.5e9 && w.size(1) >= 128 && w.size(0) % 256 == 0 && tokens * w.size(0) <= 1 << 24) return false;
  return w.size(0) < 512 || w.size(1) < 512 || work <= 4e9;
}
// y = x W^T + b (+ add) for one or more projections
struct Linear {
  Tensor x, w, b, add;
};
std::vector<Tensor> linears(const std::vector<Linear>& p) {
  bool own = p.size() <= 3;
  const bool alone = p.size() == 1 && !p[0].add.defined();
  for (const Linear& l : p) own = own && projects(l.x, l.w, alone) && l.x.numel() / l.x.size(-1) == p[0].x.numel() / p[0].x.size(-1);
  std::vector<Tensor> r;
  if (own) {
    std::vector<Projection> jobs;
    for (const Linear& l : p) jobs.push_back({l.x, l.w, l.b, l.add, Tensor(), Tensor()});
    return project(jobs, false);
  }
  for (const Linear& l : p) {
    r.push_back(at::linear(l.x, l.w, l.b));
    if (l.add.defined()) r.back().add_(l.add);
  }
  return r;
}
std::pair<Tensor, Tensor> two_linears(const Linear& a, const Linear& b) {
  if (a.x.numel() != b.x.numel()) return {linears({a})[0], linears({b})[0]};
  const std::vector<Tensor> r = linears({a, b});
  return {r[0], r[1]};
}
Tensor linear(const Tensor& x, const Tensor& w, const Tensor& b) { return linears({{x, w, b, Tensor()}})[0]; }
// gradient of x in y = x W^T, of x in y = x W^T and y2 = x W2^T, plus `add`
Tensor input_grad(const Tensor& g, const Tensor& w, const Tensor& g2 = Tensor(), const Tensor& w2 = Tensor(), const Tensor& add = Tensor()) {
  if (projects(g, w) && (!g2.defined() || projects(g2, w2))) return project({{g, w, Tensor(), add, g2, w2}}, true)[0];
  std::vector<int64_t> shape = g.sizes().vec();
  shape.back() = w.size(1);
  Tensor r = add.defined() ? at::addmm(flat(add), flat(g), w) : at::mm(flat(g), w);
  if (g2.defined()) r.addmm_(flat(g2), w2);
  return r.view(shape);
}
// gradients of W and b; kernel: by the token-splitting kernel, else torch's GEMM and column sums
std::pair<Tensor, Tensor> weight_grad(const Tensor& g, const Tensor& x, bool weight, bool bias, bool kernel) {
  if (!weight && !bias) return {};
  if (kernel && weight) return linear_wgrad(g, x, bias);
  const Tensor rows_ = flat(g);
  return {weight ? at::mm(rows_.t(), flat(x)) : Tensor(), bias ? rows_.sum(0) : Tensor()};
}
// Large blocks give up what nothing reads any more before they allocate what comes next, as the steps one by one do (inference, peak
// without / with: LinFusion 32768 x 640 bf16 441 / 200 MB, FLatten 401408 x 256 with reduced keys 1622 / 935).  Rows of up to 64 MB do not:
// kernels that write where others have just read were 2 to 5 % slower there (captured forward, FLatten 64 x 28x28 x 64 with reduced keys
// bf16 109.6 / 114.2 us, 64 x 28x28 x 256 fp32 517 / 524), and the same from 98 MB on.
bool spares(const Tensor& x) { return x.nbytes() >= size_t(64) << 20; }
template <typename... T> void release(bool large, T&... t) {
  if (large) ((t = Tensor()), ...);
}
struct NoGraph {  // (called inside an autograd function or without gradients: nothing is recorded)
  at::AutoDispatchBelowADInplaceOrView guard;
};

// The attention between the projections' rows and the block's, where the kernels of fbla_rows.hip take it: 16-bit types, heads of
// 32 channels.  `rows` are the projections with queries (and keys) first in a row.
constexpr int kPolarity = 0, kRotary = 1;
bool on_rows(const Tensor& x, int64_t heads) {
  return x.element_size() == 2 && x.size(2) == 32 * heads && x.size(0) <= 65535 && x.size(1) <= 1 << 24 && heads <= 2048;
}
struct RowState {
  Tensor planes, km;
};
fbla_block_attn row_args(int kind, const Tensor& q, int64_t q_offset, const Tensor& k, int64_t k_offset, const Tensor& v, int64_t v_offset,
                         int64_t heads, const RowState& state) {
  fbla_block_attn a{};
  auto at = [](const Tensor& t, int64_t offset) { return static_cast<char*>(ptr(t)) + offset * t.element_size(); };
  a.kind = kind, a.dtype = code_of(q), a.B = q.size(0), a.N = q.size(1), a.Nk = k.size(1), a.heads = heads, a.eps = 1e-6f;
  a.q = at(q, q_offset), a.k = at(k, k_offset), a.v = at(v, v_offset);
  a.q_row = q.size(2), a.k_row = k.size(2), a.v_row = v.size(2);
  a.state_planes = ptr(state.planes), a.state_km = f32(state.km);
  return a;
}
RowState new_row_state(int kind, const Tensor& x, int64_t heads) {
  return {like(x, {(int64_t)api.fbla_block_attn_state_elements(kind, x.size(0), heads)}),
          like_f32(x, {x.size(0), heads, kind == kPolarity ? 72 : 40})};
}
Tensor row_workspace(const fbla_block_attn& a, const Tensor& x) {
  return scratch(api.fbla_block_attn_workspace_bytes(a.kind, a.B, a.N, a.Nk, a.heads), x);
}

// layers/mlla.py: qk projection, rotary features, decoupled attention, positional convolution of the input
std::vector<Tensor> mlla_fwd(const Tensor& x, const Tensor& w, const Tensor& b, const Tensor& conv_w, const Tensor& conv_b,
                             const Tensor& rotations, int64_t side, int64_t heads, bool trains) {
  const NoGraph none;
  const bool lean = !trains && spares(x);
  Tensor qk = linear(x, w, b);
  if (on_rows(x, heads)) {
    const Tensor local = dwconv_fwd(x, conv_w, conv_b, side, side, false), xs = whole(x), rot = whole(rotations), out = like(local);
    const RowState state = new_row_state(kRotary, x, heads);
    fbla_block_attn a = row_args(kRotary, qk, 0, qk, x.size(2), xs, 0, heads, state);
    const Tensor ws = row_workspace(a, x);
    a.local = ptr(local), a.rot = f32(rot), a.out = ptr(out), a.workspace = ptr(ws), a.workspace_bytes = ws.numel();
    const On on(x);
    check(api.fbla_block_attn_forward(&a, on.stream), "fbla_block_attn_forward");
    if (!trains) return {out};
    return {out, qk, state.planes, state.km};
  }
  auto [q, k, qr, kr, v] = rotary_fwd(qk, x, rotations, heads);
  release(lean, qk);
  const Attended a = la_fwd(q, k, v, qr, kr, 1.0 / x.size(1), 1e-6, FBLA_NORMALIZE | FBLA_DECOUPLED);
  release(lean, q, k, qr, kr, v);
  const Tensor local = dwconv_fwd(x, conv_w, conv_b, side, side, false);  // (last: the merge finds it in the caches)
  const Tensor out = merge_fwd(a.o, Tensor(), local, Tensor());
  if (!trains) return {out};
  return {out, qk, q, k, qr, kr, v, a.s, a.km};
}

// saved: what mlla_fwd returned after its output, or what saved-tensor hooks made of it (any strides).  need: x, w, b, conv_w, conv_b
std::vector<Tensor> mlla_bwd(const Tensor& g, const Tensor& x, const Tensor& w, const Tensor& conv_w, const Tensor& rotations,
                             const std::vector<Tensor>& saved, int64_t side, int64_t heads, const std::array<bool, 5>& need, bool kernel) {
  const NoGraph none;
  Tensor dx, dw, db, dconv_w, dconv_b;
  if (need[3] || need[4]) std::tie(dconv_w, dconv_b) = dwconv_grad(x, g, conv_w, side, side, need[4]);
  if (need[0] || need[1] || need[2]) {
    const Tensor qk = whole(saved.at(0)), dlocal = dwconv_fwd(g, conv_w, Tensor(), side, side, true);
    Tensor dqk;
    if (saved.size() == 3) {
      const Tensor xs = whole(x), gs = whole(g), rot = whole(rotations);
      dqk = like(qk), dx = like(gs);
      const int64_t C = x.size(2);
      fbla_block_attn a = row_args(kRotary, qk, 0, qk, C, xs, 0, heads, {whole(saved[1]), whole(saved[2])});
      const Tensor ws = row_workspace(a, x);
      a.rot = f32(rot), a.workspace = ptr(ws), a.workspace_bytes = ws.numel(), a.dout = ptr(gs), a.dv_more = ptr(dlocal);
      a.dq = ptr(dqk), a.dk = static_cast<char*>(ptr(dqk)) + C * dqk.element_size(), a.dv = ptr(dx);
      a.dq_row = a.dk_row = 2 * C, a.dv_row = C;
      const On on(x);
      check(api.fbla_block_attn_backward_queries(&a, on.stream), "fbla_block_attn_backward_queries");
      check(api.fbla_block_attn_backward_keys(&a, on.stream), "fbla_block_attn_backward_keys");
    } else {
      const Tensor q = saved.at(1), k = saved.at(2), qr = saved.at(3), kr = saved.at(4), v = saved.at(5);
      MergeGrads m = merge_bwd(g, heads, false, Tensor(), Tensor(), Tensor(), Tensor());
      const AttendedGrads d = la_bwd(q, k, v, qr, kr, m.o, saved.at(6), saved.at(7), 1.0 / x.size(1), 1e-6, FBLA_NORMALIZE | FBLA_DECOUPLED);
      release(spares(x), m.o);
      std::tie(dqk, dx) = rotary_bwd(qk, rotations, heads, d.q, d.k, d.q_rope, d.k_rope, d.v, dlocal);
    }
    std::tie(dw, db) = weight_grad(dqk, x, need[1], need[2], kernel);
    if (need[0]) dx = input_grad(dqk, w, Tensor(), Tensor(), dx);
  }
  return {need[0] ? dx : Tensor(), dw, db, dconv_w, dconv_b};
}

// What the two PVT-style blocks do with the values beside the attention: interpolated to the queries' number, convolved.
struct LocalValues {
  Tensor grid, local;  // the rows that are convolved (the values themselves, or interpolated), and the result
};
LocalValues local_values(const Tensor& v_rows, int64_t tokens, const Tensor& conv_w, const Tensor& conv_b, int64_t H, int64_t W) {
  const Tensor grid = v_rows.size(1) != tokens ? interpolate_fwd(v_rows, tokens) : v_rows;
  return {grid, dwconv_fwd(grid, conv_w, conv_b, H, W, false)};
}
Tensor local_values_grad(const Tensor& dlocal, int64_t n, const Tensor& conv_w, int64_t H, int64_t W) {
  const Tensor dgrid = dwconv_fwd(dlocal, conv_w, Tensor(), H, W, true);
  return n != dlocal.size(1) ? interpolate_bwd(dgrid, n) : dgrid;
}
// the input gradients of the query and key / value projections: one tensor where both read the same rows
std::pair<Tensor, Tensor> two_input_grads(const Tensor& dq, const Tensor& q_w, bool need_x, const Tensor& dkv, const Tensor& kv_w, bool same,
                                          bool need_src) {
  if (same) {
    return {need_x ? input_grad(dq, q_w, dkv, kv_w) : Tensor(), Tensor()};
  }
  return {need_x ? input_grad(dq, q_w) : Tensor(), need_src ? input_grad(dkv, kv_w) : Tensor()};
}

struct PolaWeights {  // in the order of the Python side
  Tensor q_w, q_b, kv_w, kv_b, pe, scale, power, conv_w, conv_b, proj_w, proj_b;
};
constexpr int kPola = 11;
PolaWeights pola_weights(const std::vector<Maybe>& p) {
  TORCH_CHECK(p.size() == kPola);
  return {given(p[0]), given(p[1]), given(p[2]), given(p[3]), given(p[4]), given(p[5]), given(p[6]), given(p[7]), given(p[8]), given(p[9]),
          given(p[10])};
}

// layers/polaformer.py up to the output projection.  src: the rows of the keys and values (x unless they were reduced)
std::vector<Tensor> pola_fwd(const Tensor& x, const Tensor& src, const std::vector<Maybe>& params, double alpha, int64_t H, int64_t W,
                             int64_t heads, bool trains) {
  const NoGraph none;
  const bool lean = !trains && spares(x);
  const PolaWeights p = pola_weights(params);
  const int64_t N = x.size(1), n = src.size(1), C = x.size(2);
  auto [qg, kv] = two_linears({x, p.q_w, p.q_b, Tensor()}, {src, p.kv_w, p.kv_b, Tensor()});
  LocalValues l;
  if (on_rows(x, heads)) {
    l = local_values(kv.narrow(2, C, C), N, p.conv_w, p.conv_b, H, W);
    const Tensor merged = like(l.local), pe = whole(p.pe), scale = whole(p.scale), power = whole(p.power);
    const RowState state = new_row_state(kPolarity, x, heads);
    fbla_block_attn a = row_args(kPolarity, qg, 0, kv, 0, kv, C, heads, state);
    const Tensor ws = row_workspace(a, x);
    a.local = ptr(l.local), a.gate = static_cast<char*>(ptr(qg)) + C * qg.element_size(), a.gate_row = 2 * C, a.out = ptr(merged);
    a.pe = ptr(pe), a.scale = ptr(scale), a.power = ptr(power), a.alpha = alpha, a.workspace = ptr(ws), a.workspace_bytes = ws.numel();
    {
      const On on(x);
      check(api.fbla_block_attn_forward(&a, on.stream), "fbla_block_attn_forward");
    }
    release(lean, qg, kv, l.grid, l.local);
    const Tensor y = linear(merged, p.proj_w, p.proj_b);
    if (!trains) return {y};
    return {y, qg, kv, l.grid, l.local, state.planes, state.km, merged};
  }
  const Tensor scale = at::softplus(p.scale), sigmoid = at::sigmoid(p.power), power = at::add(at::mul(sigmoid, alpha), 1);
  auto [q_same, q_opp, k, v] = polarity_fwd(qg, kv, p.pe, scale, power, heads);
  Tensor o1, o2, s, km, s2, km2, v1, v2;
  if (n == N && pair_supported(q_same, v)) {
    const Paired a = pair_fwd(q_same, q_opp, k, v, 1.0 / n, 1e-6);
    o1 = a.o1, o2 = a.o2, s = a.s, km = a.km;
  } else {
    const int64_t half = v.size(3) / 2;
    v1 = v.narrow(3, 0, half).contiguous(), v2 = v.narrow(3, half, half).contiguous();
    const Attended a = la_fwd(q_same, k, v1, Tensor(), Tensor(), 1.0 / n, 1e-6, FBLA_NORMALIZE);
    const Attended b = la_fwd(q_opp, k, v2, Tensor(), Tensor(), 1.0 / n, 1e-6, FBLA_NORMALIZE);
    o1 = a.o, s = a.s, km = a.km, o2 = b.o, s2 = b.s, km2 = b.km;
  }
  release(lean, q_same, q_opp, k, v, v1, v2);
  l = local_values(kv.narrow(2, C, C), N, p.conv_w, p.conv_b, H, W);  // (last: the merge finds it in the caches)
  const Tensor merged = merge_fwd(o1, o2, l.local, qg.narrow(2, C, C));
  release(lean, o1, o2, l.grid, l.local, qg, kv);
  const Tensor y = linear(merged, p.proj_w, p.proj_b);
  if (!trains) return {y};
  return {y, scale, sigmoid, power, qg, kv, q_same, q_opp, k, v, l.grid, l.local, o1, o2, s, km, s2,
          km2, v1, v2, merged};
}

// saved: what pola_fwd returned after its output.  need: x, src, the eleven parameters; kernel: of q, kv, proj
std::vector<Tensor> pola_bwd(const Tensor& g, const Tensor& x, const Tensor& src, bool same, const std::vector<Maybe>& params,
                             const std::vector<Maybe>& saved, double alpha, int64_t H, int64_t W, int64_t heads,
                             const std::array<bool, 2 + kPola>& need, const std::array<bool, 3>& kernel) {
  const NoGraph none;
  const PolaWeights p = pola_weights(params);
  auto at_ = [&](int i) { return given(saved.at(i)); };
  const bool rows_ = saved.size() == 7;
  TORCH_CHECK(rows_ || saved.size() == 20);
  const Tensor qg = whole(at_(rows_ ? 0 : 3)), kv = whole(at_(rows_ ? 1 : 4)), merged = at_(rows_ ? 6 : 19);
  const int64_t n = src.size(1), C = x.size(2);
  std::vector<Tensor> r(2 + kPola);
  std::tie(r[11], r[12]) = weight_grad(g, merged, need[11], need[12], kernel[2]);
  if (std::none_of(need.begin(), need.begin() + 11, [](bool b) { return b; })) return r;
  Tensor dmerged = input_grad(g, p.proj_w);
  std::array<Tensor, 5> d;  // of qg, kv, pe, scale, power
  if (rows_) {
    const Tensor grid = at_(2), local = whole(at_(3)), pe = whole(p.pe), scale = whole(p.scale), power = whole(p.power), dlocal = like(dmerged);
    d = {like(qg), like(kv), like(pe), like(scale), like(power)};
    fbla_block_attn a = row_args(kPolarity, qg, 0, kv, 0, kv, C, heads, {whole(at_(4)), whole(at_(5))});
    const Tensor ws = row_workspace(a, x);
    auto half = [&](const Tensor& t) { return static_cast<char*>(ptr(t)) + C * t.element_size(); };
    a.local = ptr(local), a.gate = half(qg), a.gate_row = 2 * C, a.dout = ptr(dmerged), a.pe = ptr(pe), a.scale = ptr(scale);
    a.power = ptr(power), a.alpha = alpha, a.workspace = ptr(ws), a.workspace_bytes = ws.numel(), a.dq = ptr(d[0]), a.dgate = half(d[0]), a.dlocal = ptr(dlocal);
    a.dk = ptr(d[1]), a.dv = half(d[1]), a.dq_row = a.dgate_row = a.dk_row = a.dv_row = 2 * C;
    a.dpe = ptr(d[2]), a.dscale = ptr(d[3]), a.dpower = ptr(d[4]);
    {
      const On on(x);
      check(api.fbla_block_attn_backward_queries(&a, on.stream), "fbla_block_attn_backward_queries");
    }
    if (need[9] || need[10]) std::tie(r[9], r[10]) = dwconv_grad(grid, dlocal, p.conv_w, H, W, need[10]);
    if (std::none_of(need.begin(), need.begin() + 9, [](bool b) { return b; })) return r;
    const Tensor dv_rows = local_values_grad(dlocal, n, p.conv_w, H, W);
    a.dv_more = ptr(dv_rows);
    const On on(x);
    check(api.fbla_block_attn_backward_keys(&a, on.stream), "fbla_block_attn_backward_keys");
  } else {
    const Tensor scale = at_(0), power = at_(2), q_same = at_(5), q_opp = at_(6), k = at_(7), v = at_(8), grid = at_(9), s = at_(13),
                 km = at_(14), s2 = at_(15);
    MergeGrads m = merge_bwd(dmerged, heads, true, at_(11), at_(12), at_(10), qg.narrow(2, C, C));
    release(spares(x), dmerged);
    if (need[9] || need[10]) std::tie(r[9], r[10]) = dwconv_grad(grid, m.local, p.conv_w, H, W, need[10]);
    if (std::none_of(need.begin(), need.begin() + 9, [](bool b) { return b; })) return r;
    const Tensor dv_rows = local_values_grad(m.local, n, p.conv_w, H, W);
    release(spares(x), m.local);
    PairedGrads pd;
    if (!s2.defined()) {
      pd = pair_bwd(q_same, q_opp, k, v, m.o, m.o2, s, km, 1.0 / n, 1e-6);
    } else {
      const AttendedGrads a = la_bwd(q_same, k, at_(17), Tensor(), Tensor(), m.o, s, km, 1.0 / n, 1e-6, FBLA_NORMALIZE);
      const AttendedGrads b = la_bwd(q_opp, k, at_(18), Tensor(), Tensor(), m.o2, s2, at_(16), 1.0 / n, 1e-6, FBLA_NORMALIZE);
      pd = {a.q, b.q, at::add(a.k, b.k), at::cat({a.v, b.v}, -1)};
    }
    release(spares(x), m.o, m.o2);
    d = polarity_bwd(qg, kv, p.pe, scale, power, heads, pd.q1, pd.q2, pd.k, pd.v, dv_rows, m.gate);
  }
  std::tie(r[0], r[1]) = two_input_grads(d[0], p.q_w, need[0], d[1], p.kv_w, same, need[1]);
  std::tie(r[2], r[3]) = weight_grad(d[0], x, need[2], need[3], kernel[0]);
  std::tie(r[4], r[5]) = weight_grad(d[1], src, need[4], need[5], kernel[1]);
  if (need[6]) r[6] = d[2];
  if (need[7]) r[7] = rows_ ? d[3] : at::softplus_backward(d[3], p.scale, 1, 20);
  if (need[8]) r[8] = rows_ ? d[4] : at::sigmoid_backward(at::mul(d[4], alpha), at_(1));
  return r;
}

struct FocusedWeights {
  Tensor q_w, q_b, kv_w, kv_b, pe, scale, conv_w, conv_b, proj_w, proj_b;
};
constexpr int kFocused = 10;
FocusedWeights focused_weights(const std::vector<Maybe>& p) {
  TORCH_CHECK(p.size() == kFocused);
  return {given(p[0]), given(p[1]), given(p[2]), given(p[3]), given(p[4]), given(p[5]), given(p[6]), given(p[7]), given(p[8]), given(p[9])};
}

// layers/focused_la.py up to the output projection, as above
std::vector<Tensor> focused_fwd(const Tensor& x, const Tensor& src, const std::vector<Maybe>& params, int64_t H, int64_t W, int64_t heads,
                                bool trains) {
  const NoGraph none;
  const bool lean = !trains && spares(x);
  const FocusedWeights p = focused_weights(params);
  const int64_t N = x.size(1), n = src.size(1), C = x.size(2);
  auto [q_rows, kv] = two_linears({x, p.q_w, p.q_b, Tensor()}, {src, p.kv_w, p.kv_b, Tensor()});
  const Tensor scale = at::softplus(p.scale);
  auto [q, k, v] = focus_fwd(q_rows, kv, p.pe, scale, heads);
  release(lean, q_rows);
  Attended a = la_fwd(q, k, v, Tensor(), Tensor(), 1.0 / n, 1e-6, FBLA_NORMALIZE);
  release(lean, q, k, v);
  LocalValues l = local_values(kv.narrow(2, C, C), N, p.conv_w, p.conv_b, H, W);
  const Tensor merged = merge_fwd(a.o, Tensor(), l.local, Tensor());
  release(lean, a.o, l.local);
  const Tensor y = linear(merged, p.proj_w, p.proj_b);
  if (!trains) return {y};
  return {y, scale, q_rows, kv, q, k, v, l.grid, a.s, a.km, merged};
}

std::vector<Tensor> focused_bwd(const Tensor& g, const Tensor& x, const Tensor& src, bool same, const std::vector<Maybe>& params,
                                const std::vector<Maybe>& saved, int64_t H, int64_t W, int64_t heads,
                                const std::array<bool, 2 + kFocused>& need, const std::array<bool, 3>& kernel) {
  const NoGraph none;
  const FocusedWeights p = focused_weights(params);
  TORCH_CHECK(saved.size() == 10);
  auto at_ = [&](int i) { return given(saved[i]); };
  const Tensor scale = at_(0), q_rows = at_(1), kv = at_(2), q = at_(3), k = at_(4), v = at_(5), grid = at_(6), s = at_(7), km = at_(8),
               merged = at_(9);
  const int64_t n = src.size(1);
  std::vector<Tensor> r(2 + kFocused);
  std::tie(r[10], r[11]) = weight_grad(g, merged, need[10], need[11], kernel[2]);
  if (std::none_of(need.begin(), need.begin() + 10, [](bool b) { return b; })) return r;
  MergeGrads m = merge_bwd(input_grad(g, p.proj_w), heads, false, Tensor(), Tensor(), Tensor(), Tensor());
  if (need[8] || need[9]) std::tie(r[8], r[9]) = dwconv_grad(grid, m.local, p.conv_w, H, W, need[9]);
  if (std::none_of(need.begin(), need.begin() + 8, [](bool b) { return b; })) return r;
  const Tensor dv_rows = local_values_grad(m.local, n, p.conv_w, H, W);
  release(spares(x), m.local);
  AttendedGrads d = la_bwd(q, k, v, Tensor(), Tensor(), m.o, s, km, 1.0 / n, 1e-6, FBLA_NORMALIZE);
  release(spares(x), m.o);
  const auto [dq, dkv, dpe, dscale] = focus_bwd(q_rows, kv, p.pe, scale, heads, d.q, d.k, d.v, dv_rows);
  release(spares(x), d.q, d.k, d.v);
  std::tie(r[0], r[1]) = two_input_grads(dq, p.q_w, need[0], dkv, p.kv_w, same, need[1]);
  std::tie(r[2], r[3]) = weight_grad(dq, x, need[2], need[3], kernel[0]);
  std::tie(r[4], r[5]) = weight_grad(dkv, src, need[4], need[5], kernel[1]);
  if (need[6]) r[6] = dpe;
  if (need[7]) r[7] = at::softplus_backward(dscale, p.scale, 1, 20);
  return r;
}

// layers/linfusion.py on heads of 64 (the feature map inside the operator's kernels): residual projections of queries and
// keys (Linear, LayerNorm, LeakyReLU, Linear), projections, packed attention, output projection
struct LinFusionWeights {
  struct Path { Tensor in_w, in_b, norm_w, norm_b, out_w, out_b; } path[2];
  Tensor w[3], b[3], proj_w, proj_b;
};
constexpr int kLinFusion = 20;
LinFusionWeights linfusion_weights(const std::vector<Maybe>& p) {
  TORCH_CHECK(p.size() == kLinFusion);
  LinFusionWeights r;
  for (int i = 0; i < 2; ++i)
    r.path[i] = {given(p[6 * i]), given(p[6 * i + 1]), given(p[6 * i + 2]), given(p[6 * i + 3]), given(p[6 * i + 4]), given(p[6 * i + 5])};
  for (int i = 0; i < 3; ++i) r.w[i] = given(p[12 + 2 * i]), r.b[i] = given(p[13 + 2 * i]);
  r.proj_w = given(p[18]), r.proj_b = given(p[19]);
  return r;
}

std::vector<Tensor> linfusion_fwd(const Tensor& x, const Tensor& cu, const std::vector<Maybe>& params, const std::array<double, 2>& eps,
                                  const std::array<double, 2>& slope, int64_t heads, bool trains) {
  const NoGraph none;
  const bool lean = !trains && spares(x);
  const LinFusionWeights p = linfusion_weights(params);
  const int64_t B = x.size(0), N = x.size(1);
  const auto &pq = p.path[0], &pk = p.path[1];
  auto first = linears({{x, pq.in_w, pq.in_b, Tensor()}, {x, pk.in_w, pk.in_b, Tensor()}, {x, p.w[2], p.b[2], Tensor()}});
  std::vector<Normed> normed;
  {
    const Norm norms[2] = {{first[0], pq.norm_w, pq.norm_b, eps[0], slope[0]}, {first[1], pk.norm_w, pk.norm_b, eps[1], slope[1]}};
    if (first[0].sizes() == first[1].sizes()) {
      normed = norm_leaky({norms[0], norms[1]}, trains);
    } else {
      for (const Norm& n : norms) normed.push_back(norm_leaky({n}, trains)[0]);
    }
  }
  release(lean, first[0], first[1]);
  auto in = linears({{normed[0].y, pq.out_w, pq.out_b, x}, {normed[1].y, pk.out_w, pk.out_b, x}});
  release(lean, normed[0].y, normed[1].y);
  Tensor packed[3];
  {
    const auto qk = linears({{in[0], p.w[0], p.b[0], Tensor()}, {in[1], p.w[1], p.b[1], Tensor()}});
    for (int i = 0; i < 3; ++i) packed[i] = (i < 2 ? qk[i] : first[2]).view({B * N, heads, -1});
  }
  release(lean, in[0], in[1], first[2]);
  const Attended a = varlen_fwd(packed[0], packed[1], packed[2], cu, N, std::nullopt, 1e-4, FBLA_ELU1_QK);
  release(lean, packed[0], packed[1], packed[2]);
  const Tensor o = a.o.view({B, N, -1});
  std::vector<Tensor> r{linear(o, p.proj_w, p.proj_b)};
  if (!trains) return r;
  for (int i = 0; i < 2; ++i) r.insert(r.end(), {first[i], normed[i].mean, normed[i].rstd, normed[i].y, in[i]});
  r.insert(r.end(), {packed[0], packed[1], packed[2], a.s, a.km, o});
  return r;
}

std::vector<Tensor> linfusion_bwd(const Tensor& g, const Tensor& x, const Tensor& cu, const std::vector<Maybe>& params,
                                  const std::vector<Maybe>& saved, const std::array<double, 2>& slope,
                                  const std::array<bool, 1 + kLinFusion>& need, const std::array<bool, 8>& kernel) {
  const NoGraph none;
  const LinFusionWeights p = linfusion_weights(params);
  TORCH_CHECK(saved.size() == 16);
  auto at_ = [&](int i) { return given(saved[i]); };
  const int64_t N = x.size(1);
  std::vector<Tensor> r(1 + kLinFusion);
  std::tie(r[19], r[20]) = weight_grad(g, at_(15), need[19], need[20], kernel[7]);
  if (std::none_of(need.begin(), need.begin() + 19, [](bool b) { return b; })) return r;
  const Tensor qp = at_(10), kp = at_(11), vp = at_(12);
  const auto [dq, dk, dv] = varlen_bwd(qp, kp, vp, cu, N, input_grad(g, p.proj_w).view(vp.sizes()), at_(13), at_(14), std::nullopt, 1e-4,
                                       FBLA_ELU1_QK | FBLA_ELU1_GRAD);
  const Tensor d[3] = {flat(dq.view({-1, p.w[0].size(0)})), flat(dk.view({-1, p.w[1].size(0)})), flat(dv.view({-1, p.w[2].size(0)}))};
  std::tie(r[17], r[18]) = weight_grad(d[2], x, need[17], need[18], kernel[6]);
  Tensor dx = need[0] ? input_grad(d[2], p.w[2]) : Tensor();
  for (int i = 0; i < 2; ++i) {
    const auto& path = p.path[i];
    const Tensor hidden = whole(at_(5 * i)), mean = whole(at_(5 * i + 1)), rstd = whole(at_(5 * i + 2)), normed = at_(5 * i + 3),
                 in = at_(5 * i + 4);
    const int at0 = 1 + 6 * i;
    std::tie(r[13 + 2 * i], r[14 + 2 * i]) = weight_grad(d[i], in, need[13 + 2 * i], need[14 + 2 * i], kernel[4 + i]);
    const Tensor din = input_grad(d[i], p.w[i]);  // of x + residual
    std::tie(r[at0 + 4], r[at0 + 5]) = weight_grad(din, normed, need[at0 + 4], need[at0 + 5], kernel[2 * i + 1]);
    const Tensor dnormed = at::leaky_relu_backward(input_grad(din, path.out_w), flat(normed), slope[i], true);
    Tensor dhidden;
    std::tie(dhidden, r[at0 + 2], r[at0 + 3]) =
        at::native_layer_norm_backward(dnormed.view(hidden.sizes()), hidden, {hidden.size(-1)}, mean, rstd, path.norm_w, path.norm_b,
                                       {true, need[at0 + 2], need[at0 + 3]});
    std::tie(r[at0], r[at0 + 1]) = weight_grad(dhidden, x, need[at0], need[at0 + 1], kernel[2 * i]);
    if (need[0]) dx = input_grad(flat(dhidden), path.in_w, Tensor(), Tensor(), dx.add_(din));
  }
  if (need[0]) r[0] = dx.view(x.sizes());
  return r;
}

// None for a tensor that does not exist
Maybe out(const Tensor& t) { return t.defined() ? Maybe(t) : std::nullopt; }
template <typename... T> auto outs(const T&... t) { return std::make_tuple(out(t)...); }
template <size_t N> auto outs(const std::array<Tensor, N>& t) {
  return std::apply([](const auto&... e) { return std::make_tuple(out(e)...); }, t);
}
std::vector<Maybe> listed(const std::vector<Tensor>& t) {
  std::vector<Maybe> r;
  for (const Tensor& e : t) r.push_back(out(e));
  return r;
}

// ---- checks ---------------------------------------------------------------------------------------------------------------
const Tensor* tensor_of(py::handle h) { return THPVariable_Check(h.ptr()) ? &THPVariable_Unpack(h.ptr()) : nullptr; }

// Whether check_dense (ops/_check.py) has nothing to say about the operands; what is wrong with them is its to say.
bool dense_operands(py::handle q_, py::handle k_, py::handle v_, py::handle qr_, py::handle kr_) {
  const Tensor *q = tensor_of(q_), *k = tensor_of(k_), *v = tensor_of(v_);
  if (!q || !k || !v || q->dim() != 4 || k->dim() != 4 || v->dim() != 4 || !q->is_cuda()) return false;
  auto type = q->scalar_type();
  if (type != at::kHalf && type != at::kBFloat16 && type != at::kFloat) return false;
  for (const Tensor* t : {k, v})
    if (t->device() != q->device() || t->scalar_type() != type) return false;
  if (!qr_.is_none()) {
    const Tensor *qr = tensor_of(qr_), *kr = tensor_of(kr_);
    if (!qr || !kr || qr->sizes() != q->sizes() || kr->sizes() != k->sizes()) return false;
    for (const Tensor* t : {qr, kr})
      if (t->device() != q->device() || t->scalar_type() != type) return false;
  }
  return q->size(0) == k->size(0) && q->size(1) == k->size(1) && q->size(3) == k->size(3) && k->size(0) == v->size(0) &&
         k->size(1) == v->size(1) && k->size(2) == v->size(2) && q->size(3) > 0 && q->size(3) <= 128 && v->size(3) > 0 && v->size(3) <= 128;
}

// Whether these (tensors or None) are ordinary GPU tensors (`plain` types: Tensor and Parameter) of x's supported type on its
// device, none of them empty or of 2^31 elements.
bool plain_gpu_tensors(py::handle x_, py::args rest, PyObject* parameter) {
  const Tensor* x = tensor_of(x_);
  auto ordinary = [&](py::handle h) {
    return reinterpret_cast<PyObject*>(Py_TYPE(h.ptr())) == THPVariableClass || reinterpret_cast<PyObject*>(Py_TYPE(h.ptr())) == parameter;
  };
  if (!x || !ordinary(x_) || !x->is_cuda()) return false;
  const auto type = x->scalar_type();
  if (type != at::kHalf && type != at::kBFloat16 && type != at::kFloat) return false;
  auto fits = [&](const Tensor& t) {
    return t.scalar_type() == type && t.device() == x->device() && t.numel() > 0 && t.numel() < int64_t(1) << 31 && t.layout() == at::kStrided;
  };
  if (!fits(*x)) return false;
  for (py::handle h : rest) {
    if (h.is_none()) continue;
    const Tensor* t = tensor_of(h);
    if (!t || !ordinary(h) || !fits(*t)) return false;
  }
  return true;
}

// ---- which blocks run whole -----------------------------------------------------------------------------------------------
// Whether the modules are what `untouched` (ops/_check.py) asks for, given as pairs of module and class.
bool untouched_modules(const std::vector<std::pair<py::handle, py::handle>>& modules) {
  static const char* const hooks[] = {"_forward_hooks", "_forward_pre_hooks", "_backward_hooks", "_backward_pre_hooks"};
  for (const auto& [module, kind] : modules) {
    if (reinterpret_cast<PyObject*>(Py_TYPE(module.ptr())) != kind.ptr()) return false;
    const py::object dict = py::reinterpret_steal<py::object>(PyObject_GenericGetDict(module.ptr(), nullptr));
    if (!dict) throw py::error_already_set();
    for (const char* name : hooks) {
      PyObject* set = PyDict_GetItemString(dict.ptr(), name);
      if (!set || PyObject_IsTrue(set) != 0) return false;
    }
    if (PyDict_GetItemString(dict.ptr(), "forward")) return false;
    PyObject* compiled = PyDict_GetItemString(dict.ptr(), "_compiled_call_impl");
    if (compiled && compiled != Py_None) return false;
  }
  return true;
}

bool shaped(const Tensor& t, at::IntArrayRef shape) { return t.sizes() == shape; }
bool shaped_or_none(const Tensor& t, at::IntArrayRef shape) { return !t.defined() || t.sizes() == shape; }
bool linear_shapes(const Tensor& w, const Tensor& b, int64_t M, int64_t N, int64_t piece) {
  return w.defined() && shaped(w, {M, N}) && shaped_or_none(b, {M}) && M % piece == 0 && N % piece == 0;
}
bool conv_shapes(const Tensor& w, const Tensor& b, int64_t Cw, int64_t C) {
  return w.defined() && w.dim() == 4 && w.size(0) == Cw && C % Cw == 0 && w.size(1) == 1 && w.size(2) == w.size(3) &&
         (w.size(2) == 3 || w.size(2) == 5 || w.size(2) == 7) && shaped_or_none(b, {Cw});
}

// the shapes that the steps of a block take one by one (layers/_features.py, ops/depthwise.py, ops/projection.py)
bool mlla_fits(const Tensor& x, const std::vector<Maybe>& p, const Tensor& rotations, int64_t side, int64_t heads) {
  const Tensor w = given(p[0]), b = given(p[1]), conv_w = given(p[2]), conv_b = given(p[3]);
  if (x.dim() != 3 || heads < 1) return false;
  const int64_t C = x.size(2), piece = 16 / x.element_size();
  return x.size(1) == side * side && C % heads == 0 && C / heads % piece == 0 && C / heads <= 128 && linear_shapes(w, b, 2 * C, C, piece) &&
         conv_shapes(conv_w, conv_b, C, C) && rotations.scalar_type() == at::kFloat && rotations.device() == x.device() &&
         !rotations.requires_grad() && shaped(rotations, {side, side, C / 2, 2}) && 2 * x.numel() < int64_t(1) << 31;
}

bool pvt_fits(const Tensor& x, const Tensor& src, const Tensor& kv_w, const Tensor& kv_b, const Tensor& pe, const Tensor& scale,
              const Tensor& conv_w, const Tensor& conv_b, const Tensor& proj_w, const Tensor& proj_b, int64_t H, int64_t W, int64_t heads,
              int64_t unit) {
  if (x.dim() != 3 || src.dim() != 3 || heads < 1 || !proj_w.defined() || proj_w.dim() != 2) return false;
  const int64_t C = x.size(2), n = src.size(1), piece = 16 / x.element_size();
  return H > 0 && x.size(1) == H * W && C % heads == 0 && C / heads % (unit * piece) == 0 && shaped(src, {x.size(0), n, C}) &&
         linear_shapes(kv_w, kv_b, 2 * C, C, piece) && shaped(pe, {1, n, C}) && shaped(scale, {1, 1, C}) &&
         conv_shapes(conv_w, conv_b, C / heads, C) && linear_shapes(proj_w, proj_b, proj_w.size(0), C, piece) &&
         n * x.size(1) < 1 << 28 && 2 * x.numel() < int64_t(1) << 31;
}
bool pola_fits(const Tensor& x, const Tensor& src, const std::vector<Maybe>& params, int64_t H, int64_t W, int64_t heads) {
  const PolaWeights p = pola_weights(params);
  if (!pvt_fits(x, src, p.kv_w, p.kv_b, p.pe, p.scale, p.conv_w, p.conv_b, p.proj_w, p.proj_b, H, W, heads, 2)) return false;
  const int64_t C = x.size(2);
  return C / heads <= 64 && linear_shapes(p.q_w, p.q_b, 2 * C, C, 16 / x.element_size()) && shaped(p.power, {1, heads, 1, C / heads});
}
bool focused_fits(const Tensor& x, const Tensor& src, const std::vector<Maybe>& params, int64_t H, int64_t W, int64_t heads) {
  const FocusedWeights p = focused_weights(params);
  if (!pvt_fits(x, src, p.kv_w, p.kv_b, p.pe, p.scale, p.conv_w, p.conv_b, p.proj_w, p.proj_b, H, W, heads, 1)) return false;
  const int64_t C = x.size(2);
  return C / heads <= 128 && C * x.element_size() <= 4096 && linear_shapes(p.q_w, p.q_b, C, C, 16 / x.element_size());
}
bool linfusion_fits(const Tensor& x, const std::vector<Maybe>& params, int64_t heads) {
  const LinFusionWeights p = linfusion_weights(params);
  if (x.dim() != 3 || x.element_size() != 2 || !p.proj_w.defined() || p.proj_w.dim() != 2) return false;
  const int64_t C = x.size(2), inner = 64 * heads;
  for (const auto& path : p.path) {
    if (!path.in_w.defined() || path.in_w.dim() != 2) return false;
    const int64_t width = path.in_w.size(0);
    if (width > 2048 || !linear_shapes(path.in_w, path.in_b, width, C, 8) || !shaped_or_none(path.norm_w, {width}) || !shaped_or_none(path.norm_b, {width}) ||
        !linear_shapes(path.out_w, path.out_b, C, width, 8))
      return false;
  }
  for (int i = 0; i < 3; ++i)
    if (!linear_shapes(p.w[i], p.b[i], inner, C, 8)) return false;
  return linear_shapes(p.proj_w, p.proj_b, p.proj_w.size(0), inner, 8);
}

}  // namespace

PYBIND11_MODULE(fbla_torch, m) {
  // what torch's own calls raise stays what it is (out of memory, tensors without storage)
  py::register_local_exception_translator([](std::exception_ptr p) {
    try {
      if (p) std::rethrow_exception(p);
    } catch (const c10::Error&) {
      torch::translate_exception_to_python(p);
    }
  });
  m.def("load", &load);
  // Without the interpreter's lock: a launch waits where the queue is full, an allocation where it frees memory, and other Python
  // threads (those that drive other GPUs among them) run meanwhile.
  auto op = [&m](const char* name, auto f, const auto&... more) { m.def(name, f, py::call_guard<py::gil_scoped_release>(), more...); };
  op("la_fwd", [](const Tensor& q, const Tensor& k, const Tensor& v, const Maybe& qr, const Maybe& kr, double scale, double eps,
                     int flags) {
    const Attended r = la_fwd(q, k, v, given(qr), given(kr), scale, eps, flags);
    return outs(r.o, r.s, r.km);
  });
  op("la_bwd", [](const Tensor& q, const Tensor& k, const Tensor& v, const Maybe& qr, const Maybe& kr, const Tensor& g, const Tensor& s,
                     const Maybe& km, double scale, double eps, int flags) {
    const AttendedGrads d = la_bwd(q, k, v, given(qr), given(kr), g, s, given(km), scale, eps, flags);
    return outs(d.q, d.k, d.v, d.q_rope, d.k_rope);
  });
  m.def("pair_supported", &pair_supported);
  op("pair_fwd", [](const Tensor& q1, const Tensor& q2, const Tensor& k, const Tensor& v, double scale, double eps) {
    const Paired r = pair_fwd(q1, q2, k, v, scale, eps);
    return outs(r.o1, r.o2, r.s, r.km);
  });
  op("pair_bwd", [](const Tensor& q1, const Tensor& q2, const Tensor& k, const Tensor& v, const Tensor& g1, const Tensor& g2,
                       const Tensor& s, const Tensor& km, double scale, double eps) {
    const PairedGrads d = pair_bwd(q1, q2, k, v, g1, g2, s, km, scale, eps);
    return outs(d.q1, d.q2, d.k, d.v);
  });
  op("varlen_fwd", [](const Tensor& q, const Tensor& k, const Tensor& v, const Tensor& cu, int64_t longest, std::optional<double> scale,
                         double eps, int extra) {
    const Attended r = varlen_fwd(q, k, v, cu, longest, scale, eps, extra);
    return outs(r.o, r.s, r.km);
  }, py::arg("q"), py::arg("k"), py::arg("v"), py::arg("cu_seqlens"), py::arg("max_seqlen"), py::arg("scale"), py::arg("eps"),
        py::arg("extra_flags") = 0);
  op("varlen_bwd", &varlen_bwd, py::arg("q"), py::arg("k"), py::arg("v"), py::arg("cu_seqlens"), py::arg("max_seqlen"), py::arg("do"),
        py::arg("s"), py::arg("km"), py::arg("scale"), py::arg("eps"), py::arg("extra_flags") = 0);
  op("chunk_reduce", [](const Tensor& q, const Tensor& k, const Tensor& v, int64_t chunk, bool with_norm, double p_norm) {
    const Statistics r = chunk_reduce(q, k, v, chunk, with_norm, p_norm);
    return outs(r.qc, r.kc, r.vc, r.h, r.h_norm);
  }, py::arg("q"), py::arg("k"), py::arg("v"), py::arg("chunk"), py::arg("with_norm") = false, py::arg("p_norm") = 2.0);
  op("select_blocks", [](const Tensor& qc, const Tensor& kc, const Maybe& bias, int64_t top_k, double scale) {
    return select_blocks(qc, kc, given(bias), top_k, scale);
  });
  m.def("piecewise_supported", &piecewise_supported);
  op("piecewise_fwd", &piecewise_fwd);
  op("elu1_fwd", [](const Tensor& x0, const Maybe& x1) -> std::variant<Tensor, std::pair<Tensor, Tensor>> {
    const auto y = elu1_fwd(x0, given(x1));
    if (x1) return y;
    return y.first;
  }, py::arg("x0"), py::arg("x1") = py::none());
  op("elu1_bwd", &elu1_bwd);
  op("dwconv_fwd", [](const Tensor& x, const Tensor& w, const Maybe& bias, int64_t H, int64_t W, bool flip) {
    return dwconv_fwd(x, w, given(bias), H, W, flip);
  }, py::arg("x"), py::arg("w"), py::arg("bias"), py::arg("H"), py::arg("W"), py::arg("flip") = false);
  op("dwconv_grad", [](const Tensor& x, const Tensor& g, const Tensor& w, int64_t H, int64_t W, bool with_bias) {
    const auto r = dwconv_grad(x, g, w, H, W, with_bias);
    return outs(r.first, r.second);
  });
  op("linear_wgrad", [](const Tensor& g, const Tensor& x, bool with_bias) {
    const auto r = linear_wgrad(g, x, with_bias);
    return outs(r.first, r.second);
  });
  op("project", [](const std::vector<std::array<Maybe, 6>>& p, bool rows_of_w) {
    std::vector<Projection> jobs;
    for (const auto& t : p) jobs.push_back({given(t[0]), given(t[1]), given(t[2]), given(t[3]), given(t[4]), given(t[5])});
    return project(jobs, rows_of_w);
  });
  op("norm_leaky", [](const std::vector<std::tuple<Tensor, Maybe, Maybe, double, double>>& p, bool with_stats) {
    std::vector<Norm> jobs;
    for (const auto& [x, w, b, eps, slope] : p) jobs.push_back({x, given(w), given(b), eps, slope});
    std::vector<std::tuple<Maybe, Maybe, Maybe>> r;
    for (const Normed& n : norm_leaky(jobs, with_stats)) r.push_back(outs(n.y, n.mean, n.rstd));
    return r;
  });
  op("polarity_fwd", [](const Tensor& qg, const Tensor& kv, const Tensor& pe, const Tensor& scale, const Tensor& power, int64_t heads) {
    return outs(polarity_fwd(qg, kv, pe, scale, power, heads));
  });
  op("polarity_bwd", [](const Tensor& qg, const Tensor& kv, const Tensor& pe, const Tensor& scale, const Tensor& power, int64_t heads,
                           const Tensor& a, const Tensor& b, const Tensor& c, const Tensor& d, const Tensor& e, const Tensor& f) {
    return outs(polarity_bwd(qg, kv, pe, scale, power, heads, a, b, c, d, e, f));
  });
  op("rotary_fwd", [](const Tensor& qk, const Tensor& x, const Tensor& rotations, int64_t heads) {
    return outs(rotary_fwd(qk, x, rotations, heads));
  });
  op("rotary_bwd", [](const Tensor& qk, const Tensor& rotations, int64_t heads, const Tensor& a, const Tensor& b, const Tensor& c,
                         const Tensor& d, const Tensor& e, const Tensor& f) {
    const auto r = rotary_bwd(qk, rotations, heads, a, b, c, d, e, f);
    return outs(r.first, r.second);
  });
  op("merge_fwd", [](const Tensor& o, const Maybe& o2, const Tensor& local, const Maybe& gate) {
    return merge_fwd(o, given(o2), local, given(gate));
  });
  op("merge_bwd", [](const Tensor& dout, int64_t heads, bool halves, const Maybe& o, const Maybe& o2, const Maybe& local,
                        const Maybe& gate) {
    const MergeGrads r = merge_bwd(dout, heads, halves, given(o), given(o2), given(local), given(gate));
    return outs(r.o, r.o2, r.local, r.gate);
  });
  op("interpolate_fwd", &interpolate_fwd);
  op("interpolate_bwd", &interpolate_bwd);
  op("focus_fwd", [](const Tensor& q, const Tensor& kv, const Tensor& pe, const Tensor& scale, int64_t heads) {
    return outs(focus_fwd(q, kv, pe, scale, heads));
  });
  op("focus_bwd", [](const Tensor& q, const Tensor& kv, const Tensor& pe, const Tensor& scale, int64_t heads, const Tensor& a,
                        const Tensor& b, const Tensor& c, const Tensor& d) { return outs(focus_bwd(q, kv, pe, scale, heads, a, b, c, d)); });
  op("turn_fwd", [](const Tensor& q, const Tensor& k, const Tensor& weight, const Tensor& rotations) {
    return outs(turn_fwd(q, k, weight, rotations));
  });
  op("turn_bwd", [](const Tensor& k, const Tensor& weight, const Tensor& rotations, const Tensor& a, const Tensor& b, const Tensor& c) {
    return outs(turn_bwd(k, weight, rotations, a, b, c));
  });

  op("mlla_fwd", [](const Tensor& x, const std::vector<Maybe>& p, const Tensor& rotations, int64_t side, int64_t heads, bool trains) {
    return listed(mlla_fwd(x, given(p[0]), given(p[1]), given(p[2]), given(p[3]), rotations, side, heads, trains));
  });
  op("mlla_bwd", [](const Tensor& g, const Tensor& x, const Tensor& w, const Tensor& conv_w, const Tensor& rotations,
                       const std::vector<Tensor>& s, int64_t side, int64_t heads, const std::array<bool, 5>& need, bool kernel) {
    return listed(mlla_bwd(g, x, w, conv_w, rotations, s, side, heads, need, kernel));
  });
  op("pola_fwd", [](const Tensor& x, const Tensor& src, const std::vector<Maybe>& p, double alpha, int64_t H, int64_t W, int64_t heads,
                    bool trains) { return listed(pola_fwd(x, src, p, alpha, H, W, heads, trains)); });
  op("pola_bwd", [](const Tensor& g, const Tensor& x, const Tensor& src, bool same, const std::vector<Maybe>& p,
                       const std::vector<Maybe>& s, double alpha, int64_t H, int64_t W, int64_t heads, const std::array<bool, 13>& need,
                       const std::array<bool, 3>& kernel) { return listed(pola_bwd(g, x, src, same, p, s, alpha, H, W, heads, need, kernel)); });
  op("focused_fwd", [](const Tensor& x, const Tensor& src, const std::vector<Maybe>& p, int64_t H, int64_t W, int64_t heads,
                       bool trains) { return listed(focused_fwd(x, src, p, H, W, heads, trains)); });
  op("focused_bwd", [](const Tensor& g, const Tensor& x, const Tensor& src, bool same, const std::vector<Maybe>& p,
                          const std::vector<Maybe>& s, int64_t H, int64_t W, int64_t heads, const std::array<bool, 12>& need,
                          const std::array<bool, 3>& kernel) { return listed(focused_bwd(g, x, src, same, p, s, H, W, heads, need, kernel)); });
  op("linfusion_fwd", [](const Tensor& x, const Tensor& cu, const std::vector<Maybe>& p, const std::array<double, 2>& eps,
                            const std::array<double, 2>& slope, int64_t heads, bool trains) {
    return listed(linfusion_fwd(x, cu, p, eps, slope, heads, trains));
  });
  op("linfusion_bwd", [](const Tensor& g, const Tensor& x, const Tensor& cu, const std::vector<Maybe>& p, const std::vector<Maybe>& s,
                            const std::array<double, 2>& slope, const std::array<bool, 21>& need, const std::array<bool, 8>& kernel) {
    return listed(linfusion_bwd(g, x, cu, p, s, slope, need, kernel));
  });
  m.def("dense_operands", &dense_operands);
  const py::object parameter = py::module_::import("torch.nn").attr("Parameter");
  m.def("plain_gpu_tensors", [parameter](py::handle x, py::args rest) { return plain_gpu_tensors(x, rest, parameter.ptr()); });
  m.def("untouched_modules", &untouched_modules);
  m.def("projects", &projects);
  m.def("mlla_fits", &mlla_fits);
  m.def("pola_fits", &pola_fits);
  m.def("focused_fits", &focused_fits);
  m.def("linfusion_fits", &linfusion_fits);
}
