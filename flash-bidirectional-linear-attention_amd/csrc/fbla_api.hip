// C-ABI layer of libfbla_hip.so: argument checks, kernel-family dispatch and
// error reporting.  Declarations and the reference call sites each entry point
// replaces are in include/flash_bla_hip.h.
#include <stdarg.h>
#include <stdio.h>
#include <stdlib.h>

#include <atomic>
#include <initializer_list>
#include <mutex>

#include "../../include/flash_bla_hip.h"
#include "fbla_kernels.h"

namespace fbla {

static thread_local char g_err[512] = "";

void set_error(const char* fmt, ...) {
  va_list ap;
  va_start(ap, fmt);
  vsnprintf(g_err, sizeof(g_err), fmt, ap);
  va_end(ap);
}

static thread_local unsigned g_phase_mask = kPhaseAll;
unsigned phase_mask() { return g_phase_mask; }

static int check_launch(const char* what) {
  hipError_t e = hipGetLastError();
  if (e != hipSuccess) {
    set_error("%s: kernel launch failed: %s", what, hipGetErrorString(e));
    return kErrLaunch;
  }
  return kOk;
}

static int check_dims(const char* what, int64_t N, int64_t H, int64_t L, int DK, int DV,
                      int dtype, int flags) {
  if (N < 0 || H <= 0 || L < 0) {
    set_error("%s: bad sizes N=%lld H=%lld L=%lld", what, (long long)N, (long long)H, (long long)L);
    return kErrBadArg;
  }
  if (DK < 1 || DK > 128 || DV < 1 || DV > 128) {
    set_error("%s: head dims must be in [1,128], got DK=%d DV=%d", what, DK, DV);
    return kErrUnsupported;
  }
  if (dtype != kF16 && dtype != kBF16 && dtype != kF32) {
    set_error("%s: unknown dtype %d", what, dtype);
    return kErrBadArg;
  }
  if (flags & ~kPublicFlags) {
    set_error("%s: unknown flag bits 0x%x", what, flags & ~kPublicFlags);
    return kErrBadArg;
  }
  if ((flags & kDecoupled) && !(flags & kNormalize)) {
    set_error("%s: FBLA_DECOUPLED requires FBLA_NORMALIZE", what);
    return kErrBadArg;
  }
  if (N * H > 0x7fffffffLL / 4 || L > 0x7fffffffLL / 2) {
    set_error("%s: problem too large for 32-bit grid indexing", what);
    return kErrUnsupported;
  }
  return kOk;
}

// The kernels move 16-byte pieces of rows.
static int check_aligned(const char* what, std::initializer_list<const void*> ptrs) {
  for (const void* ptr : ptrs)
    if (reinterpret_cast<uintptr_t>(ptr) & 15) {
      set_error("%s: tensor pointers must be 16-byte aligned", what);
      return kErrBadArg;
    }
  return kOk;
}

static Prob make_prob(const int32_t* cu, int64_t N, int64_t H, int64_t L, int64_t T, int DK, int DV,
                      int flags, float scale, float eps) {
  Prob p{};
  p.cu = cu;
  p.perm = nullptr;
  p.chunk_base = nullptr;
  p.N = (int)N;
  p.H = (int)H;
  p.L = (int)L;
  p.Lk = 0;
  p.T = T;
  p.DK = DK;
  p.DV = DV;
  p.RK = p.RV = 0;
  p.scale = scale;
  p.eps = eps;
  p.flags = flags;
  return p;
}

static size_t workspace_bytes(const Prob& p, int dtype, int pass) {
  return pass == 0 ? plan::fwd_workspace_bytes(p, dtype) : plan::bwd_workspace_bytes(p, dtype);
}

// The dense forward of fbla_la_fwd and fbla_la_fwd_static.  Finer chunks for few heads (up to 8 MiB of partials) are not taken
// where the problem fits the built-in scratch without them only: what that entry point takes does not depend on them.
static Prob forward_prob(const Prob& p, int dtype) {
  if (workspace_bytes(p, dtype, 0) <= FBLA_STATIC_SCRATCH_BYTES) return p;
  Prob coarse = p;
  coarse.flags |= kCoarse;
  return workspace_bytes(coarse, dtype, 0) <= FBLA_STATIC_SCRATCH_BYTES ? coarse : p;
}

static int run_fwd(const char* what, const Prob& p, int dtype, const FwdArgs& a, hipStream_t st) {
  if ((int64_t)p.N * p.H == 0 || p.L == 0) return kOk;
  if (check_aligned(what, {a.q, a.k, a.v, a.q_rope, a.k_rope, a.o, a.s, a.km, a.workspace}) != kOk)
    return kErrBadArg;
  const size_t need = workspace_bytes(p, dtype, 0);
  if (a.workspace_bytes < need || (need && !a.workspace)) {
    set_error("%s: workspace too small (%zu < %zu bytes)", what, a.workspace_bytes, need);
    return kErrWorkspace;
  }
  int rc = plan::forward(p, dtype, a, st);
  if (rc != kOk) return rc;
  return check_launch(what);
}

static int run_bwd(const char* what, const Prob& p, int dtype, const BwdArgs& a, hipStream_t st) {
  if ((int64_t)p.N * p.H == 0 || p.L == 0) return kOk;
  if (check_aligned(what, {a.q, a.k, a.v, a.q_rope, a.k_rope, a.dout, a.s, a.km, a.dq, a.dk, a.dv, a.dq_rope,
                           a.dk_rope, a.workspace}) != kOk)
    return kErrBadArg;
  const size_t need = workspace_bytes(p, dtype, 1);
  if (a.workspace_bytes < need || (need && !a.workspace)) {
    set_error("%s: workspace too small (%zu < %zu bytes)", what, a.workspace_bytes, need);
    return kErrWorkspace;
  }
  int rc = plan::backward(p, dtype, a, st);
  if (rc != kOk) return rc;
  return check_launch(what);
}

}  // namespace fbla

using namespace fbla;

extern "C" {

int fbla_version(void) { return 100; }

// Only honoured when the process opted in through the environment: a caller cannot switch kernels
// off by accident, and a mask left set by a profiling script that died cannot outlive its process.
void fbla_set_phase_mask(unsigned mask) {
  static const bool allowed = [] { const char* v = getenv("FBLA_ALLOW_PHASE_MASK"); return v && v[0] == '1'; }();
  g_phase_mask = (allowed && mask) ? mask : kPhaseAll;
}

const char* fbla_last_error(void) { return g_err; }

size_t fbla_la_workspace_bytes(int pass, int64_t B, int64_t H, int64_t L, int DK, int DV, int dtype,
                               int flags) {
  if (check_dims("fbla_la_workspace_bytes", B, H, L, DK, DV, dtype, flags) != kOk) return 0;
  Prob p = make_prob(nullptr, B, H, L, B * L, DK, DV, flags, 1.f, 0.f);
  return workspace_bytes(pass == 0 ? forward_prob(p, dtype) : p, dtype, pass);
}

int fbla_la_fwd(const void* q, const void* k, const void* v, const void* q_rope,
                const void* k_rope, void* o, float* s, float* km, void* workspace,
                size_t workspace_bytes_, int64_t B, int64_t H, int64_t L, int DK, int DV, int dtype,
                int flags, float scale, float eps, void* stream) {
  const char* what = "fbla_la_fwd";
  int rc = check_dims(what, B, H, L, DK, DV, dtype, flags);
  if (rc != kOk) return rc;
  if (flags & kDefaultScale) {
    set_error("%s: FBLA_DEFAULT_SCALE is only valid for the packed entry points", what);
    return kErrBadArg;
  }
  if (!q || !k || !v || !o || !s || ((flags & kNormalize) && !km) ||
      ((flags & kDecoupled) && (!q_rope || !k_rope))) {
    if (B * H * L != 0) {
      set_error("%s: null tensor pointer", what);
      return kErrBadArg;
    }
  }
  const Prob p = forward_prob(make_prob(nullptr, B, H, L, B * L, DK, DV, flags, scale, eps), dtype);
  FwdArgs a{q, k, v, q_rope, k_rope, o, s, km, workspace, workspace_bytes_};
  return run_fwd(what, p, dtype, a, (hipStream_t)stream);
}

int fbla_la_bwd(const void* q, const void* k, const void* v, const void* q_rope,
                const void* k_rope, const void* dout, const float* s, const float* km, void* dq,
                void* dk, void* dv, void* dq_rope, void* dk_rope, void* workspace,
                size_t workspace_bytes_, int64_t B, int64_t H, int64_t L, int DK, int DV, int dtype,
                int flags, float scale, float eps, void* stream) {
  const char* what = "fbla_la_bwd";
  int rc = check_dims(what, B, H, L, DK, DV, dtype, flags);
  if (rc != kOk) return rc;
  if (flags & kDefaultScale) {
    set_error("%s: FBLA_DEFAULT_SCALE is only valid for the packed entry points", what);
    return kErrBadArg;
  }
  const bool dec = flags & kDecoupled;
  if (B * H * L != 0 &&
      (!q || !v || !dout || !s || !dq || !dk || !dv || (!dec && !k) || ((flags & kNormalize) && !km) ||
       (dec && (!q_rope || !k_rope || !dq_rope || !dk_rope)))) {
    set_error("%s: null tensor pointer", what);
    return kErrBadArg;
  }
  Prob p = make_prob(nullptr, B, H, L, B * L, DK, DV, flags, scale, eps);
  BwdArgs a{q, k, v, q_rope, k_rope, dout, s, km, dq, dk, dv, dq_rope, dk_rope, workspace,
            workspace_bytes_};
  return run_bwd(what, p, dtype, a, (hipStream_t)stream);
}

// ---- the entry point that allocates nothing ------------------------------------------------
// Workspace of fbla_la_fwd_static: a fixed array in the library's device image.  Every GPU the
// library runs on holds its own copy at its own address until the process ends; host code may
// only use the address hipGetSymbolAddress returns for the current device, never the array's
// name (which is a host-side stand-in).
static constexpr size_t kStaticScratchBytes = (size_t)FBLA_STATIC_SCRATCH_BYTES;
static __device__ __align__(256) unsigned char scratch[kStaticScratchBytes];

static constexpr int kMaxDevices = 64;
static std::atomic<void*> g_scratch_ptr[kMaxDevices];  // zero-initialised: not looked up yet
static std::mutex g_scratch_mutex;

// Device address of `scratch` on the current device (looked up once per device), or null with
// the error text set.
static void* static_scratch(const char* what) {
  int dev = -1;
  hipError_t e = hipGetDevice(&dev);
  if (e != hipSuccess || dev < 0 || dev >= kMaxDevices) {
    set_error("%s: cannot identify the current device (%s)", what,
              e != hipSuccess ? hipGetErrorString(e) : "device index out of range");
    return nullptr;
  }
  void* ptr = g_scratch_ptr[dev].load(std::memory_order_acquire);
  if (ptr) return ptr;
  std::lock_guard<std::mutex> lock(g_scratch_mutex);
  ptr = g_scratch_ptr[dev].load(std::memory_order_relaxed);
  if (ptr) return ptr;
  e = hipGetSymbolAddress(&ptr, HIP_SYMBOL(scratch));
  if (e != hipSuccess || !ptr) {
    set_error("%s: hipGetSymbolAddress(scratch) failed on device %d: %s", what, dev, hipGetErrorString(e));
    return nullptr;
  }
  g_scratch_ptr[dev].store(ptr, std::memory_order_release);
  return ptr;
}

size_t fbla_static_scratch_bytes(void) { return kStaticScratchBytes; }

int fbla_la_fwd_static(const void* q, const void* k, const void* v, const void* q_rope, const void* k_rope,
                       void* o, float* s, float* km, int64_t B, int64_t H, int64_t L, int DK, int DV,
                       int dtype, int flags, float scale, float eps, void* stream) {
  const char* what = "fbla_la_fwd_static";
  int rc = check_dims(what, B, H, L, DK, DV, dtype, flags);
  if (rc != kOk) return rc;
  if (flags & kDefaultScale) {
    set_error("%s: FBLA_DEFAULT_SCALE is only valid for the packed entry points", what);
    return kErrBadArg;
  }
  if (B * H * L == 0) return kOk;
  if (!q || !k || !v || !o || !s || ((flags & kNormalize) && !km) ||
      ((flags & kDecoupled) && (!q_rope || !k_rope))) {
    set_error("%s: null tensor pointer", what);
    return kErrBadArg;
  }
  const Prob p = forward_prob(make_prob(nullptr, B, H, L, B * L, DK, DV, flags, scale, eps), dtype);
  const size_t need = workspace_bytes(p, dtype, 0);
  if (need > kStaticScratchBytes) {
    set_error("%s: this problem needs %zu bytes of workspace, the built-in scratch holds %zu; "
              "use fbla_la_fwd with a caller-provided workspace", what, need, kStaticScratchBytes);
    return kErrWorkspace;
  }
  void* ws = static_scratch(what);
  if (!ws) return kErrLaunch;
  // Every partial the reductions read is written earlier in the same call, so nothing in the
  // scratch has to start at zero.
  FwdArgs a{q, k, v, q_rope, k_rope, o, s, km, ws, kStaticScratchBytes};
  return run_fwd(what, p, dtype, a, (hipStream_t)stream);
}

// ---- two queries on shared keys and values ---------------------------------------------------
size_t fbla_la_pair_workspace_bytes(int pass, int64_t B, int64_t H, int64_t L, int DK, int DV, int dtype) {
  if (check_dims("fbla_la_pair_workspace_bytes", B, H, L, DK, DV, dtype, kNormalize) != kOk) return 0;
  Prob p = make_prob(nullptr, B, H, L, B * L, DK, DV, kNormalize, 1.f, 0.f);
  if (!plan::pair_supported(p, dtype)) return 0;
  return pass == 0 ? plan::pair_fwd_workspace_bytes(p, dtype) : plan::pair_bwd_workspace_bytes(p, dtype);
}

int fbla_la_pair_fwd(const void* q1, const void* q2, const void* k, const void* v, void* o1, void* o2, float* s,
                     float* km, void* workspace, size_t workspace_bytes_, int64_t B, int64_t H, int64_t L, int DK,
                     int DV, int dtype, float scale, float eps, void* stream) {
  const char* what = "fbla_la_pair_fwd";
  int rc = check_dims(what, B, H, L, DK, DV, dtype, kNormalize);
  if (rc != kOk) return rc;
  if (B * H * L == 0) return kOk;
  if (!q1 || !q2 || !k || !v || !o1 || !o2 || !s || !km) {
    set_error("%s: null tensor pointer", what);
    return kErrBadArg;
  }
  if (check_aligned(what, {q1, q2, k, v, o1, o2, s, km, workspace}) != kOk) return kErrBadArg;
  Prob p = make_prob(nullptr, B, H, L, B * L, DK, DV, kNormalize, scale, eps);
  if (!plan::pair_supported(p, dtype)) {
    set_error("%s: needs dense fp16 / bf16 tensors with DK, DV/2 multiples of 8 (got DK=%d DV=%d dtype=%d)", what, DK,
              DV, dtype);
    return kErrUnsupported;
  }
  const size_t need = plan::pair_fwd_workspace_bytes(p, dtype);
  if (workspace_bytes_ < need || !workspace) {
    set_error("%s: workspace too small (%zu < %zu bytes)", what, workspace_bytes_, need);
    return kErrWorkspace;
  }
  PairFwdArgs a{{q1, q2}, k, v, {o1, o2}, s, km, workspace, workspace_bytes_};
  rc = plan::pair_forward(p, dtype, a, (hipStream_t)stream);
  return rc != kOk ? rc : check_launch(what);
}

int fbla_la_pair_bwd(const void* q1, const void* q2, const void* k, const void* v, const void* dout1,
                     const void* dout2, const float* s, const float* km, void* dq1, void* dq2, void* dk, void* dv,
                     void* workspace, size_t workspace_bytes_, int64_t B, int64_t H, int64_t L, int DK, int DV,
                     int dtype, float scale, float eps, void* stream) {
  const char* what = "fbla_la_pair_bwd";
  int rc = check_dims(what, B, H, L, DK, DV, dtype, kNormalize);
  if (rc != kOk) return rc;
  if (B * H * L == 0) return kOk;
  if (!q1 || !q2 || !k || !v || !dout1 || !dout2 || !s || !km || !dq1 || !dq2 || !dk || !dv) {
    set_error("%s: null tensor pointer", what);
    return kErrBadArg;
  }
  if (check_aligned(what, {q1, q2, k, v, dout1, dout2, s, km, dq1, dq2, dk, dv, workspace}) != kOk) return kErrBadArg;
  Prob p = make_prob(nullptr, B, H, L, B * L, DK, DV, kNormalize, scale, eps);
  if (!plan::pair_supported(p, dtype)) {
    set_error("%s: needs dense fp16 / bf16 tensors with DK, DV/2 multiples of 8 (got DK=%d DV=%d dtype=%d)", what, DK,
              DV, dtype);
    return kErrUnsupported;
  }
  const size_t need = plan::pair_bwd_workspace_bytes(p, dtype);
  if (workspace_bytes_ < need || !workspace) {
    set_error("%s: workspace too small (%zu < %zu bytes)", what, workspace_bytes_, need);
    return kErrWorkspace;
  }
  PairBwdArgs a{{q1, q2}, k, v, {dout1, dout2}, s, km, {dq1, dq2}, dk, dv, workspace, workspace_bytes_};
  rc = plan::pair_backward(p, dtype, a, (hipStream_t)stream);
  return rc != kOk ? rc : check_launch(what);
}

static int check_cross(const char* what, int64_t Lk, int flags) {
  if (Lk <= 0 || Lk > 0x7fffffffLL / 2) {
    set_error("%s: the number of keys must be positive and fit 32-bit indexing, got %lld", what, (long long)Lk);
    return kErrBadArg;
  }
  if (flags & kDefaultScale) {
    set_error("%s: FBLA_DEFAULT_SCALE is only valid for the packed entry points", what);
    return kErrBadArg;
  }
  return kOk;
}

size_t fbla_la_cross_workspace_bytes(int pass, int64_t B, int64_t H, int64_t Lq, int64_t Lk, int DK, int DV,
                                     int dtype, int flags) {
  const char* what = "fbla_la_cross_workspace_bytes";
  if (check_dims(what, B, H, Lq, DK, DV, dtype, flags) != kOk || check_cross(what, Lk, flags) != kOk) return 0;
  Prob p = make_prob(nullptr, B, H, Lq, B * Lq, DK, DV, flags, 1.f, 0.f);
  p.Lk = (int)Lk;
  return workspace_bytes(p, dtype, pass);
}

static int cross_fwd(const char* what, const void* q, const void* k, const void* v, const void* q_rope,
                     const void* k_rope, void* o, float* s, float* km, void* workspace, size_t workspace_bytes_,
                     int64_t B, int64_t H, int64_t Lq, int64_t Lk, int DK, int DV, int dtype, int flags, float scale,
                     float eps, void* stream) {
  int rc = check_dims(what, B, H, Lq, DK, DV, dtype, flags);
  if (rc == kOk) rc = check_cross(what, Lk, flags);
  if (rc != kOk) return rc;
  if (B * H > 0 && Lq > 0 &&
      (!q || !k || !v || !o || !s || ((flags & kNormalize) && !km) || ((flags & kDecoupled) && (!q_rope || !k_rope)))) {
    set_error("%s: null tensor pointer", what);
    return kErrBadArg;
  }
  Prob p = make_prob(nullptr, B, H, Lq, B * Lq, DK, DV, flags, scale, eps);
  p.Lk = (int)Lk;
  FwdArgs a{q, k, v, q_rope, k_rope, o, s, km, workspace, workspace_bytes_};
  return run_fwd(what, p, dtype, a, (hipStream_t)stream);
}

int fbla_la_cross_fwd(const void* q, const void* k, const void* v, void* o, float* s, float* km,
                      void* workspace, size_t workspace_bytes_, int64_t B, int64_t H, int64_t Lq, int64_t Lk,
                      int DK, int DV, int dtype, int flags, float scale, float eps, void* stream) {
  if (flags & kDecoupled) {
    set_error("fbla_la_cross_fwd: the decoupled operator takes its rotary rows through fbla_decoupled_cross_fwd");
    return kErrBadArg;
  }
  return cross_fwd("fbla_la_cross_fwd", q, k, v, nullptr, nullptr, o, s, km, workspace, workspace_bytes_, B, H, Lq, Lk,
                   DK, DV, dtype, flags, scale, eps, stream);
}

int fbla_decoupled_cross_fwd(const void* q, const void* k, const void* q_rope, const void* k_rope, const void* v,
                             void* o, float* s, float* km, void* workspace, size_t workspace_bytes_, int64_t B,
                             int64_t H, int64_t Lq, int64_t Lk, int DK, int DV, int dtype, float scale, float eps,
                             void* stream) {
  return cross_fwd("fbla_decoupled_cross_fwd", q, k, v, q_rope, k_rope, o, s, km, workspace, workspace_bytes_, B, H, Lq,
                   Lk, DK, DV, dtype, kNormalize | kDecoupled, scale, eps, stream);
}

static int cross_bwd(const char* what, const void* q, const void* k, const void* v, const void* q_rope,
                     const void* k_rope, const void* dout, const float* s, const float* km, void* dq, void* dk,
                     void* dv, void* dq_rope, void* dk_rope, void* workspace, size_t workspace_bytes_, int64_t B,
                     int64_t H, int64_t Lq, int64_t Lk, int DK, int DV, int dtype, int flags, float scale, float eps,
                     void* stream) {
  int rc = check_dims(what, B, H, Lq, DK, DV, dtype, flags);
  if (rc == kOk) rc = check_cross(what, Lk, flags);
  if (rc != kOk) return rc;
  const bool dec = flags & kDecoupled;
  if (B * H > 0 && Lq > 0 &&
      (!q || !v || !dout || !s || ((flags & kNormalize) && !km) || !dq || !dk || !dv || (!dec && !k) ||
       (dec && (!q_rope || !k_rope || !dq_rope || !dk_rope)))) {
    set_error("%s: null tensor pointer", what);
    return kErrBadArg;
  }
  Prob p = make_prob(nullptr, B, H, Lq, B * Lq, DK, DV, flags, scale, eps);
  p.Lk = (int)Lk;
  BwdArgs a{q, k, v, q_rope, k_rope, dout, s, km, dq, dk, dv, dq_rope, dk_rope, workspace, workspace_bytes_};
  return run_bwd(what, p, dtype, a, (hipStream_t)stream);
}

int fbla_la_cross_bwd(const void* q, const void* k, const void* v, const void* dout, const float* s,
                      const float* km, void* dq, void* dk, void* dv, void* workspace, size_t workspace_bytes_,
                      int64_t B, int64_t H, int64_t Lq, int64_t Lk, int DK, int DV, int dtype, int flags,
                      float scale, float eps, void* stream) {
  if (flags & kDecoupled) {
    set_error("fbla_la_cross_bwd: the decoupled operator takes its rotary rows through fbla_decoupled_cross_bwd");
    return kErrBadArg;
  }
  return cross_bwd("fbla_la_cross_bwd", q, k, v, nullptr, nullptr, dout, s, km, dq, dk, dv, nullptr, nullptr, workspace,
                   workspace_bytes_, B, H, Lq, Lk, DK, DV, dtype, flags, scale, eps, stream);
}

int fbla_decoupled_cross_bwd(const void* q, const void* k, const void* q_rope, const void* k_rope, const void* v,
                             const void* dout, const float* s, const float* km, void* dq, void* dk, void* dq_rope,
                             void* dk_rope, void* dv, void* workspace, size_t workspace_bytes_, int64_t B, int64_t H,
                             int64_t Lq, int64_t Lk, int DK, int DV, int dtype, float scale, float eps, void* stream) {
  return cross_bwd("fbla_decoupled_cross_bwd", q, k, v, q_rope, k_rope, dout, s, km, dq, dk, dv, dq_rope, dk_rope,
                   workspace, workspace_bytes_, B, H, Lq, Lk, DK, DV, dtype, kNormalize | kDecoupled, scale, eps, stream);
}

size_t fbla_varlen_workspace_bytes(int pass, int64_t total_tokens, int64_t N, int64_t H,
                                   int64_t max_seqlen, int DK, int DV, int dtype, int flags) {
  if (check_dims("fbla_varlen_workspace_bytes", N, H, max_seqlen, DK, DV, dtype, flags) != kOk)
    return 0;
  static const int32_t dummy = 0;
  Prob p = make_prob(&dummy, N, H, max_seqlen, total_tokens, DK, DV, flags, 1.f, 0.f);
  return workspace_bytes(p, dtype, pass);
}

int fbla_varlen_fwd(const void* q, const void* k, const void* v, const int32_t* cu_seqlens,
                    void* o, float* s, float* km, void* workspace, size_t workspace_bytes_,
                    int64_t total_tokens, int64_t N, int64_t H, int64_t max_seqlen, int DK, int DV,
                    int dtype, int flags, float scale, float eps, void* stream) {
  const char* what = "fbla_varlen_fwd";
  int rc = check_dims(what, N, H, max_seqlen, DK, DV, dtype, flags);
  if (rc != kOk) return rc;
  if ((flags & kDecoupled) || !(flags & kNormalize)) {
    set_error("%s: only the normalised, non-decoupled operator has a packed form", what);
    return kErrUnsupported;
  }
  if (total_tokens == 0 || N == 0) return kOk;
  if (!q || !k || !v || !o || !s || !km || !cu_seqlens) {
    set_error("%s: null tensor pointer", what);
    return kErrBadArg;
  }
  Prob p = make_prob(cu_seqlens, N, H, max_seqlen, total_tokens, DK, DV, flags, scale, eps);
  FwdArgs a{q, k, v, nullptr, nullptr, o, s, km, workspace, workspace_bytes_};
  return run_fwd(what, p, dtype, a, (hipStream_t)stream);
}

int fbla_varlen_bwd(const void* q, const void* k, const void* v, const int32_t* cu_seqlens,
                    const void* dout, const float* s, const float* km, void* dq, void* dk, void* dv,
                    void* workspace, size_t workspace_bytes_, int64_t total_tokens, int64_t N,
                    int64_t H, int64_t max_seqlen, int DK, int DV, int dtype, int flags,
                    float scale, float eps, void* stream) {
  const char* what = "fbla_varlen_bwd";
  int rc = check_dims(what, N, H, max_seqlen, DK, DV, dtype, flags);
  if (rc != kOk) return rc;
  if ((flags & kDecoupled) || !(flags & kNormalize)) {
    set_error("%s: only the normalised, non-decoupled operator has a packed form", what);
    return kErrUnsupported;
  }
  if (total_tokens == 0 || N == 0) return kOk;
  if (!q || !k || !v || !dout || !s || !km || !dq || !dk || !dv || !cu_seqlens) {
    set_error("%s: null tensor pointer", what);
    return kErrBadArg;
  }
  Prob p = make_prob(cu_seqlens, N, H, max_seqlen, total_tokens, DK, DV, flags, scale, eps);
  BwdArgs a{q, k, v, nullptr, nullptr, dout, s, km, dq, dk, dv, nullptr, nullptr, workspace,
            workspace_bytes_};
  return run_bwd(what, p, dtype, a, (hipStream_t)stream);
}

size_t fbla_chunk_reduce_workspace_bytes(int64_t BH, int64_t T, int K, int V, int chunk, int dtype,
                                         int with_norm) {
  if (check_dims("fbla_chunk_reduce_workspace_bytes", BH, 1, T, K, V, dtype, 0) != kOk || chunk < 1)
    return 0;
  return piecewise::chunk_reduce_workspace_bytes(BH, T, K, V, chunk, dtype, with_norm != 0);
}

int fbla_chunk_reduce(const void* q, const void* k, const void* v, float* qc, float* kc, float* vc,
                      float* h, float* h_norm, void* workspace, size_t workspace_bytes_, int64_t BH,
                      int64_t T, int K, int V, int chunk, float p_norm, int dtype, void* stream) {
  const char* what = "fbla_chunk_reduce";
  int rc = check_dims(what, BH, 1, T, K, V, dtype, 0);
  if (rc != kOk) return rc;
  if (chunk < 1 || (h_norm && !(p_norm > 0.f))) {
    set_error("%s: chunk must be positive and the norm order > 0", what);
    return kErrBadArg;
  }
  if (BH == 0 || T == 0) return kOk;
  if (!q || !k || !v || !qc || !kc || !vc || !h) {
    set_error("%s: null tensor pointer", what);
    return kErrBadArg;
  }
  const size_t need = piecewise::chunk_reduce_workspace_bytes(BH, T, K, V, chunk, dtype, h_norm != nullptr);
  if (workspace_bytes_ < need || !workspace) {
    set_error("%s: workspace too small (%zu < %zu bytes)", what, workspace_bytes_, need);
    return kErrWorkspace;
  }
  rc = piecewise::chunk_reduce(q, k, v, qc, kc, vc, h, h_norm, workspace, BH, T, K, V, chunk, p_norm,
                               dtype, (hipStream_t)stream);
  if (rc != kOk) return rc;
  return check_launch(what);
}

// 16-bit inputs, blocks of a multiple of 64 tokens, head dims other than 64 / 128: the matrix-core kernel runs on copies
// widened with zeros to 64 / 128 (zero key features leave every score as it is, zero value columns give
// zero output columns, which are dropped again) instead of the shape-generic kernel, which is about ten
// times slower.  q | k | v | o | kc | vc | h (widened) | the kernel's own workspace
static int pw_wide(int d) { return d <= 64 ? 64 : 128; }
static bool pw_widen(int K, int V, int block, int dtype) {
  return (dtype == kF16 || dtype == kBF16) && piecewise::attention_supported(64, 64, block, dtype) && K <= 128 &&
         V <= 128 &&
         !piecewise::attention_supported(K, V, block, dtype);
}
static size_t pw_widened_bytes(int64_t BH, int64_t T, int K, int V, int block) {
  const int Kw = pw_wide(K), Vw = pw_wide(V);
  const int64_t NT = (T + block - 1) / block;
  return 2 * align_up((size_t)BH * T * Kw * 2, 256) + 2 * align_up((size_t)BH * T * Vw * 2, 256) +
         align_up((size_t)BH * NT * Kw * 4, 256) + align_up((size_t)BH * NT * Vw * 4, 256) +
         align_up((size_t)BH * Kw * Vw * 4, 256) + piecewise::attention_workspace_bytes(BH, T, Kw, Vw, block);
}

size_t fbla_piecewise_workspace_bytes(int64_t BH, int64_t T, int K, int V, int block, int dtype) {
  if (check_dims("fbla_piecewise_workspace_bytes", BH, 1, T, K, V, dtype, 0) != kOk) return 0;
  if (piecewise::attention_supported(K, V, block, dtype)) return piecewise::attention_workspace_bytes(BH, T, K, V, block);
  if (pw_widen(K, V, block, dtype)) return pw_widened_bytes(BH, T, K, V, block);
  // the shape-generic kernel needs no workspace; a token size keeps "0 = not supported"
  return piecewise::attention_generic_supported(T, K, V, block, dtype) ? 256 : 0;
}

int fbla_piecewise_fwd(const void* q, const void* k, const void* v, const float* kc, const float* vc,
                       const float* h, const int32_t* indices, void* o, void* workspace,
                       size_t workspace_bytes_, int64_t BH, int64_t T, int K, int V, int block, int NS,
                       float scale, int dtype, void* stream) {
  const char* what = "fbla_piecewise_fwd";
  int rc = check_dims(what, BH, 1, T, K, V, dtype, 0);
  if (rc != kOk) return rc;
  const bool widen = pw_widen(K, V, block, dtype);
  const bool fast = widen || piecewise::attention_supported(K, V, block, dtype);
  if (!fast && !piecewise::attention_generic_supported(T, K, V, block, dtype)) {
    set_error("%s: needs head dims in [1,128], a positive block size and block flags that fit LDS "
              "(got K=%d V=%d block=%d dtype=%d T=%lld)", what, K, V, block, dtype, (long long)T);
    return kErrUnsupported;
  }
  const int64_t NT = (T + block - 1) / block;
  if (NS < 1 || NS > NT) {
    set_error("%s: the number of selected blocks must be in [1, %lld], got %d", what, (long long)NT, NS);
    return kErrBadArg;
  }
  if (BH == 0 || T == 0) return kOk;
  if (!q || !k || !v || !kc || !vc || !h || !indices || !o) {
    set_error("%s: null tensor pointer", what);
    return kErrBadArg;
  }
  if (!fast) {
    rc = piecewise::attention_generic(q, k, v, kc, vc, h, indices, o, BH, T, K, V, block, NS, scale, dtype,
                                      (hipStream_t)stream);
    if (rc != kOk) return rc;
    return check_launch(what);
  }
  const size_t need = widen ? pw_widened_bytes(BH, T, K, V, block) : piecewise::attention_workspace_bytes(BH, T, K, V, block);
  if (workspace_bytes_ < need || !workspace) {
    set_error("%s: workspace too small (%zu < %zu bytes)", what, workspace_bytes_, need);
    return kErrWorkspace;
  }
  if (widen) {
    hipStream_t st = (hipStream_t)stream;
    const int Kw = pw_wide(K), Vw = pw_wide(V);
    char* ws = (char*)workspace;
    auto take = [&](size_t bytes) { void* r = ws; ws += align_up(bytes, 256); return r; };
    void* qw = take((size_t)BH * T * Kw * 2);
    void* kw = take((size_t)BH * T * Kw * 2);
    void* vw = take((size_t)BH * T * Vw * 2);
    void* ow = take((size_t)BH * T * Vw * 2);
    float* kcw = (float*)take((size_t)BH * NT * Kw * 4);
    float* vcw = (float*)take((size_t)BH * NT * Vw * 4);
    float* hw = (float*)take((size_t)BH * Kw * Vw * 4);
    generic::resize_matrices(q, BH * T, K, qw, BH * T, Kw, 1, 2, st);
    generic::resize_matrices(k, BH * T, K, kw, BH * T, Kw, 1, 2, st);
    generic::resize_matrices(v, BH * T, V, vw, BH * T, Vw, 1, 2, st);
    generic::resize_matrices(kc, BH * NT, K, kcw, BH * NT, Kw, 1, 4, st);
    generic::resize_matrices(vc, BH * NT, V, vcw, BH * NT, Vw, 1, 4, st);
    generic::resize_matrices(h, K, V, hw, Kw, Vw, BH, 4, st);
    rc = piecewise::attention(qw, kw, vw, kcw, vcw, hw, indices, ow, ws, BH, T, Kw, Vw, block, NS, scale, dtype, st);
    if (rc != kOk) return rc;
    generic::resize_matrices(ow, BH * T, Vw, o, BH * T, V, 1, 2, st);
    return check_launch(what);
  }
  rc = piecewise::attention(q, k, v, kc, vc, h, indices, o, workspace, BH, T, K, V, block, NS, scale, dtype,
                            (hipStream_t)stream);
  if (rc != kOk) return rc;
  return check_launch(what);
}

int fbla_select_blocks(const float* qc, const float* kc, const float* bias, int32_t* indices,
                       int64_t BH, int64_t NT, int K, int NS, float scale, void* stream) {
  const char* what = "fbla_select_blocks";
  if (BH < 0 || NT < 0 || NT > 0x7fffffffLL / 64) {
    set_error("%s: bad sizes BH=%lld NT=%lld", what, (long long)BH, (long long)NT);
    return kErrBadArg;
  }
  if (BH == 0 || NT == 0) return kOk;
  if (NS < 1 || NS > NT) {
    set_error("%s: the number of selected blocks must be in [1, %lld], got %d", what, (long long)NT, NS);
    return kErrBadArg;
  }
  if (!piecewise::select_blocks_supported((int)NT, K)) {
    set_error("%s: needs K in [1,128] and a score row that fits LDS (got K=%d NT=%lld)", what, K,
              (long long)NT);
    return kErrUnsupported;
  }
  if (!qc || !kc || !indices) {
    set_error("%s: null tensor pointer", what);
    return kErrBadArg;
  }
  int rc = piecewise::select_blocks(qc, kc, bias, indices, BH, (int)NT, K, NS, scale, (hipStream_t)stream);
  if (rc != kOk) return rc;
  return check_launch(what);
}

int fbla_elu1_fwd(const void* x0, void* y0, int64_t n0, const void* x1, void* y1, int64_t n1, int dtype,
                  void* stream) {
  const char* what = "fbla_elu1_fwd";
  if (n0 < 0 || n1 < 0 || (dtype != kF16 && dtype != kBF16 && dtype != kF32)) {
    set_error("%s: bad sizes or dtype (n0=%lld n1=%lld dtype=%d)", what, (long long)n0, (long long)n1, dtype);
    return kErrBadArg;
  }
  if (n0 == 0 && n1 == 0) return kOk;
  if ((n0 > 0 && (!x0 || !y0)) || (n1 > 0 && (!x1 || !y1))) {
    set_error("%s: null tensor pointer", what);
    return kErrBadArg;
  }
  if (check_aligned(what, {n0 > 0 ? x0 : nullptr, n0 > 0 ? y0 : nullptr, n1 > 0 ? x1 : nullptr,
                           n1 > 0 ? y1 : nullptr}) != kOk)
    return kErrBadArg;
  feature::elu1_fwd(x0, y0, n0, x1, y1, n1, dtype, (hipStream_t)stream);
  return check_launch(what);
}

int fbla_elu1_bwd(const void* x, const void* dy, void* dx, int64_t n, int dtype, void* stream) {
  const char* what = "fbla_elu1_bwd";
  if (n < 0 || (dtype != kF16 && dtype != kBF16 && dtype != kF32)) {
    set_error("%s: bad size or dtype (n=%lld dtype=%d)", what, (long long)n, dtype);
    return kErrBadArg;
  }
  if (n == 0) return kOk;
  if (!x || !dy || !dx) {
    set_error("%s: null tensor pointer", what);
    return kErrBadArg;
  }
  if (check_aligned(what, {x, dy, dx}) != kOk) return kErrBadArg;
  feature::elu1_bwd(x, dy, dx, n, dtype, (hipStream_t)stream);
  return check_launch(what);
}

// common checks of the depth-wise convolution entry points; fills `c` (x, y, w, bias and strides are the caller's)
static int check_dwconv(const char* what, dwconv::Conv& c, int64_t B, int64_t H, int64_t W, int C, int Cw, int K,
                        int dtype) {
  if (B < 0 || H < 1 || W < 1 || C < 1 || Cw < 1 || (dtype != kF16 && dtype != kBF16 && dtype != kF32)) {
    set_error("%s: bad sizes or dtype (B=%lld H=%lld W=%lld C=%d Cw=%d dtype=%d)", what, (long long)B, (long long)H,
              (long long)W, C, Cw, dtype);
    return kErrBadArg;
  }
  if (!dwconv::supported(C, Cw, K, dtype)) {
    set_error("%s: needs 3, 5 or 7 taps a side, channels in whole 16-byte pieces and a multiple of the filters "
              "(K=%d C=%d Cw=%d)", what, K, C, Cw);
    return kErrUnsupported;
  }
  if (H > 0x7fffffffLL / W || B > 0x7fffffffLL / (H * W) || C > 64 * 65535) {
    set_error("%s: too many tokens or channels", what);
    return kErrBadArg;
  }
  c.B = (int)B;
  c.H = (int)H;
  c.W = (int)W;
  c.C = C;
  c.Cw = Cw;
  return kOk;
}
static int check_row_strides(const char* what, int C, int dtype, std::initializer_list<int64_t> strides) {
  const int vec = dtype == kF32 ? 4 : 8;
  for (int64_t s : strides)
    if (s < C || s % vec) {
      set_error("%s: strides must be at least C elements and whole 16-byte pieces (got %lld)", what, (long long)s);
      return kErrBadArg;
    }
  return kOk;
}

int fbla_dwconv_fwd(const void* x, int64_t x_batch, int64_t x_row, const void* w, const void* bias, void* y,
                    int64_t y_batch, int64_t y_row, int64_t B, int64_t H, int64_t W, int C, int Cw, int K, int flip,
                    int dtype, void* stream) {
  const char* what = "fbla_dwconv_fwd";
  dwconv::Conv c{x, x_batch, x_row, w, bias, y, y_batch, y_row};
  int rc = check_dwconv(what, c, B, H, W, C, Cw, K, dtype);
  if (rc != kOk || B == 0) return rc;
  if (!x || !w || !y) {
    set_error("%s: null tensor pointer", what);
    return kErrBadArg;
  }
  if (check_aligned(what, {x, y}) != kOk || check_row_strides(what, C, dtype, {x_batch, x_row, y_batch, y_row}) != kOk)
    return kErrBadArg;
  // the rows of y are written by different workgroups: batches one after the other, or interleaved by tokens
  if (B > 1 && y_batch < (H * W - 1) * y_row + C && y_row < (B - 1) * y_batch + C) {
    set_error("%s: the batches of y overlap (y_batch=%lld y_row=%lld for %lld x %lld tokens)", what, (long long)y_batch,
              (long long)y_row, (long long)H, (long long)W);
    return kErrBadArg;
  }
  dwconv::forward(c, K, dtype, flip != 0, (hipStream_t)stream);
  return check_launch(what);
}

size_t fbla_dwconv_grad_workspace_bytes(int64_t B, int64_t H, int64_t W, int C, int Cw, int K, int dtype) {
  dwconv::Conv c{};
  if (check_dwconv("fbla_dwconv_grad_workspace_bytes", c, B, H, W, C, Cw, K, dtype) != kOk || B == 0) return 0;
  return dwconv::grad_workspace_bytes(c, K, dtype);
}

int fbla_dwconv_grad(const void* x, int64_t x_batch, int64_t x_row, const void* g, int64_t g_batch, int64_t g_row,
                     void* dw, void* db, void* workspace, size_t workspace_bytes, int64_t B, int64_t H, int64_t W,
                     int C, int Cw, int K, int dtype, void* stream) {
  const char* what = "fbla_dwconv_grad";
  dwconv::Conv c{x, x_batch, x_row};
  int rc = check_dwconv(what, c, B, H, W, C, Cw, K, dtype);
  if (rc != kOk) return rc;
  if (B == 0) {
    set_error("%s: empty batch", what);
    return kErrBadArg;
  }
  if (!x || !g || (!dw && !db)) {
    set_error("%s: null tensor pointer", what);
    return kErrBadArg;
  }
  if (check_aligned(what, {x, g, workspace}) != kOk ||
      check_row_strides(what, C, dtype, {x_batch, x_row, g_batch, g_row}) != kOk)
    return kErrBadArg;
  const size_t need = dwconv::grad_workspace_bytes(c, K, dtype);
  if (!workspace || workspace_bytes < need) {
    set_error("%s: workspace too small (%zu < %zu bytes)", what, workspace_bytes, need);
    return kErrWorkspace;
  }
  dwconv::grad(c, g, g_batch, g_row, dw, db, (float*)workspace, K, dtype, (hipStream_t)stream);
  return check_launch(what);
}

static int check_linear(const char* what, int64_t tokens, int M, int N, int dtype) {
  if (tokens < 1 || M < 1 || N < 1 || (dtype != kF16 && dtype != kBF16 && dtype != kF32)) {
    set_error("%s: bad sizes or dtype (tokens=%lld M=%d N=%d dtype=%d)", what, (long long)tokens, M, N, dtype);
    return kErrBadArg;
  }
  // the bound on the product keeps the result's indexes in 31 bits, the one on the tokens the chunks' lengths
  const int vec = dtype == kF32 ? 4 : 8;
  if (M % vec || N % vec || (int64_t)M * N > (1 << 28) || tokens > (1LL << 30)) {
    set_error("%s: needs rows of whole 16-byte pieces and at most 2^28 weights and 2^30 tokens "
              "(tokens=%lld M=%d N=%d dtype=%d)", what, (long long)tokens, M, N, dtype);
    return kErrUnsupported;
  }
  return kOk;
}

size_t fbla_linear_wgrad_workspace_bytes(int64_t tokens, int M, int N, int dtype) {
  if (check_linear("fbla_linear_wgrad_workspace_bytes", tokens, M, N, dtype) != kOk) return 0;
  return linear::wgrad_workspace_bytes(tokens, M, N);
}

int fbla_linear_wgrad(const void* g, int64_t g_row, const void* x, int64_t x_row, void* dw, void* db, void* workspace,
                      size_t workspace_bytes, int64_t tokens, int M, int N, int dtype, void* stream) {
  const char* what = "fbla_linear_wgrad";
  const int rc = check_linear(what, tokens, M, N, dtype);
  if (rc != kOk) return rc;
  if (!g || !x || !dw) {
    set_error("%s: null tensor pointer", what);
    return kErrBadArg;
  }
  if (check_aligned(what, {g, x, workspace}) != kOk || check_row_strides(what, M, dtype, {g_row}) != kOk ||
      check_row_strides(what, N, dtype, {x_row}) != kOk)
    return kErrBadArg;
  const size_t need = linear::wgrad_workspace_bytes(tokens, M, N);
  if (!workspace || workspace_bytes < need) {
    set_error("%s: workspace too small (%zu < %zu bytes)", what, workspace_bytes, need);
    return kErrWorkspace;
  }
  linear::wgrad(g, g_row, x, x_row, tokens, M, N, dw, db, (float*)workspace, dtype, (hipStream_t)stream);
  return check_launch(what);
}

int fbla_project(const fbla_projection* jobs, int count, int64_t tokens, int rows_of_w, int dtype, void* stream) {
  const char* what = "fbla_project";
  if (!jobs || count < 1 || count > gemm::kMostJobs || tokens < 0) {
    set_error("%s: bad sizes (count=%d tokens=%lld)", what, count, (long long)tokens);
    return kErrBadArg;
  }
  if (dtype != kF16 && dtype != kBF16) {
    set_error("%s: fp16 and bf16 only (dtype=%d)", what, dtype);
    return kErrUnsupported;
  }
  if (tokens == 0) return kOk;
  gemm::Job js[gemm::kMostJobs];
  int64_t tiles = 0;
  for (int i = 0; i < count; ++i) {
    const fbla_projection& j = jobs[i];
    const int K2 = j.a2 ? j.K2 : 0;
    // (32-bit offsets into W and into the rows of a tile)
    if (j.N > 1 << 16 || j.K > 1 << 16 || K2 > 1 << 16 || (int64_t)j.N * (j.K > K2 ? j.K : K2) > 1 << 29 || j.a_row > 1 << 22 ||
        (j.a2 && j.a2_row > 1 << 22)) {
      set_error("%s: too many channels (N=%d K=%d K2=%d)", what, j.N, j.K, K2);
      return kErrUnsupported;
    }
    if (!j.a || !j.w || !j.out || (j.a2 && !j.w2) || j.N < 8 || j.K < 8 || (j.a2 && j.K2 < 8) || j.N % 8 || j.K % 8 || K2 % 8) {
      set_error("%s: null pointers, or channels that are no multiples of 8 (N=%d K=%d K2=%d)", what, j.N, j.K, K2);
      return kErrBadArg;
    }
    if (check_aligned(what, {j.a, j.w, j.a2, j.w2, j.bias, j.add, j.out}) != kOk || check_row_strides(what, j.K, dtype, {j.a_row}) != kOk ||
        check_row_strides(what, j.N, dtype, {j.out_row}) != kOk || (j.a2 && check_row_strides(what, j.K2, dtype, {j.a2_row}) != kOk) ||
        (j.add && check_row_strides(what, j.N, dtype, {j.add_row}) != kOk))
      return kErrBadArg;
    js[i] = {{j.a, j.a2}, {j.a_row, j.a2_row}, {j.w, j.w2}, {j.K, K2}, j.N, j.bias, j.add, j.add_row, j.out, j.out_row};
    tiles += (j.N + 63) / 64;
  }
  if (tokens > (1LL << 31) || cdiv64(tokens, 64) * tiles > 0x7fffffffLL) {
    set_error("%s: too many tokens (%lld)", what, (long long)tokens);
    return kErrUnsupported;
  }
  gemm::project(js, count, tokens, rows_of_w != 0, dtype, (hipStream_t)stream);
  return check_launch(what);
}

int fbla_norm_leaky(const fbla_norm* jobs, int count, int64_t tokens, int C, int dtype, void* stream) {
  const char* what = "fbla_norm_leaky";
  if (!jobs || count < 1 || count > 2 || tokens < 0 || C < 8) {
    set_error("%s: bad sizes (count=%d tokens=%lld C=%d)", what, count, (long long)tokens, C);
    return kErrBadArg;
  }
  if ((dtype != kF16 && dtype != kBF16) || C % 8 || C > 2048 || tokens > 1LL << 30) {
    set_error("%s: fp16 and bf16 rows of whole 16-byte pieces, at most 2048 channels (dtype=%d C=%d tokens=%lld)", what, dtype, C,
              (long long)tokens);
    return kErrUnsupported;
  }
  if (tokens == 0) return kOk;
  gemm::NormJob js[2];
  for (int i = 0; i < count; ++i) {
    const fbla_norm& j = jobs[i];
    if (!j.x || !j.out || !j.mean != !j.rstd) {
      set_error("%s: null tensor pointer", what);
      return kErrBadArg;
    }
    if (check_aligned(what, {j.x, j.weight, j.bias, j.out}) != kOk) return kErrBadArg;
    js[i] = {j.x, j.weight, j.bias, j.out, j.mean, j.rstd, j.eps, j.slope};
  }
  gemm::norm_leaky(js, count, tokens, C, dtype, (hipStream_t)stream);
  return check_launch(what);
}

// what: 0 forward, 1 backward over the queries, 2 over the keys
static int block_attn(const char* name, const fbla_block_attn* p, int what, rows::Attn& a) {
  if (!p || (p->kind != 0 && p->kind != 1) || p->B < 1 || p->N < 1 || p->Nk < 1 || p->heads < 1) {
    set_error("%s: bad sizes or kind", name);
    return kErrBadArg;
  }
  const bool pola = p->kind == 0;
  const int64_t n = p->N > p->Nk ? p->N : p->Nk, C = (int64_t)p->heads * 32;
  if ((p->dtype != kF16 && p->dtype != kBF16) || p->B > 65535 || p->heads > 2048 || n > (1 << 24) || (int64_t)p->B * n * C > 1LL << 40 ||
      (!pola && p->N != p->Nk)) {
    set_error("%s: fp16 / bf16, at most 65535 batches, 2048 heads and 2^24 tokens, as many keys as queries for kind 1", name);
    return kErrUnsupported;
  }
  auto need = [&](std::initializer_list<const void*> ptrs) -> int {
    for (const void* q : ptrs)
      if (!q) {
        set_error("%s: null tensor pointer", name);
        return kErrBadArg;
      }
    return check_aligned(name, ptrs);
  };
  int rc = need({p->q, p->k, p->v, p->state_planes, p->state_km, p->workspace});
  if (rc == kOk && pola) rc = need({p->pe, p->scale, p->power});
  if (rc == kOk && !pola) rc = need({p->rot});
  if (rc == kOk && (what == 0 || pola)) rc = need({p->local});
  if (rc == kOk && pola) rc = need({p->gate});
  if (rc == kOk && what == 0) rc = need({p->out});
  if (rc == kOk && what == 1) rc = need({p->dout, p->dq});
  if (rc == kOk && what == 1 && pola) rc = need({p->dlocal, p->dgate});
  if (rc == kOk && what == 2) rc = need({p->dk, p->dv, p->dv_more});
  if (rc == kOk && what == 2 && pola) rc = need({p->dpe, p->dscale, p->dpower});
  if (rc == kOk) rc = check_row_strides(name, (int)C, p->dtype, {p->q_row, p->k_row, p->v_row});
  if (rc == kOk && pola) rc = check_row_strides(name, (int)C, p->dtype, {p->gate_row});
  if (rc == kOk && what == 1) rc = check_row_strides(name, (int)C, p->dtype, {p->dq_row});
  if (rc == kOk && what == 1 && pola) rc = check_row_strides(name, (int)C, p->dtype, {p->dgate_row});
  if (rc == kOk && what == 2) rc = check_row_strides(name, (int)C, p->dtype, {p->dk_row, p->dv_row});
  if (rc != kOk) return rc;
  for (int64_t row : {p->q_row, p->k_row, p->v_row, p->gate_row, p->dq_row, p->dk_row, p->dv_row, p->dgate_row})
    if (row > 1 << 22) {  // (32-bit offsets within a tile's rows)
      set_error("%s: rows too long (%lld elements)", name, (long long)row);
      return kErrUnsupported;
    }
  a = {pola, p->B, p->N, p->Nk, p->heads, p->eps, p->q, p->k, p->v, p->local, p->gate, p->q_row, p->k_row, p->v_row, p->gate_row, p->pe,
       p->scale, p->power, p->alpha, p->rot, p->out, p->state_planes, p->state_km, p->dout, p->dv_more, p->dq, p->dk, p->dv, p->dlocal, p->dgate,
       p->dq_row, p->dk_row, p->dv_row, p->dgate_row, p->dpe, p->dscale, p->dpower, p->workspace};
  if (p->workspace_bytes < rows::workspace_bytes(a)) {
    set_error("%s: workspace too small (%zu < %zu bytes)", name, p->workspace_bytes, rows::workspace_bytes(a));
    return kErrWorkspace;
  }
  return kOk;
}

size_t fbla_block_attn_workspace_bytes(int kind, int64_t B, int64_t N, int64_t Nk, int heads) {
  if (B < 1 || N < 1 || Nk < 1 || heads < 1 || B > 65535 || N > 1 << 24 || Nk > 1 << 24 || heads > 2048) return 0;
  rows::Attn a{};
  a.pola = kind == 0;
  a.B = (int)B, a.N = (int)N, a.Nk = (int)Nk, a.heads = heads;
  return rows::workspace_bytes(a);
}
size_t fbla_block_attn_state_elements(int kind, int64_t B, int heads) {
  rows::Attn a{};
  a.pola = kind == 0;
  a.B = (int)B, a.heads = heads;
  return B < 1 || heads < 1 ? 0 : rows::planes_elements(a);
}
int fbla_block_attn_forward(const fbla_block_attn* p, void* stream) {
  const char* name = "fbla_block_attn_forward";
  rows::Attn a;
  const int rc = block_attn(name, p, 0, a);
  if (rc != kOk) return rc;
  rows::forward(a, p->dtype, (hipStream_t)stream);
  return check_launch(name);
}
int fbla_block_attn_backward_queries(const fbla_block_attn* p, void* stream) {
  const char* name = "fbla_block_attn_backward_queries";
  rows::Attn a;
  int rc = block_attn(name, p, 1, a);
  if (rc == kOk) rc = rows::backward_queries(a, p->dtype, (hipStream_t)stream);
  return rc != kOk ? rc : check_launch(name);
}
int fbla_block_attn_backward_keys(const fbla_block_attn* p, void* stream) {
  const char* name = "fbla_block_attn_backward_keys";
  rows::Attn a;
  const int rc = block_attn(name, p, 2, a);
  if (rc != kOk) return rc;
  rows::backward_keys(a, p->dtype, (hipStream_t)stream);
  return check_launch(name);
}

static int check_blocks(const char* what, blocks::Shape& s, int64_t B, int64_t N, int64_t Nk, int heads, int d, int unit,
                        int dtype) {
  if (B < 1 || N < 1 || Nk < 1 || heads < 1 || d < 1 || (dtype != kF16 && dtype != kBF16 && dtype != kF32)) {
    set_error("%s: bad sizes or dtype (B=%lld N=%lld Nk=%lld heads=%d d=%d dtype=%d)", what, (long long)B, (long long)N,
              (long long)Nk, heads, d, dtype);
    return kErrBadArg;
  }
  const int64_t n = N > Nk ? N : Nk;
  if (d % (unit * blocks::vec_of(dtype)) || heads > (1 << 20) / d || n > 0x7fffffffLL / B ||
      B * n > 0x7fffffffLL / ((int64_t)heads * d / blocks::vec_of(dtype))) {
    set_error("%s: needs head dims of whole 16-byte pieces, at most 2^20 channels and 2^31 pieces "
              "(B=%lld N=%lld Nk=%lld heads=%d d=%d dtype=%d)", what, (long long)B, (long long)N, (long long)Nk, heads, d, dtype);
    return kErrUnsupported;
  }
  s = {(int)B, (int)N, (int)Nk, heads, d};
  return kOk;
}
static int check_tensors(const char* what, std::initializer_list<const void*> ptrs) {
  for (const void* p : ptrs)
    if (!p) {
      set_error("%s: null tensor pointer", what);
      return kErrBadArg;
    }
  return check_aligned(what, ptrs);
}

int fbla_polarity_fwd(const void* qg, const void* kv, const void* pe, const void* scale, const void* power, void* q_same,
                      void* q_opp, void* k_both, void* v_heads, int64_t B, int64_t N, int64_t Nk, int heads, int d, int dtype,
                      void* stream) {
  const char* what = "fbla_polarity_fwd";
  blocks::Shape s;
  int rc = check_blocks(what, s, B, N, Nk, heads, d, 1, dtype);
  if (rc == kOk) rc = check_tensors(what, {qg, kv, pe, scale, power, q_same, q_opp, k_both, v_heads});
  if (rc != kOk) return rc;
  blocks::polarity_fwd(s, {qg, kv, pe, scale, power}, q_same, q_opp, k_both, v_heads, dtype, (hipStream_t)stream);
  return check_launch(what);
}

size_t fbla_polarity_bwd_workspace_bytes(int64_t B, int64_t N, int64_t Nk, int heads, int d, int dtype) {
  blocks::Shape s;
  if (check_blocks("fbla_polarity_bwd_workspace_bytes", s, B, N, Nk, heads, d, 1, dtype) != kOk) return 0;
  return blocks::polarity_bwd_workspace_bytes(s, dtype);
}

int fbla_polarity_bwd(const void* qg, const void* kv, const void* pe, const void* scale, const void* power,
                      const void* dq_same, const void* dq_opp, const void* dk_both, const void* dv_heads, const void* dv_rows,
                      const void* dgate, void* dqg, void* dkv, void* dpe, void* dscale, void* dpower, void* workspace,
                      size_t workspace_bytes, int64_t B, int64_t N, int64_t Nk, int heads, int d, int dtype, void* stream) {
  const char* what = "fbla_polarity_bwd";
  blocks::Shape s;
  int rc = check_blocks(what, s, B, N, Nk, heads, d, 1, dtype);
  if (rc == kOk)
    rc = check_tensors(what, {qg, kv, pe, scale, power, dq_same, dq_opp, dk_both, dv_heads, dv_rows, dgate, dqg, dkv, dpe,
                              dscale, dpower, workspace});
  if (rc != kOk) return rc;
  const size_t need = blocks::polarity_bwd_workspace_bytes(s, dtype);
  if (workspace_bytes < need) {
    set_error("%s: workspace too small (%zu < %zu bytes)", what, workspace_bytes, need);
    return kErrWorkspace;
  }
  blocks::polarity_bwd(s, {qg, kv, pe, scale, power}, {dq_same, dq_opp, dk_both, dv_heads, dv_rows, dgate}, dqg, dkv, dpe,
                       dscale, dpower, (float*)workspace, dtype, (hipStream_t)stream);
  return check_launch(what);
}

static int check_rotation(const char* what, int rot_channels, int heads, int d, int dtype) {
  if (rot_channels < 1 || (heads * d) % rot_channels || rot_channels % blocks::vec_of(dtype)) {
    set_error("%s: the rotation's channels must be whole 16-byte pieces and divide the tokens' (%d, %d)", what, rot_channels,
              heads * d);
    return kErrBadArg;
  }
  return kOk;
}

int fbla_rotary_fwd(const void* qk, const void* x, const float* rot, int rot_channels, void* q, void* k, void* q_rot,
                    void* k_rot, void* v, int64_t B, int64_t N, int heads, int d, int dtype, void* stream) {
  const char* what = "fbla_rotary_fwd";
  blocks::Shape s;
  int rc = check_blocks(what, s, B, N, N, heads, d, 1, dtype);
  if (rc == kOk) rc = check_rotation(what, rot_channels, heads, d, dtype);
  if (rc == kOk) rc = check_tensors(what, {qk, x, rot, q, k, q_rot, k_rot, v});
  if (rc != kOk) return rc;
  blocks::rotary_fwd(s, qk, x, rot, rot_channels, q, k, q_rot, k_rot, v, dtype, (hipStream_t)stream);
  return check_launch(what);
}

int fbla_rotary_bwd(const void* qk, const float* rot, int rot_channels, const void* dq, const void* dk, const void* dq_rot,
                    const void* dk_rot, const void* dv, const void* dv_rows, void* dqk, void* dx, int64_t B, int64_t N,
                    int heads, int d, int dtype, void* stream) {
  const char* what = "fbla_rotary_bwd";
  blocks::Shape s;
  int rc = check_blocks(what, s, B, N, N, heads, d, 1, dtype);
  if (rc == kOk) rc = check_rotation(what, rot_channels, heads, d, dtype);
  if (rc == kOk) rc = check_tensors(what, {qk, rot, dq, dk, dq_rot, dk_rot, dv, dv_rows, dqk, dx});
  if (rc != kOk) return rc;
  blocks::rotary_bwd(s, qk, rot, rot_channels, {dq, dk, dq_rot, dk_rot, dv, dv_rows}, dqk, dx, dtype, (hipStream_t)stream);
  return check_launch(what);
}

static int check_merge(const char* what, blocks::Shape& s, const void* o2, const void* gate, int64_t gate_row, int64_t B,
                       int64_t N, int heads, int d, int dtype) {
  int rc = check_blocks(what, s, B, N, N, heads, d, o2 ? 2 : 1, dtype);
  if (rc == kOk && gate) rc = check_row_strides(what, heads * d, dtype, {gate_row});
  if (rc == kOk) rc = check_aligned(what, {o2, gate});
  return rc;
}

int fbla_merge_fwd(const void* o, const void* o2, const void* local, const void* gate, int64_t gate_row, void* out, int64_t B,
                   int64_t N, int heads, int d, int dtype, void* stream) {
  const char* what = "fbla_merge_fwd";
  blocks::Shape s;
  int rc = check_merge(what, s, o2, gate, gate_row, B, N, heads, d, dtype);
  if (rc == kOk) rc = check_tensors(what, {o, local, out});
  if (rc != kOk) return rc;
  blocks::merge_fwd(s, {o, o2, local, gate, gate_row}, out, dtype, (hipStream_t)stream);
  return check_launch(what);
}

int fbla_merge_bwd(const void* dout, const void* o, const void* o2, const void* local, const void* gate, int64_t gate_row,
                   void* d_o, void* d_o2, void* dlocal, void* dgate, int64_t B, int64_t N, int heads, int d, int dtype,
                   void* stream) {
  const char* what = "fbla_merge_bwd";
  blocks::Shape s;
  int rc = check_merge(what, s, d_o2, gate, gate_row, B, N, heads, d, dtype);
  if (rc == kOk) rc = check_tensors(what, {dout, d_o});
  if (rc == kOk && gate) rc = check_tensors(what, {o, local, dlocal, dgate});
  if (rc != kOk) return rc;
  if (gate && !o2 != !d_o2) {
    set_error("%s: one or two tensors of heads, on both sides alike", what);
    return kErrBadArg;
  }
  blocks::merge_bwd(s, {o, o2, local, gate, gate_row}, dout, d_o, d_o2, dlocal, dgate, dtype, (hipStream_t)stream);
  return check_launch(what);
}

static int check_interpolate(const char* what, int64_t B, int64_t from, int64_t to, int C, int dtype) {
  blocks::Shape s;
  const int rc = check_blocks(what, s, B, from, to, 1, C, 1, dtype);
  if (rc == kOk && from * to >= (1 << 28)) {  // the places are whole numbers of 32 bits
    set_error("%s: too many tokens (%lld to %lld)", what, (long long)from, (long long)to);
    return kErrUnsupported;
  }
  return rc;
}

int fbla_interpolate_fwd(const void* x, int64_t x_batch, int64_t x_row, void* y, int64_t B, int64_t from, int64_t to, int C,
                         int dtype, void* stream) {
  const char* what = "fbla_interpolate_fwd";
  int rc = check_interpolate(what, B, from, to, C, dtype);
  if (rc == kOk) rc = check_tensors(what, {x, y});
  if (rc == kOk) rc = check_row_strides(what, C, dtype, {x_batch, x_row});
  if (rc != kOk) return rc;
  blocks::interpolate_fwd(x, x_batch, x_row, (int)B, (int)from, (int)to, C, y, dtype, (hipStream_t)stream);
  return check_launch(what);
}

int fbla_interpolate_bwd(const void* g, void* dx, int64_t B, int64_t from, int64_t to, int C, int dtype, void* stream) {
  const char* what = "fbla_interpolate_bwd";
  int rc = check_interpolate(what, B, from, to, C, dtype);
  if (rc == kOk) rc = check_tensors(what, {g, dx});
  if (rc != kOk) return rc;
  blocks::interpolate_bwd(g, (int)B, (int)from, (int)to, C, dx, dtype, (hipStream_t)stream);
  return check_launch(what);
}

static int check_row(const char* what, int C, int dtype) {
  if (C > blocks::most_row_channels(dtype)) {
    set_error("%s: at most %d channels (got %d)", what, blocks::most_row_channels(dtype), C);
    return kErrUnsupported;
  }
  return kOk;
}

int fbla_focus_fwd(const void* q, const void* kv, const void* pe, const void* scale, void* q_out, void* k_out, void* v_out,
                   int64_t B, int64_t N, int64_t Nk, int heads, int d, int dtype, void* stream) {
  const char* what = "fbla_focus_fwd";
  blocks::Shape s;
  int rc = check_blocks(what, s, B, N, Nk, heads, d, 1, dtype);
  if (rc == kOk) rc = check_row(what, heads * d, dtype);
  if (rc == kOk) rc = check_tensors(what, {q, kv, pe, scale, q_out, k_out, v_out});
  if (rc != kOk) return rc;
  blocks::focus_fwd(s, {q, kv, pe, scale}, q_out, k_out, v_out, dtype, (hipStream_t)stream);
  return check_launch(what);
}

size_t fbla_focus_bwd_workspace_bytes(int64_t B, int64_t N, int64_t Nk, int heads, int d, int dtype) {
  const char* what = "fbla_focus_bwd_workspace_bytes";
  blocks::Shape s;
  if (check_blocks(what, s, B, N, Nk, heads, d, 1, dtype) != kOk || check_row(what, heads * d, dtype) != kOk) return 0;
  return blocks::focus_bwd_workspace_bytes(s, dtype);
}

int fbla_focus_bwd(const void* q, const void* kv, const void* pe, const void* scale, const void* dq_heads,
                   const void* dk_heads, const void* dv_heads, const void* dv_rows, void* dq, void* dkv, void* dpe,
                   void* dscale, void* workspace, size_t workspace_bytes, int64_t B, int64_t N, int64_t Nk, int heads, int d,
                   int dtype, void* stream) {
  const char* what = "fbla_focus_bwd";
  blocks::Shape s;
  int rc = check_blocks(what, s, B, N, Nk, heads, d, 1, dtype);
  if (rc == kOk) rc = check_row(what, heads * d, dtype);
  if (rc == kOk)
    rc = check_tensors(what, {q, kv, pe, scale, dq_heads, dk_heads, dv_heads, dv_rows, dq, dkv, dpe, dscale, workspace});
  if (rc != kOk) return rc;
  const size_t need = blocks::focus_bwd_workspace_bytes(s, dtype);
  if (workspace_bytes < need) {
    set_error("%s: workspace too small (%zu < %zu bytes)", what, workspace_bytes, need);
    return kErrWorkspace;
  }
  blocks::focus_bwd(s, {q, kv, pe, scale}, {dq_heads, dk_heads, dv_heads, dv_rows}, dq, dkv, dpe, dscale, (float*)workspace,
                    dtype, (hipStream_t)stream);
  return check_launch(what);
}

static int check_turn(const char* what, blocks::Shape& s, int64_t B, int64_t N, int heads, int d, int dtype) {
  const int rc = check_blocks(what, s, B, N, N, heads, d, 1, dtype);
  const int pieces = rc == kOk ? d / blocks::vec_of(dtype) : 1;
  if (pieces > 64 || (pieces & (pieces - 1))) {
    set_error("%s: a head must be a power of two of at most 64 16-byte pieces (d=%d)", what, d);
    return kErrUnsupported;
  }
  return rc;
}

int fbla_turn_fwd(const void* q, const void* k, const void* weight, const float* rot, void* k_out, void* q_rot, void* k_rot,
                  int64_t B, int64_t N, int heads, int d, int dtype, void* stream) {
  const char* what = "fbla_turn_fwd";
  blocks::Shape s;
  int rc = check_turn(what, s, B, N, heads, d, dtype);
  if (rc == kOk) rc = check_tensors(what, {q, k, weight, rot, k_out, q_rot, k_rot});
  if (rc != kOk) return rc;
  blocks::turn_fwd(s, q, k, weight, rot, k_out, q_rot, k_rot, dtype, (hipStream_t)stream);
  return check_launch(what);
}

int fbla_turn_bwd(const void* k, const void* weight, const float* rot, const void* dk_out, const void* dq_rot,
                  const void* dk_rot, void* dq, void* dk, void* dweight, int64_t B, int64_t N, int heads, int d, int dtype,
                  void* stream) {
  const char* what = "fbla_turn_bwd";
  blocks::Shape s;
  int rc = check_turn(what, s, B, N, heads, d, dtype);
  if (rc == kOk) rc = check_tensors(what, {k, weight, rot, dk_out, dq_rot, dk_rot, dq, dk, dweight});
  if (rc != kOk) return rc;
  blocks::turn_bwd(s, k, weight, rot, dk_out, dq_rot, dk_rot, dq, dk, dweight, dtype, (hipStream_t)stream);
  return check_launch(what);
}

}  // extern "C"
