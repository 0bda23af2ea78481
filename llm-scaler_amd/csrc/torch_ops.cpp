// The hot ops' host path in C++: operand checks, workspace, stream and the call of the C ABI, registered for the
// CUDA dispatch key (which ROCm tensors use) of the operators that mi355x_qlinear/ops.py declares.  A decode step's
// kernels take 4-13 us; the same path in Python takes 12-18 us of host time per call and was what a chain of calls
// waited for (INT4 4096 x 4096, one row: 14.2 us per call for a kernel of 5).
//
// A function here takes a call when every operand is as the kernels want it.  Any other call - a wrong type, size
// or device, a non-contiguous operand, a form that needs preparation - goes to the Python implementation of the same
// operator (registered as mi355x_checked::<name>), which runs it or raises, so that accepted calls, results and
// error messages are those of that implementation.  Only the checks decide that, before anything is enqueued: once an
// entry of the C ABI has been called, a status other than 0 is raised.  Running the call again would hide a launch that
// failed and would add to an in-place operand twice (the residual of the norm operators).
#include <ATen/core/dispatch/Dispatcher.h>
#include <ATen/core/stack.h>
#include <ATen/hip/impl/HIPStreamMasqueradingAsCUDA.h>
#include <ATen/ops/empty.h>
#include <c10/core/DeviceGuard.h>
#include <torch/library.h>

#include <algorithm>
#include <climits>
#include <initializer_list>

#include "../../include/mi355x_qlinear.h"

namespace {

using at::Tensor;

// The operator's Python implementation, called on the CUDA key directly (the dispatcher is already past the others).
template <class... A>
Tensor checked(const c10::OperatorHandle& op, const A&... args) {
  torch::jit::Stack stack;
  torch::jit::push(stack, args...);
  op.redispatchBoxed(c10::DispatchKeySet(c10::DispatchKey::CUDA), &stack);
  return stack.back().toTensor();
}
#define CHECKED(name, ...)                                                                                  \
  do {                                                                                                      \
    static const c10::OperatorHandle op = c10::Dispatcher::singleton().findSchemaOrThrow("mi355x_checked::" name, ""); \
    return checked(op, __VA_ARGS__);                                                                        \
  } while (0)

// Raises what the Python implementations raise for the same status.
void status(const char* entry, int rc) {
  if (rc == 0) return;
  const char* why = rc == -1 ? "invalid argument (null pointer or bad enum)"
                    : rc == -2 ? "unsupported shape or divisibility"
                    : rc == -3 ? "kernel launch failed" : nullptr;
  if (why) TORCH_CHECK(false, entry, " failed: ", why);
  TORCH_CHECK(false, entry, " failed: ", rc);
}
#define CALL(entry, ...) status(#entry, entry(__VA_ARGS__))

// on x's device, contiguous, strided
bool plain(const Tensor& x, std::initializer_list<const Tensor*> ts) {
  if (!x.is_cuda() || !x.is_contiguous()) return false;
  for (const Tensor* t : ts)
    if (!t->is_cuda() || t->device() != x.device() || !t->is_contiguous()) return false;
  return true;
}
bool is16(const Tensor& t) { return t.scalar_type() == at::kHalf || t.scalar_type() == at::kBFloat16; }
bool is_fp8(const Tensor& t) { return t.scalar_type() == at::kFloat8_e4m3fn || t.scalar_type() == at::kByte; }
int act(const Tensor& t) { return t.scalar_type() == at::kHalf ? 0 : 1; }
bool fits(int64_t v) { return v > 0 && v <= INT_MAX; }
// rows of x over K, 0 when K does not divide it or a size does not fit the C ABI
int64_t rows_of(const Tensor& x, int64_t K) {
  if (!fits(K) || x.numel() % K) return 0;
  return fits(x.numel() / K) ? x.numel() / K : 0;
}

struct On {                                            // x's device and its current stream
  c10::DeviceGuard guard;
  void* stream;
  explicit On(const Tensor& x)
      : guard(x.device()), stream((void*)c10::hip::getCurrentHIPStreamMasqueradingAsCUDA(x.device().index()).stream()) {}
};
Tensor buffer(const Tensor& x, int64_t bytes) { return at::empty({bytes}, x.options().dtype(at::kByte)); }

constexpr int kMaxMat = 3;
// One linear layer call: up to three matrices over the same rows of x.
struct Linear {
  int n = 0, N[kMaxMat], M, K, adt;
  const void *w[kMaxMat], *s[kMaxMat];
  void* o[kMaxMat];
  void add(const Tensor& w_, const Tensor& s_, const Tensor& o_, int64_t N_) {
    w[n] = w_.data_ptr(); s[n] = s_.data_ptr(); o[n] = o_.data_ptr(); N[n++] = (int)N_;
  }
  bool prefill() const { return M > 64 && K % 128 == 0; }
  Tensor workspace(const Tensor& x, long long& bytes) const {
    long long need = 0;
    bytes = 0;
    for (int i = 0; i < n; ++i) {
      CALL(mi_gemm_tiled_workspace_split, M, N[i], K, &need);
      bytes = std::max(bytes, need);
    }
    return buffer(x, bytes);
  }
};

// ---------------------------------------------------------------------------------------- FP8
enum Scale { kPern = 0, kPert = 1, kBlock = 2 };

void run_fp8(const Tensor& x, Linear& l, Scale mode, bool scale_f16) {
  const On on(x);
  const void* xp = x.data_ptr();
  if (l.prefill()) {
    long long bytes;
    const Tensor ws = l.workspace(x, bytes);
    for (int i = 0; i < l.n; ++i)
      CALL(mi_gemm_fp8_tiled_ws, xp, l.w[i], l.s[i], mode, scale_f16, l.o[i], ws.data_ptr(), bytes, l.M, l.N[i], l.K, l.adt,
           on.stream);
    return;
  }
  const float* const* s = reinterpret_cast<const float* const*>(l.s);
  if (mode == kPern) CALL(mi_gemm_fp8_pern_multi, xp, l.n, l.w, l.s, l.o, l.N, l.M, l.K, l.adt, scale_f16, on.stream);
  else if (mode == kPert) CALL(mi_gemm_fp8_pert_multi, xp, l.n, l.w, s, l.o, l.N, l.M, l.K, l.adt, on.stream);
  else CALL(mi_gemm_fp8_blockscale_multi, xp, l.n, l.w, s, l.o, l.N, l.M, l.K, l.adt, on.stream);
}

struct Mat { const Tensor &w, &s, &o; int64_t N; };    // N < 0: the weight's rows

bool fp8_linear(const Tensor& x, std::initializer_list<Mat> mats, int64_t K, Scale mode) {
  const Tensor& w0 = mats.begin()->w;
  if (mode != kPern) {
    if (w0.dim() != 2) return false;
    K = w0.size(1);
  }
  Linear l;
  const int64_t M = rows_of(x, K);
  if (!M || !is16(x) || (mode == kBlock && (x.dim() != 2 || x.size(1) != K || K % 128))) return false;
  l.M = (int)M; l.K = (int)K; l.adt = act(x);
  const auto sdt = mats.begin()->s.scalar_type();
  if (mode == kPern ? sdt != at::kHalf && sdt != at::kFloat : sdt != at::kFloat) return false;
  for (const Mat& m : mats) {
    const int64_t N = m.N < 0 ? (m.w.dim() == 2 ? m.w.size(0) : 0) : m.N;
    if (!plain(x, {&m.w, &m.s, &m.o}) || !fits(N) || !is_fp8(m.w) || m.w.numel() != N * K || m.s.scalar_type() != sdt ||
        m.o.scalar_type() != x.scalar_type() || m.o.numel() != M * N)
      return false;
    if (mode == kPern ? m.s.numel() != N : m.w.dim() != 2 || m.w.size(1) != K) return false;
    if (mode == kPert && m.s.numel() < 1) return false;
    if (mode == kBlock && (m.s.dim() != 2 || m.s.size(0) != (N + 127) / 128 || m.s.size(1) != K / 128)) return false;
    l.add(m.w, m.s, m.o, N);
  }
  run_fp8(x, l, mode, sdt == at::kHalf);
  return true;
}

#define FP8_PERN(name)                                                                                        \
  Tensor name(const Tensor& x, const Tensor& w, const Tensor& s, const Tensor& o, int64_t N, int64_t K) {     \
    if (N >= 0 && fp8_linear(x, {{w, s, o, N}}, K, kPern)) return o;                                          \
    CHECKED(#name, x, w, s, o, N, K);                                                                         \
  }
FP8_PERN(esimd_gemv_fp8_pern)
Tensor esimd_gemv_fp8_pern_fused2(const Tensor& x, const Tensor& w0, const Tensor& s0, const Tensor& o0, int64_t N0,
                                  const Tensor& w1, const Tensor& s1, const Tensor& o1, int64_t N1, int64_t K) {
  if (N0 >= 0 && N1 >= 0 && fp8_linear(x, {{w0, s0, o0, N0}, {w1, s1, o1, N1}}, K, kPern)) return o0;
  CHECKED("esimd_gemv_fp8_pern_fused2", x, w0, s0, o0, N0, w1, s1, o1, N1, K);
}
Tensor esimd_gemv_fp8_pern_fused3(const Tensor& x, const Tensor& w0, const Tensor& s0, const Tensor& o0, int64_t N0,
                                  const Tensor& w1, const Tensor& s1, const Tensor& o1, int64_t N1, const Tensor& w2,
                                  const Tensor& s2, const Tensor& o2, int64_t N2, int64_t K) {
  if (N0 >= 0 && N1 >= 0 && N2 >= 0 && fp8_linear(x, {{w0, s0, o0, N0}, {w1, s1, o1, N1}, {w2, s2, o2, N2}}, K, kPern))
    return o0;
  CHECKED("esimd_gemv_fp8_pern_fused3", x, w0, s0, o0, N0, w1, s1, o1, N1, w2, s2, o2, N2, K);
}
#define FP8_PERT(name)                                                                       \
  Tensor name(const Tensor& x, const Tensor& w, const Tensor& s, const Tensor& o) {          \
    if (fp8_linear(x, {{w, s, o, -1}}, 0, kPert)) return o;                                  \
    CHECKED(#name, x, w, s, o);                                                              \
  }
FP8_PERT(esimd_gemv_fp8_pert)
FP8_PERT(esimd_gemv_fp8_pert_bmg)
FP8_PERT(esimd_gemm_fp8_pert)
Tensor esimd_gemv_fp8_pert_fused2(const Tensor& x, const Tensor& w0, const Tensor& s0, const Tensor& o0, const Tensor& w1,
                                  const Tensor& s1, const Tensor& o1) {
  if (fp8_linear(x, {{w0, s0, o0, -1}, {w1, s1, o1, -1}}, 0, kPert)) return o0;
  CHECKED("esimd_gemv_fp8_pert_fused2", x, w0, s0, o0, w1, s1, o1);
}
Tensor esimd_gemv_fp8_pert_fused3(const Tensor& x, const Tensor& w0, const Tensor& s0, const Tensor& o0, const Tensor& w1,
                                  const Tensor& s1, const Tensor& o1, const Tensor& w2, const Tensor& s2, const Tensor& o2) {
  if (fp8_linear(x, {{w0, s0, o0, -1}, {w1, s1, o1, -1}, {w2, s2, o2, -1}}, 0, kPert)) return o0;
  CHECKED("esimd_gemv_fp8_pert_fused3", x, w0, s0, o0, w1, s1, o1, w2, s2, o2);
}
Tensor esimd_gemm_fp8_blockscale(const Tensor& x, const Tensor& w, const Tensor& s, const Tensor& o, int64_t bn, int64_t bk) {
  if (bn == 128 && bk == 128 && fp8_linear(x, {{w, s, o, -1}}, 0, kBlock)) return o;
  CHECKED("esimd_gemm_fp8_blockscale", x, w, s, o, bn, bk);
}
Tensor esimd_gemv_fp8_blockscale_fused2(const Tensor& x, const Tensor& w0, const Tensor& s0, const Tensor& o0, const Tensor& w1,
                                        const Tensor& s1, const Tensor& o1, int64_t bn, int64_t bk) {
  if (bn == 128 && bk == 128 && fp8_linear(x, {{w0, s0, o0, -1}, {w1, s1, o1, -1}}, 0, kBlock)) return o0;
  CHECKED("esimd_gemv_fp8_blockscale_fused2", x, w0, s0, o0, w1, s1, o1, bn, bk);
}

// ---------------------------------------------------------------------------------------- INT4 group 128
// K of an int4 weight given as uint8 [N, K/2] or int32 [N, K/8]; 0 for anything else
int64_t int4_k(const Tensor& w) {
  if (w.dim() != 2) return 0;
  return w.scalar_type() == at::kByte ? w.size(1) * 2 : w.scalar_type() == at::kInt ? w.size(1) * 8 : 0;
}
bool int4_linear(const Tensor& x, std::initializer_list<Mat> mats, const Tensor* zp, bool gemm) {
  const int64_t K = int4_k(mats.begin()->w), M = rows_of(x, K);
  if (!M || K % 128 || !is16(x)) return false;
  Linear l;
  l.M = (int)M; l.K = (int)K; l.adt = act(x);
  for (const Mat& m : mats) {
    if (int4_k(m.w) != K || !plain(x, {&m.w, &m.s, &m.o})) return false;
    const int64_t N = m.w.size(0);
    if (!fits(N) || m.s.scalar_type() != at::kHalf || m.s.numel() != N * (K / 128) ||
        m.o.scalar_type() != x.scalar_type() || m.o.numel() != M * N)
      return false;
    if (zp && (zp->scalar_type() != at::kByte || !plain(x, {zp}) || zp->numel() != N * (K / 128))) return false;
    l.add(m.w, m.s, m.o, N);
  }
  const On on(x);
  if (!gemm) {
    CALL(mi_gemv_int4_multi, x.data_ptr(), l.n, l.w, l.s, nullptr, l.o, l.N, l.M, l.K, l.adt, on.stream);
    return true;
  }
  long long bytes = 0;
  Tensor ws;
  if (l.prefill()) ws = l.workspace(x, bytes);
  CALL(mi_gemm_int4_ws, x.data_ptr(), l.w[0], l.s[0], zp ? zp->data_ptr() : nullptr, l.o[0], bytes ? ws.data_ptr() : nullptr, bytes,
       l.M, l.N[0], l.K, l.adt, on.stream);
  return true;
}
Tensor esimd_gemv_int4(const Tensor& x, const Tensor& w, const Tensor& s, const Tensor& o) {
  if (int4_linear(x, {{w, s, o, -1}}, nullptr, false)) return o;
  CHECKED("esimd_gemv_int4", x, w, s, o);
}
Tensor esimd_gemv_int4_fused2(const Tensor& x, const Tensor& w0, const Tensor& s0, const Tensor& o0, const Tensor& w1,
                              const Tensor& s1, const Tensor& o1) {
  if (int4_linear(x, {{w0, s0, o0, -1}, {w1, s1, o1, -1}}, nullptr, false)) return o0;
  CHECKED("esimd_gemv_int4_fused2", x, w0, s0, o0, w1, s1, o1);
}
Tensor esimd_gemm_int4_pgrp(const Tensor& x, const Tensor& w, const Tensor& s, const Tensor& o) {
  if (int4_linear(x, {{w, s, o, -1}}, nullptr, true)) return o;
  CHECKED("esimd_gemm_int4_pgrp", x, w, s, o);
}
Tensor esimd_gemm_int4_pgrp_zp(const Tensor& x, const Tensor& w, const Tensor& s, const Tensor& z, const Tensor& o) {
  if (int4_linear(x, {{w, s, o, -1}}, &z, true)) return o;
  CHECKED("esimd_gemm_int4_pgrp_zp", x, w, s, z, o);
}

// ---------------------------------------------------------------------------------------- GGUF
enum Gguf { kQ4K = 2, kQ40 = 3, kQ80 = 4, kQ5K = 5, kQ6K = 6 };   // the format numbers of mi_gemm_gguf_tiled_pays

bool gguf_tiled(int fmt, const Linear& l) {
  int pays = 0;
  CALL(mi_gemm_gguf_tiled_pays, fmt, l.M, l.N[0], l.K, &pays);
  return pays;
}
bool gguf_linear(int fmt, const Tensor& x, const Tensor& w, const Tensor* qh, const Tensor& s, const Tensor* mn, const Tensor& o) {
  if (w.dim() != 2 || !plain(x, {&w, &s, &o}) || (qh && !plain(x, {qh})) || (mn && !plain(x, {mn}))) return false;
  if (fmt == kQ80 ? w.scalar_type() != at::kChar && w.scalar_type() != at::kByte : w.scalar_type() != at::kByte) return false;
  const int64_t N = w.size(0), K = w.size(1) * (fmt == kQ80 ? 1 : 2), M = rows_of(x, K);
  const int64_t scales = N * (K / (fmt == kQ6K ? 16 : 32));
  if (!M || !fits(N) || K % (fmt == kQ5K || fmt == kQ6K ? 512 : 32)) return false;
  if (x.scalar_type() != at::kHalf || o.scalar_type() != at::kHalf || o.numel() != M * N) return false;
  if (s.scalar_type() != at::kHalf || s.numel() != scales) return false;
  if (mn && (mn->scalar_type() != at::kHalf || mn->numel() != scales)) return false;
  if (qh && (qh->scalar_type() != at::kByte || qh->dim() != 2 || qh->size(0) != N || qh->size(1) != K / (fmt == kQ6K ? 4 : 8)))
    return false;
  Linear l;
  l.M = (int)M; l.K = (int)K; l.adt = 0;
  l.add(w, s, o, N);
  const On on(x);
  const void *xp = x.data_ptr(), *hp = qh ? qh->data_ptr() : nullptr, *mp = mn ? mn->data_ptr() : nullptr;
  if (gguf_tiled(fmt, l)) {
    long long bytes;
    const Tensor ws = l.workspace(x, bytes);
    if (fmt == kQ4K) CALL(mi_gemm_q4k_tiled_ws, xp, l.w[0], l.s[0], mp, l.o[0], ws.data_ptr(), bytes, l.M, l.N[0], l.K, on.stream);
    else CALL(mi_gemm_gguf_tiled_ws, fmt, xp, l.w[0], hp, l.s[0], mp, l.o[0], ws.data_ptr(), bytes, l.M, l.N[0], l.K, on.stream);
    return true;
  }
  switch (fmt) {
    case kQ4K: CALL(mi_gemv_q4k, xp, l.w[0], l.s[0], mp, l.o[0], l.M, l.N[0], l.K, on.stream); break;
    case kQ40: CALL(mi_gemv_q4_0, xp, l.w[0], l.s[0], l.o[0], l.M, l.N[0], l.K, on.stream); break;
    case kQ80: CALL(mi_gemv_q8_0, xp, l.w[0], l.s[0], l.o[0], l.M, l.N[0], l.K, on.stream); break;
    case kQ5K: CALL(mi_gemv_q5k, xp, l.w[0], hp, l.s[0], mp, l.o[0], l.M, l.N[0], l.K, on.stream); break;
    default: CALL(mi_gemv_q6k, xp, l.w[0], hp, l.s[0], l.o[0], l.M, l.N[0], l.K, on.stream);
  }
  return true;
}
Tensor esimd_gemv_q4_k(const Tensor& x, const Tensor& w, const Tensor& s, const Tensor& mn, const Tensor& o) {
  if (gguf_linear(kQ4K, x, w, nullptr, s, &mn, o)) return o;
  CHECKED("esimd_gemv_q4_k", x, w, s, mn, o);
}
#define GGUF_PLAIN(name, fmt)                                                                     \
  Tensor name(const Tensor& x, const Tensor& w, const Tensor& s, const Tensor& o) {               \
    if (gguf_linear(fmt, x, w, nullptr, s, nullptr, o)) return o;                                 \
    CHECKED(#name, x, w, s, o);                                                                   \
  }
GGUF_PLAIN(esimd_gemv_q4_0, kQ40)
GGUF_PLAIN(esimd_gemm_q4_0, kQ40)
GGUF_PLAIN(esimd_gemv_q8_0, kQ80)
GGUF_PLAIN(esimd_gemv_q8_0_m, kQ80)
Tensor esimd_gemv_q5_k(const Tensor& x, const Tensor& w, const Tensor& qh, const Tensor& s, const Tensor& mn, const Tensor& o) {
  if (gguf_linear(kQ5K, x, w, &qh, s, &mn, o)) return o;
  CHECKED("esimd_gemv_q5_k", x, w, qh, s, mn, o);
}
#define GGUF_Q6K(name)                                                                                   \
  Tensor name(const Tensor& x, const Tensor& w, const Tensor& qh, const Tensor& s, const Tensor& o) {    \
    if (gguf_linear(kQ6K, x, w, &qh, s, nullptr, o)) return o;                                           \
    CHECKED(#name, x, w, qh, s, o);                                                                      \
  }
GGUF_Q6K(esimd_gemv_q6_k)
GGUF_Q6K(esimd_gemv_q6_k_m)

// ---------------------------------------------------------------------------------------- norm + linear, one row
bool resadd_norm_gemv(bool int4, const Tensor& x, const Tensor& res, const Tensor& nw, const Tensor& w, const Tensor& s,
                      const Tensor& o, const Tensor& normed, double eps) {
  if (!plain(x, {&res, &nw, &w, &s, &o, &normed}) || !is16(x) || w.dim() != 2 || x.dim() < 1) return false;
  const auto dt = x.scalar_type();
  if (res.scalar_type() != dt || nw.scalar_type() != dt || o.scalar_type() != dt || normed.scalar_type() != dt) return false;
  const int64_t K = int4 ? int4_k(w) : w.size(1), N = w.size(0);
  if (!fits(K) || !fits(N) || x.numel() != K || x.size(-1) != K || res.numel() != K || nw.numel() != K || normed.numel() < K ||
      o.numel() != N)
    return false;
  if (int4 ? K % 128 || s.scalar_type() != at::kHalf || s.numel() != N * (K / 128)
           : !is_fp8(w) || s.scalar_type() != at::kFloat || s.numel() < 1)
    return false;
  const On on(x);
  const void *wp = w.data_ptr(), *sp = s.data_ptr();
  void* op = o.data_ptr();
  const int n = (int)N;
  CALL(mi_norm_gemv_scaled, x.data_ptr(), res.data_ptr(), nullptr, nw.data_ptr(), normed.data_ptr(), (int)K, (float)eps, 1.0f,
       int4 ? 2 : 0, 1, &wp, &sp, &op, &n, (int)K, act(x), on.stream);
  return true;
}
#define RESADD_NORM(name, int4)                                                                                        \
  Tensor name(const Tensor& x, const Tensor& res, const Tensor& nw, const Tensor& w, const Tensor& s, const Tensor& o, \
              const Tensor& normed, double eps) {                                                                      \
    if (resadd_norm_gemv(int4, x, res, nw, w, s, o, normed, eps)) return o;                                            \
    CHECKED(#name, x, res, nw, w, s, o, normed, eps);                                                                  \
  }
RESADD_NORM(esimd_resadd_norm_gemv_int4_pert, true)
RESADD_NORM(esimd_resadd_norm_gemv_fp8_pert, false)

// ---------------------------------------------------------------------------------------- MoE decode
bool shape_is(const Tensor& t, at::IntArrayRef s) { return t.sizes() == s; }

// Up to 96 (token, route) pairs: top-k with the shared expert's gate | gate_up rows of all routes and the shared expert | down rows, SiLU(gate) x up
// applied as they are staged | their weighted sum.  The first two and the last two are one launch each where the plan says so.  More
// pairs take Python's grouped path, which reads an expert once and rounds once between gate_up and down.
bool moe_full_decode(const Tensor& x, const Tensor& logits, const Tensor& out, const Tensor& w13, const Tensor& s13,
                     const Tensor& sw13, const Tensor& ss13, const Tensor& w2, const Tensor& s2, const Tensor& sw2,
                     const Tensor& ss2, const Tensor& gw, int64_t k, int64_t shared, int64_t E) {
  if (x.dim() != 2 || x.size(0) < 1 || w13.dim() != 3 || !is16(x) || shared != 1) return false;
  const int64_t T = x.size(0), H = x.size(1), I = w13.size(1) / 2, P = T * k;
  if (k < 1 || k > 64 || E < k || E > 1024 || P > INT32_MAX || H < 128 || I < 128 || H % 128 || I % 128 || w13.size(1) % 2)
    return false;
  if (!plain(x, {&logits, &out, &w13, &s13, &sw13, &ss13, &w2, &s2, &sw2, &ss2, &gw}) || out.data_ptr() == x.data_ptr()) return false;
  const auto dt = x.scalar_type();
  if (out.scalar_type() != dt || logits.scalar_type() != dt || gw.scalar_type() != dt) return false;
  for (const Tensor* w : {&w13, &sw13, &w2, &sw2})
    if (!is_fp8(*w)) return false;
  for (const Tensor* s : {&s13, &ss13, &s2, &ss2})
    if (s->scalar_type() != at::kFloat) return false;
  if (!shape_is(out, {T, H}) || !shape_is(logits, {T, E}) || !shape_is(w13, {E, 2 * I, H}) || !shape_is(w2, {E, H, I}) ||
      !shape_is(sw13, {2 * I, H}) || !shape_is(sw2, {H, I}) || !shape_is(s13, {E, 2 * I / 128, H / 128}) ||
      !shape_is(s2, {E, H / 128, I / 128}) || !shape_is(ss13, {2 * I / 128, H / 128}) || !shape_is(ss2, {H / 128, I / 128}) ||
      !shape_is(gw, {1, H}))
    return false;
  int plan = 0;
  if (H > INT32_MAX || I > INT32_MAX || mi_moe_decode_plan((int)T, (int)k, (int)E, (int)H, (int)I, &plan) != 0 ||
      !(plan & MI_DECODE_ROUTED))
    return false;
  const On on(x);
  const int adt = act(x);
  // one allocation: gate_up rows | down rows | routing weights | gates | expert ids, 256 bytes apart
  int64_t at_ = 0;
  auto take = [&](int64_t bytes) { const int64_t here = at_; at_ += (bytes + 255) / 256 * 256; return here; };
  const bool sum = plan & MI_DECODE_DOWN_SUM;         // the down launch adds the routes up itself
  const int64_t gu_at = take((P + T) * 2 * I * 2), y_at = take(sum ? 0 : (P + T) * H * 2), tw_at = take(P * 2), g_at = take(T * 4),
                id_at = take(P * 4);
  const Tensor ws = buffer(x, at_);
  char* base = (char*)ws.data_ptr();
  void *gu = base + gu_at, *y = sum ? nullptr : base + y_at, *tw = base + tw_at;
  float* gate = (float*)(base + g_at);
  int32_t* ids = (int32_t*)(base + id_at);
  const void* xp = x.data_ptr();
  void* st = on.stream;
  if (plan & MI_DECODE_GATE_UP_TOPK) {
    CALL(mi_moe_gate_up_topk_fp8_block, xp, logits.data_ptr(), gw.data_ptr(), w13.data_ptr(), s13.data_ptr<float>(), sw13.data_ptr(),
         ss13.data_ptr<float>(), gu, ids, tw, gate, (int)T, (int)k, (int)E, (int)H, (int)I, adt, st);
  } else {
    CALL(mi_moe_topk, logits.data_ptr(), tw, ids, (int)T, (int)E, (int)k, 1, nullptr, xp, gw.data_ptr(), gate, (int)H, adt, st);
    CALL(mi_moe_gemv_fp8_block_routed, xp, (int)k, 0, w13.data_ptr(), s13.data_ptr<float>(), gu, 2 * I, ids, nullptr, (int)P, (int)E,
         sw13.data_ptr(), ss13.data_ptr<float>(), (int)T, 0, (int)(2 * I), (int)H, adt, st);
  }
  if (sum) {
    CALL(mi_moe_down_sum_fp8_block, gu, w2.data_ptr(), s2.data_ptr<float>(), sw2.data_ptr(), ss2.data_ptr<float>(), ids, tw, gate,
         out.data_ptr(), (int)T, (int)k, (int)E, (int)H, (int)I, adt, st);
    return true;
  }
  CALL(mi_moe_gemv_fp8_block_routed, gu, 1, 1, w2.data_ptr(), s2.data_ptr<float>(), y, H, ids, tw, (int)P, (int)E, sw2.data_ptr(),
       ss2.data_ptr<float>(), (int)T, (int)P, (int)H, (int)I, adt, st);
  CALL(mi_moe_combine_shared, y, nullptr, nullptr, out.data_ptr(), (char*)y + P * H * 2, gate, (int)H, (int)k, (int)T, 0, adt, 0, st);
  return true;
}
Tensor moe_forward_full_fp8_block(const Tensor& x, const Tensor& logits, const Tensor& out, const Tensor& w13, const Tensor& s13,
                                  const Tensor& sw13, const Tensor& ss13, const Tensor& w2, const Tensor& s2, const Tensor& sw2,
                                  const Tensor& ss2, const Tensor& gw, int64_t k, int64_t shared, int64_t E) {
  if (moe_full_decode(x, logits, out, w13, s13, sw13, ss13, w2, s2, sw2, ss2, gw, k, shared, E)) return out;
  CHECKED("moe_forward_full_fp8_block", x, logits, out, w13, s13, sw13, ss13, w2, s2, sw2, ss2, gw, k, shared, E);
}

}  // namespace

#define IMPL(name) m.impl(#name, &name)
#define DECODE_OPS()                                                                                         \
  IMPL(esimd_gemv_fp8_pern); IMPL(esimd_gemv_fp8_pern_fused2); IMPL(esimd_gemv_fp8_pern_fused3);             \
  IMPL(esimd_gemv_fp8_pert); IMPL(esimd_gemv_fp8_pert_bmg); IMPL(esimd_gemv_fp8_pert_fused2);                \
  IMPL(esimd_gemv_fp8_pert_fused3); IMPL(esimd_gemv_int4); IMPL(esimd_gemv_int4_fused2);                     \
  IMPL(esimd_resadd_norm_gemv_int4_pert); IMPL(esimd_resadd_norm_gemv_fp8_pert)
#define GEMM_OPS()                                                                                           \
  IMPL(esimd_gemm_int4_pgrp); IMPL(esimd_gemm_int4_pgrp_zp); IMPL(esimd_gemm_fp8_pert);                      \
  IMPL(esimd_gemm_fp8_blockscale); IMPL(esimd_gemv_fp8_blockscale_fused2)

TORCH_LIBRARY_IMPL(custom_esimd_kernels_vllm, CUDA, m) { DECODE_OPS(); GEMM_OPS(); }
TORCH_LIBRARY_IMPL(custom_esimd_kernels, CUDA, m) { GEMM_OPS(); }
TORCH_LIBRARY_IMPL(custom_esimd_kernels_sglang, CUDA, m) {
  DECODE_OPS();
  IMPL(esimd_gemv_q4_k); IMPL(esimd_gemv_q4_0); IMPL(esimd_gemm_q4_0); IMPL(esimd_gemv_q8_0); IMPL(esimd_gemv_q8_0_m);
  IMPL(esimd_gemv_q5_k); IMPL(esimd_gemv_q6_k); IMPL(esimd_gemv_q6_k_m);
}
TORCH_LIBRARY_IMPL(moe_ops, CUDA, m) { IMPL(moe_forward_full_fp8_block); }
