// torch custom-op registrations (namespace `mpamd`) of the fine-tuning path's kernels (train.hip).  Same rules as
// bindings.cpp: outputs come from the caller, launches go to the current stream, shapes and dtypes are checked here.
#include <c10/hip/HIPGuard.h>

#include "bind_check.h"

extern "C" {
int mp_train_attn(const void* qkv, int64_t ld, int B, int T, int nh, int nkv, int D, float scale, void* out, float* out32,
                  float* lse, hipStream_t stream);
int mp_train_attn_grad(const void* qkv, int64_t ld, int B, int T, int nh, int nkv, int D, float scale, const float* out32,
                       const float* lse, const void* dout, float* delta, const float* cs, float* part, void* dqkv,
                       hipStream_t stream);
int mp_train_angles(const double* inv, float* out, int n, int64_t T, hipStream_t stream);
int mp_train_rope(void* x, int64_t ld, const float* cs, int64_t rows, int T, int heads, int D, hipStream_t stream);
int mp_train_norm(const void* x, const void* y, const void* w, void* sum, void* out, int64_t rows, int H, float eps, int grad,
                  const void* deep, int P, int T, int64_t apart, hipStream_t stream);
int mp_train_glu_grad(void* gu, const void* da, int64_t rows, int F, hipStream_t stream);
}

namespace {

typedef c10::optional<at::Tensor> opt_tensor;

void* bf16_rows(const at::Tensor& t, int64_t rows, int64_t cols, const char* name) {
  MP_CHECK(t.is_cuda() && t.scalar_type() == at::kBFloat16 && t.is_contiguous() && t.dim() == 2 && t.size(0) == rows &&
               t.size(1) == cols && reinterpret_cast<uintptr_t>(t.data_ptr()) % 16 == 0,
           std::string(name) + ": bf16 [rows, cols], contiguous, 16-B aligned");
  return t.data_ptr();
}
float* f32_rows(const at::Tensor& t, int64_t n, const char* name) {
  MP_CHECK(reinterpret_cast<uintptr_t>(t.data_ptr()) % 16 == 0, std::string(name) + " must be 16-B aligned");
  return const_cast<float*>(f32_vec(t, n, name));
}

struct AttnShape {
  int64_t B, T, D, ld;
};
// qkv [B T, (nh + 2 nkv) D]
AttnShape attn_shape(const at::Tensor& qkv, int64_t B, int64_t nh, int64_t nkv) {
  MP_CHECK(B >= 1 && nkv >= 1 && nh >= nkv && nh % nkv == 0 && nh <= 65535 && B <= 65535, "heads and sequences");
  MP_CHECK(qkv.dim() == 2 && qkv.size(0) >= B && qkv.size(0) % B == 0 && qkv.size(1) % (nh + 2 * nkv) == 0, "qkv shape");
  AttnShape s{B, qkv.size(0) / B, qkv.size(1) / (nh + 2 * nkv), qkv.size(1)};
  MP_CHECK((s.D == 64 || s.D == 128) && s.T <= (1 << 24), "head size 64 or 128");
  bf16_rows(qkv, B * s.T, s.ld, "qkv");
  return s;
}

void train_attn(const at::Tensor& qkv, int64_t B, int64_t nh, int64_t nkv, double scale, at::Tensor& out,
                const opt_tensor& out32, const opt_tensor& lse) {
  const AttnShape s = attn_shape(qkv, B, nh, nkv);
  const c10::hip::HIPGuard guard(qkv.device().index());
  check_launch(mp_train_attn(qkv.data_ptr(), s.ld, B, s.T, nh, nkv, s.D, (float)scale,
                             bf16_rows(out, B * s.T, nh * s.D, "out"),
                             out32.has_value() ? f32_rows(*out32, B * s.T * nh * s.D, "out32") : nullptr,
                             lse.has_value() ? f32_rows(*lse, B * nh * s.T, "lse") : nullptr, cur_stream()),
               "train_attn");
}

void train_attn_grad(const at::Tensor& qkv, int64_t B, int64_t nh, int64_t nkv, double scale, const at::Tensor& out32,
                     const at::Tensor& lse, const at::Tensor& dout, at::Tensor& delta, const at::Tensor& cs, at::Tensor& part,
                     at::Tensor& dqkv) {
  const AttnShape s = attn_shape(qkv, B, nh, nkv);
  const c10::hip::HIPGuard guard(qkv.device().index());
  const int64_t n = B * s.T;
  check_launch(mp_train_attn_grad(qkv.data_ptr(), s.ld, B, s.T, nh, nkv, s.D, (float)scale,
                                  f32_rows(out32, n * nh * s.D, "out32"), f32_rows(lse, n * nh, "lse"),
                                  bf16_rows(dout, n, nh * s.D, "dout"), f32_rows(delta, n * nh, "delta"),
                                  f32_rows(cs, s.T * s.D, "cs"), f32_rows(part, 2 * n * nh * s.D, "part"),
                                  bf16_rows(dqkv, n, s.ld, "dqkv"), cur_stream()),
               "train_attn_grad");
}

// out[T, 2 n]: cos, then sin of t inv[d]
void train_angles(const at::Tensor& inv, at::Tensor& out) {
  MP_CHECK(inv.is_cuda() && inv.scalar_type() == at::kDouble && inv.dim() == 1 && inv.is_contiguous() && inv.numel() >= 1, "inv");
  MP_CHECK(out.is_cuda() && out.device() == inv.device() && out.scalar_type() == at::kFloat && out.dim() == 2 && out.is_contiguous() &&
               out.size(0) >= 1 && out.size(1) == 2 * inv.numel() && out.numel() < (1ll << 38),
           "out fp32 [T, 2 n]");
  const c10::hip::HIPGuard guard(inv.device().index());
  check_launch(mp_train_angles(inv.data_ptr<double>(), out.data_ptr<float>(), inv.numel(), out.size(0), cur_stream()),
               "train_angles");
}

void train_rope(at::Tensor& x, const at::Tensor& cs, int64_t heads, int64_t D) {
  MP_CHECK(x.dim() == 2 && heads >= 1 && D >= 16 && D % 16 == 0 && heads * D <= x.size(1) && x.size(1) % 8 == 0, "rope shape");
  const int64_t T = cs.numel() / D;
  MP_CHECK(T >= 1 && x.size(0) % T == 0, "whole sequences");
  const c10::hip::HIPGuard guard(x.device().index());
  check_launch(mp_train_rope(bf16_rows(x, x.size(0), x.size(1), "x"), x.size(1), f32_rows(cs, T * D, "cs"), x.size(0), T,
                             heads, D, cur_stream()),
               "train_rope");
}

// forward (res absent): out = norm of x + y, ``sum`` = x + y where y is given; backward (grad): out = sum + norm's gradient
// deep [1 or sequences, P, H]: added to every sequence's first P rows
void train_norm(const at::Tensor& x, const opt_tensor& y, const at::Tensor& w, const opt_tensor& sum, at::Tensor& out,
                double eps, bool grad, const opt_tensor& deep, int64_t T) {
  MP_CHECK(x.dim() == 2 && x.size(1) % 8 == 0 && x.size(1) >= 8 && x.size(1) <= 16384 && x.size(0) >= 1, "norm width");
  MP_CHECK(sum.has_value() == (y.has_value() || deep.has_value()) && (!grad || (y.has_value() && !deep.has_value())), "norm operands");
  const int64_t R = x.size(0), H = x.size(1);
  const c10::hip::HIPGuard guard(x.device().index());
  MP_CHECK(w.is_cuda() && w.scalar_type() == at::kBFloat16 && w.is_contiguous() && w.numel() == H &&
               reinterpret_cast<uintptr_t>(w.data_ptr()) % 16 == 0,
           "norm weight");
  const void* first = nullptr;
  int64_t P = 0, apart = 0;
  if (deep.has_value()) {
    MP_CHECK(deep->dim() == 3 && T >= 1 && R % T == 0 && (deep->size(0) == 1 || deep->size(0) == R / T) && deep->size(1) <= T, "deep prompt");
    P = deep->size(1), apart = deep->size(0) == 1 ? 0 : P * H;
    first = bf16_rows(deep->view({deep->size(0) * P, deep->size(2)}), deep->size(0) * P, H, "deep");
  }
  check_launch(mp_train_norm(bf16_rows(x, R, H, "x"), y.has_value() ? bf16_rows(*y, R, H, "y") : nullptr, w.data_ptr(),
                             sum.has_value() ? bf16_rows(*sum, R, H, "sum") : nullptr, bf16_rows(out, R, H, "out"), R, H,
                             (float)eps, grad, first, (int)P, (int)T, apart, cur_stream()),
               "train_norm");
}

void train_glu_grad(at::Tensor& gu, const at::Tensor& da) {
  MP_CHECK(da.dim() == 2 && da.size(1) % 16 == 0 && da.size(0) >= 1 && da.size(1) >= 16, "activation gradient shape");
  const c10::hip::HIPGuard guard(gu.device().index());
  check_launch(mp_train_glu_grad(bf16_rows(gu, da.size(0), 2 * da.size(1), "gu"), bf16_rows(da, da.size(0), da.size(1), "da"),
                                 da.size(0), da.size(1), cur_stream()),
               "train_glu_grad");
}

}  // namespace

TORCH_LIBRARY_FRAGMENT(mpamd, m) {
  m.def(
      "train_attn(Tensor qkv, int B, int nh, int nkv, float scale, Tensor(a!) out, Tensor(b!)? out32=None, Tensor(c!)? "
      "lse=None) -> ()");
  m.def(
      "train_attn_grad(Tensor qkv, int B, int nh, int nkv, float scale, Tensor out32, Tensor lse, Tensor dout, Tensor(a!) "
      "delta, Tensor cs, Tensor(b!) part, Tensor(c!) dqkv) -> ()");
  m.def("train_angles(Tensor inv, Tensor(a!) out) -> ()");
  m.def("train_rope(Tensor(a!) x, Tensor cs, int heads, int D) -> ()");
  m.def(
      "train_norm(Tensor x, Tensor? y, Tensor w, Tensor(a!)? sum, Tensor(b!) out, float eps, bool grad=False, Tensor? deep=None, "
      "int T=0) -> ()");
  m.def("train_glu_grad(Tensor(a!) gu, Tensor da) -> ()");
}

TORCH_LIBRARY_IMPL(mpamd, CUDA, m) {
  m.impl("train_attn", &train_attn);
  m.impl("train_attn_grad", &train_attn_grad);
  m.impl("train_angles", &train_angles);
  m.impl("train_rope", &train_rope);
  m.impl("train_norm", &train_norm);
  m.impl("train_glu_grad", &train_glu_grad);
}
