// torch custom-op registrations (namespace `mpamd`) of the prompt product (gemm_prompt.hip).  Same rules as bindings.cpp:
// outputs come from the caller, launches go to the current stream, shapes and dtypes are checked here.
#include <c10/hip/HIPGuard.h>

#include "bind_check.h"

extern "C" {
int64_t mp_gemm_prompt_ws(int M, int N, int K, int frags);
int mp_gemm_prompt_frags(int M, int N, int K);
int mp_gemm_prompt(const void* x, int64_t xs, const void* w, void* out, int M, int N, int K, int epi, float limit, float* ws,
                 int frags, hipStream_t stream);
int64_t mp_gemm_mid_ws(int M, int N, int K);
int mp_gemm_mid(const void* x, int64_t xs, const void* w, void* out, int M, int N, int K, int epi, float limit, float* ws,
              hipStream_t stream);
}

namespace {

void check_height(int64_t frags) { MP_CHECK(frags == 0 || (frags >= 4 && frags <= 8), "fragments of a wave's rows: 4 to 8, or 0"); }
int64_t gemm_prompt_ws(int64_t M, int64_t N, int64_t K, int64_t frags) {
  check_height(frags);
  return mp_gemm_prompt_ws((int)M, (int)N, (int)K, (int)frags);
}
int64_t gemm_prompt_frags(int64_t M, int64_t N, int64_t K) { return mp_gemm_prompt_frags((int)M, (int)N, (int)K); }
int64_t gemm_mid_ws(int64_t M, int64_t N, int64_t K) { return mp_gemm_mid_ws((int)M, (int)N, (int)K); }

// out[M, N'] = epilogue(x[M, K] w[N, K]^T); epi 8: x[M, K] w[K, N]; frags: fragments of 16 rows of a wave, half a tile's (0: the estimate's)
template <class Room, class Run>
void product(const Room& room, const Run& run, const char* name, const at::Tensor& x, const at::Tensor& w, at::Tensor& out,
             const c10::optional<at::Tensor>& ws, int64_t epi) {
  MP_CHECK(x.is_cuda() && w.is_cuda() && out.is_cuda() && x.dim() == 2 && w.dim() == 2 && out.dim() == 2, "2-d GPU tensors");
  MP_CHECK(x.scalar_type() == at::kBFloat16 && w.scalar_type() == at::kBFloat16 && out.scalar_type() == at::kBFloat16, "bf16");
  const int64_t M = x.size(0), K = x.size(1), N = w.size(epi == 8 ? 1 : 0);
  MP_CHECK(M >= 1 && K >= 64 && K % 64 == 0 && N >= 16 && N % 16 == 0 && w.size(epi == 8 ? 0 : 1) == K, "K in steps of 64, N in steps of 16");
  check_rows(x, M, K, "x");
  check_rows(w, w.size(0), w.size(1), "w");
  check_rows(out, M, epi == 1 ? N / 2 : N, "out");
  MP_CHECK(w.is_contiguous() && out.is_contiguous() && out.size(0) == M && x.stride(0) % 8 == 0 && x.stride(0) >= K, "strides");
  MP_CHECK(M * x.stride(0) < (1ll << 31) && N * K < (1ll << 31), "operands of at most 4 GiB");
  const int64_t need = room((int)M, (int)N, (int)K);
  MP_CHECK(need == 0 || ws.has_value(), "this shape needs a workspace");
  const c10::hip::HIPGuard guard(x.device().index());
  float* p = nullptr;
  if (need) {
    MP_CHECK(ws->is_cuda() && ws->scalar_type() == at::kFloat && ws->is_contiguous() && ws->numel() >= need, "workspace");
    p = ws->data_ptr<float>();
  }
  check_launch(run((int)M, (int)N, (int)K, p), name);
}
void gemm_prompt(const at::Tensor& x, const at::Tensor& w, at::Tensor& out, const c10::optional<at::Tensor>& ws, int64_t epi,
               double limit, int64_t frags) {
  check_height(frags);
  product([&](int M, int N, int K) { return mp_gemm_prompt_ws(M, N, K, (int)frags); },
          [&](int M, int N, int K, float* p) {
            return mp_gemm_prompt(x.data_ptr(), x.stride(0), w.data_ptr(), out.data_ptr(), M, N, K, (int)epi, (float)limit, p, (int)frags,
                                  cur_stream());
          },
          "gemm_prompt", x, w, out, ws, epi);
}
void gemm_mid(const at::Tensor& x, const at::Tensor& w, at::Tensor& out, const c10::optional<at::Tensor>& ws, int64_t epi, double limit) {
  MP_CHECK(x.dim() == 2 && w.dim() == 2 && x.size(0) < (1 << 16), "at most 65535 rows");
  MP_CHECK((x.size(0) + 64) * std::max(w.size(0), w.size(1)) < (1ll << 31), "an output and parts of fewer than 2^31 elements");
  product(mp_gemm_mid_ws,
          [&](int M, int N, int K, float* p) {
            return mp_gemm_mid(x.data_ptr(), x.stride(0), w.data_ptr(), out.data_ptr(), M, N, K, (int)epi, (float)limit, p, cur_stream());
          },
          "gemm_mid", x, w, out, ws, epi);
}

}  // namespace

TORCH_LIBRARY_FRAGMENT(mpamd, m) {
  m.def("gemm_prompt_ws(int M, int N, int K, int frags=0) -> int", &gemm_prompt_ws);
  m.def("gemm_prompt_frags(int M, int N, int K) -> int", &gemm_prompt_frags);
  m.def("gemm_mid_ws(int M, int N, int K) -> int", &gemm_mid_ws);
  m.def("gemm_mid(Tensor x, Tensor w, Tensor(a!) out, Tensor(b!)? ws, int epi, float limit) -> ()");
  m.def("gemm_prompt(Tensor x, Tensor w, Tensor(a!) out, Tensor(b!)? ws, int epi, float limit, int frags=0) -> ()");
}

TORCH_LIBRARY_IMPL(mpamd, CUDA, m) {
  m.impl("gemm_prompt", &gemm_prompt);
  m.impl("gemm_mid", &gemm_mid);
}
