// Ends of the products over row-major operands (gemm_prompt.hip, gemm_mid.hip): 0 none, 1 the gated forms of a gate and an up value,
// 4 max(y, 0)^2.
#pragma once
#include "common.h"

namespace mp {

constexpr int GW_COLUMNS = 8;  // in place of an epilogue: w is [K, N], no epilogue

// (divisions, ten instructions each: v_rcp_f32 in their place takes 2 % off 2700 x 28672 x 4096, but is off by 1 unit in 24 bits
// instead of a half, and 0 where 1 + exp(-v) is 2^126 and more)
template <int EPI, bool LIMIT>
__device__ __forceinline__ void gw_act(float limit, const f32x4& v, const f32x4& u, float (&y)[4]) {
#pragma unroll
  for (int r = 0; r < 4; ++r) {
    if (EPI == 1 && LIMIT) {
      const float g = fminf(v[r], limit), w = fminf(fmaxf(u[r], -limit), limit);
      y[r] = g / (1.f + __expf(-1.702f * g)) * (w + 1.f);
    } else if (EPI == 1) {
      y[r] = v[r] / (1.f + __expf(-v[r])) * u[r];
    } else if (EPI == 4) {
      const float p = v[r] < 0.f ? 0.f : v[r];  // (not a number stays one)
      y[r] = p * p;
    } else {
      y[r] = v[r];
    }
  }
}


}  // namespace mp
