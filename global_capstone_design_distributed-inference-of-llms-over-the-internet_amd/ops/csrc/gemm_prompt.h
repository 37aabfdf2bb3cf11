// The tiles of gemm_prompt.hip, by how high they are: its own of 256 rows, gemm_prompt_low.hip's of 128 to 224.
#pragma once
#include "act_io.h"
#include "gemm_act.h"
#include "wide_tile.h"

namespace mp {

constexpr int GW_CUS = WideTile::CUS, GW_BAND = 8;
constexpr int64_t GW_SLAB = 256 * 256;  // fp32 elements of a part

struct GemmPrompt {
  const bf16_t* x;
  int64_t xs;
  const bf16_t* w;
  bf16_t* out;
  int M, N, K;
  float limit;
  int mt, nt;      // row and weight tiles
  int frags;       // fragments of 16 rows that a wave has in a tile, 4 to 8
  int full, rest, parts;  // tiles made whole; tiles cut into parts
  float* slabs;           // [parts][rest][4 waves][8][8][64 lanes][4]
};

__device__ __forceinline__ void gw_tile(const GemmPrompt& a, int id, int& m0, int& n0) {
  const int band = id / (GW_BAND * a.nt), h = min(GW_BAND, a.mt - GW_BAND * band), r = id - band * GW_BAND * a.nt;
  m0 = (GW_BAND * band + r % h) * 32 * a.frags;
  n0 = r / h * WideTile::BN;
}
// A workgroup's tiles: every ``step``-th whole one of its XCD's run from ``first`` on, then a part of a left-over tile.
template <int EPI, int FRAGS_>
struct PromptWork {
  static constexpr int FRAGS = FRAGS_, STORES = WideTile::put_stores(EPI == 1) * FRAGS / WideTile::MW;
  static constexpr bool TURNS = false;
  typedef WideTile W;
  const GemmPrompt& a;
  int first, step, whole;  // (whole: how many whole ones)
  int g;                   // the part
  __device__ int id(int k) const { return k < whole ? first + k * step : a.full + g % a.rest; }
  __device__ int begin(int k) const { return k < whole ? 0 : g / a.rest * (a.K / 64) / a.parts; }
  __device__ int stages(int k) const {
    return k < whole ? a.K / 64 : (g / a.rest + 1) * (a.K / 64) / a.parts - g / a.rest * (a.K / 64) / a.parts;
  }
  __device__ void row_offsets(W::Source& s) const {
#pragma unroll
    for (int j = 0; j < FRAGS; ++j) s.off[j] = (uint32_t)W::piece_row(j, FRAGS) * (uint32_t)(a.xs * 2) + W::piece_byte();
  }
  __device__ void weight_offsets(W::Source& s) const {
#pragma unroll
    for (int j = 0; j < W::PIECES; ++j)
      s.off[j] = EPI == GW_COLUMNS ? ((uint32_t)W::column_row(j) * (uint32_t)a.N + W::column_first(j)) * 2
                                   : (uint32_t)W::piece_row(j) * (uint32_t)(a.K * 2) + W::piece_byte();
  }
  __device__ void rows(int k, W::Source& s) const {  // (the launcher checks that the bytes fit 32 bits)
    int m0, n0;
    gw_tile(a, id(k), m0, n0);
    s.from(a.x + m0 * a.xs, ((uint32_t)(a.M - 1 - m0) * (uint32_t)a.xs + (uint32_t)a.K) * 2, begin(k) * 128, 128);
  }
  __device__ void weights(int k, W::Source& s) const {  // (columns past the last of a row are the next row's first: not stored)
    int m0, n0;
    gw_tile(a, id(k), m0, n0);
    if (EPI == GW_COLUMNS)
      s.from(a.w + n0, ((uint32_t)a.N * (uint32_t)a.K - n0) * 2, begin(k) * (uint32_t)a.N * 128, (uint32_t)a.N * 128);
    else
      s.from(a.w + (int64_t)n0 * a.K, (uint32_t)(a.N - n0) * (uint32_t)a.K * 2, begin(k) * 128, 128);
  }
  __device__ bool half(int k) const {
    int m0, n0;
    gw_tile(a, id(k), m0, n0);
    return a.M - m0 <= W::BM / 2;
  }
  template <int M>
  __device__ int store(int k, const f32x4 (&acc)[W::NW][W::MW]) const {
    if (k == whole) {  // (nothing comes behind it)
      float* s = a.slabs + (int64_t)g * GW_SLAB + (W::wave() * W::NW * W::MW * 64 + (threadIdx.x & 63)) * 4;
#pragma unroll
      for (int i = 0; i < W::NW; ++i)
#pragma unroll
        for (int j = 0; j < M; ++j) {
          *reinterpret_cast<f32x4*>(s + (i * W::MW + j) * 256) = W::taken(acc[i][j]);
          __builtin_amdgcn_sched_barrier(0);
        }
      return 0;
    }
    int m0, n0;
    gw_tile(a, id(k), m0, n0);
    const int nw = n0 + 16 * W::NW * W::wn(), cols = EPI == 1 ? a.N / 2 : a.N;
    auto go = [&](auto limit) {
      return W::put<EPI == 1, M>(a.out + (int64_t)m0 * cols, cols, a.M - m0, EPI == 1 ? nw / 2 : nw, acc,
                                 [&](const f32x4& v, const f32x4& u, float(&y)[4]) { gw_act<EPI, limit.value>(a.limit, v, u, y); });
    };
    return EPI == 1 && a.limit > 0.f ? go(W::Int<1>()) : go(W::Int<0>());
  }
};

template <int EPI, int FRAGS>
__global__ __launch_bounds__(WideTile::THREADS, 1) void gemm_prompt_kernel(GemmPrompt a) {
  extern __shared__ __attribute__((aligned(1024))) char smem[];
  const int xcd = blockIdx.x & 7, at = blockIdx.x >> 3, step = gridDim.x >> 3;
  const int per = (a.full + 7) / 8, lo = xcd * per, run = min(per, a.full - lo);  // the XCD's run of whole tiles
  const int all = a.rest * a.parts, each = (all + 7) / 8, g = xcd * each + at;
  const int whole = at < run ? (run - at + step - 1) / step : 0, count = whole + (at < each && g < all);
  if (count == 0) return;
  WideTile::run<EPI == GW_COLUMNS ? WideTile::COLUMNS : WideTile::ROWS>(smem, count, PromptWork<EPI, FRAGS>{a, lo + at, step, whole, g});
}

// as many workgroups to an XCD as it has tiles or parts, up to its CUs
template <int EPI, int FRAGS>
static void launch_prompt(const GemmPrompt& a, hipStream_t stream) {
  const int per = (a.full + 7) / 8, each = (a.rest * a.parts + 7) / 8, most = per > each ? per : each;
  const dim3 grid(8 * (most < GW_CUS / 8 ? most : GW_CUS / 8));
  (void)hipFuncSetAttribute((const void*)gemm_prompt_kernel<EPI, FRAGS>, hipFuncAttributeMaxDynamicSharedMemorySize, WideTile::LDS);
  hipLaunchKernelGGL((gemm_prompt_kernel<EPI, FRAGS>), grid, dim3(WideTile::THREADS), WideTile::LDS, stream, a);
}

}  // namespace mp
