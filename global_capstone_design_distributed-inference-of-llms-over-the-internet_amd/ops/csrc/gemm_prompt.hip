// Products of prompt-sized steps: y[M, N'] = epilogue(x[M, K] w[N, K]^T), both operands row-major, or x[M, K] w[K, N] for
// gradients; 256 x 256 tiles of wide_tile.h.  Epilogues: none; the gated forms over gate / up rows in blocks of 16 (silu(g) u, or with a limit
// g sigmoid(1.702 g) (u + 1) on clamped inputs), N' = N / 2; max(y, 0)^2.  Everything up to the one store is 32 bits: next to
// a library product and an activation kernel, the product's rows are neither written, read back nor rounded.
//
// Tiles that fill the 256 CUs go out whole, in bands of 8 row tiles and contiguous runs per XCD.  What is left over would
// hold the chip for another whole tile's time with some of its CUs: up to 128 such tiles have their K cut into 2 or more
// equal parts, one per CU, fp32 parts go to a workspace and a second kernel adds a tile's parts in order and stores it.
// Workgroups of the same part are neighbours, so that an XCD's CUs still walk the same columns of shared rows (ranges that
// begin anywhere, as many as CUs, lost that: 176 left-over tiles of K 11008 took 310 us, made whole 216 us).
#include "act_io.h"
#include "gemm_act.h"
#include "wide_tile.h"

namespace mp {

constexpr int GW_CUS = WideTile::CUS, GW_BAND = 8;
constexpr int64_t GW_SLAB = 256 * 256;  // fp32 elements of a part
// stages that a part has to save: 272 tiles of K 4096 (64 stages, 16 parts) 175 -> 138 us, of K 11008 434 -> 316 us; 112
// tiles of K 4096 (2 parts, 32 saved) 81 -> 66 us
constexpr int GW_SPLIT_STAGES = 24;

struct GemmPrompt {
  const bf16_t* x;
  int64_t xs;
  const bf16_t* w;
  bf16_t* out;
  int M, N, K;
  float limit;
  int mt, nt;      // row and weight tiles
  int full, rest, parts;  // tiles made whole; tiles cut into parts
  float* slabs;           // [parts][rest][4 waves][8][8][64 lanes][4]
};

__device__ __forceinline__ void gw_tile(const GemmPrompt& a, int id, int& m0, int& n0) {
  const int band = id / (GW_BAND * a.nt), h = min(GW_BAND, a.mt - GW_BAND * band), r = id - band * GW_BAND * a.nt;
  m0 = (GW_BAND * band + r % h) * WideTile::BM;
  n0 = r / h * WideTile::BN;
}
// A workgroup's tiles: every ``step``-th whole one of its XCD's run from ``first`` on, then a part of a left-over tile.
template <int EPI>
struct PromptWork {
  static constexpr int STORES = WideTile::put_stores(EPI == 1);
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
    for (int j = 0; j < W::PIECES; ++j) s.off[j] = (uint32_t)W::piece_row(j) * (uint32_t)(a.xs * 2) + W::piece_byte();
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

template <int EPI>
__global__ __launch_bounds__(WideTile::THREADS, 1) void gemm_prompt_kernel(GemmPrompt a) {
  extern __shared__ __attribute__((aligned(1024))) char smem[];
  const int xcd = blockIdx.x & 7, at = blockIdx.x >> 3, step = gridDim.x >> 3;
  const int per = (a.full + 7) / 8, lo = xcd * per, run = min(per, a.full - lo);  // the XCD's run of whole tiles
  const int all = a.rest * a.parts, each = (all + 7) / 8, g = xcd * each + at;
  const int whole = at < run ? (run - at + step - 1) / step : 0, count = whole + (at < each && g < all);
  if (count == 0) return;
  WideTile::run<EPI == GW_COLUMNS ? WideTile::COLUMNS : WideTile::ROWS>(smem, count, PromptWork<EPI>{a, lo + at, step, whole, g});
}

// a left-over tile's parts added and stored; blockIdx.y: two of a wave's eight fragments of weights, two of the eight of rows
template <int EPI>
__global__ __launch_bounds__(WideTile::THREADS) void gemm_prompt_close_kernel(GemmPrompt a) {
  typedef WideTile W;
  const int lane = threadIdx.x & 63, c16 = lane & 15, g4 = lane >> 4, r = blockIdx.x;
  const int i0 = 2 * (blockIdx.y / (W::MW / 2)), j0 = 2 * (blockIdx.y % (W::MW / 2));
  int m0, n0;
  gw_tile(a, a.full + r, m0, n0);
  const int frags = a.M - m0 <= W::BM / 2 ? W::MW / 2 : W::MW;
  const int m = m0 + 16 * (frags * W::wm() + j0) + c16, o = n0 + 16 * (W::NW * W::wn() + i0);
  if (j0 >= frags || m - c16 >= a.M || o >= a.N) return;
  f32x4 acc[2][2];
#pragma unroll
  for (int i = 0; i < 2; ++i)
#pragma unroll
    for (int j = 0; j < 2; ++j) acc[i][j] = (f32x4)(0.f);
  for (int p = 0; p < a.parts; ++p) {
    const float* s = a.slabs + (p * a.rest + r) * GW_SLAB + ((W::wave() * W::NW * W::MW + i0 * W::MW + j0) * 64 + lane) * 4;
#pragma unroll
    for (int i = 0; i < 2; ++i)
#pragma unroll
      for (int j = 0; j < 2; ++j) acc[i][j] += *reinterpret_cast<const f32x4*>(s + (i * W::MW + j) * 256);
  }
#pragma unroll
  for (int j = 0; j < 2; ++j) {
    if (m + 16 * j >= a.M) continue;
#pragma unroll
    for (int i = 0; i < 2; i += EPI == 1 ? 2 : 1)
      if (o + 16 * i < a.N) {
        float y[4];
        if (EPI == 1 && a.limit > 0.f) gw_act<EPI, true>(a.limit, acc[i][j], acc[EPI == 1 ? i + 1 : i][j], y);
        else gw_act<EPI, false>(a.limit, acc[i][j], acc[EPI == 1 ? i + 1 : i][j], y);
        st_vec<4>(a.out + (int64_t)(m + 16 * j) * (EPI == 1 ? a.N / 2 : a.N) + (EPI == 1 ? o / 2 + 8 * i : o + 16 * i) + 4 * g4, y);
      }
  }
}

// into how many parts the tiles past the last whole wave of CUs are cut (1: they are made whole like the others): where
// the stages that a CU saves are worth the parts' way through memory
static int gw_parts(int tiles, int ks) {
  const int rest = tiles % GW_CUS;
  if (!rest || ks < 8) return 1;
  const int parts = GW_CUS / rest < ks / 4 ? GW_CUS / rest : ks / 4;  // (at least four stages a part)
  return ks - (ks + parts - 1) / parts >= GW_SPLIT_STAGES ? parts : 1;
}

}  // namespace mp

// fp32 elements of the workspace
extern "C" int64_t mp_gemm_prompt_ws(int M, int N, int K) {
  using namespace mp;
  const int tiles = ((M + 255) / 256) * ((N + 255) / 256), parts = gw_parts(tiles, K / 64);
  return parts > 1 ? parts * (tiles % GW_CUS) * GW_SLAB : 0;
}

extern "C" int mp_gemm_prompt(const void* x, int64_t xs, const void* w, void* out, int M, int N, int K, int epi, float limit,
                            float* ws, hipStream_t stream) {
  (void)hipGetLastError();
  using namespace mp;
  if (M < 1 || N < 16 || N % 16 || K < 64 || K % 64 || xs % 8 || (int64_t)M * xs >= (1ll << 31) || (int64_t)N * K >= (1ll << 31))
    return -1;
  if (epi == 1 && N % 32) return -2;
  GemmPrompt a{(const bf16_t*)x, xs, (const bf16_t*)w, (bf16_t*)out, M, N, K, limit, (M + 255) / 256, (N + 255) / 256, 0, 0, 1, ws};
  const int tiles = a.mt * a.nt;
  a.parts = gw_parts(tiles, K / 64);
  a.rest = a.parts > 1 ? tiles % GW_CUS : 0;
  if (a.rest && ws == nullptr) return -3;
  a.full = tiles - a.rest;
  // as many workgroups to an XCD as it has tiles or parts, up to its CUs
  const int per = (a.full + 7) / 8, each = (a.rest * a.parts + 7) / 8, most = per > each ? per : each;
  const dim3 grid(8 * (most < GW_CUS / 8 ? most : GW_CUS / 8));
#define MP_GW(E_)                                                                                                          \
  {                                                                                                                        \
    (void)hipFuncSetAttribute((const void*)gemm_prompt_kernel<E_>, hipFuncAttributeMaxDynamicSharedMemorySize, WideTile::LDS); \
    hipLaunchKernelGGL((gemm_prompt_kernel<E_>), grid, dim3(WideTile::THREADS), WideTile::LDS, stream, a);                                  \
    if (a.rest) hipLaunchKernelGGL((gemm_prompt_close_kernel<E_>), dim3(a.rest, WideTile::MW * WideTile::NW / 4),          \
                                   dim3(WideTile::THREADS), 0, stream, a);                                               \
  }
  if (epi == 0) MP_GW(0)
  else if (epi == 1) MP_GW(1)
  else if (epi == 4) MP_GW(4)
  else if (epi == GW_COLUMNS) MP_GW(GW_COLUMNS)
  else return -4;
#undef MP_GW
  return (int)hipGetLastError();
}
