// Products of prompt-sized steps: y[M, N'] = epilogue(x[M, K] w[N, K]^T), both operands row-major, or x[M, K] w[K, N] for
// gradients; tiles of wide_tile.h, 256 weight rows wide and 128 to 256 rows high.  Epilogues: none; the gated forms over gate / up rows in blocks of 16 (silu(g) u, or with a limit
// g sigmoid(1.702 g) (u + 1) on clamped inputs), N' = N / 2; max(y, 0)^2.  Everything up to the one store is 32 bits: next to
// a library product and an activation kernel, the product's rows are neither written, read back nor rounded.
//
// Tiles that fill the 256 CUs go out whole, in bands of 8 row tiles and contiguous runs per XCD.  What is left over would
// hold the chip for another whole tile's time with some of its CUs: up to 128 such tiles have their K cut into 2 or more
// equal parts, one per CU, fp32 parts go to a workspace and a second kernel adds a tile's parts in order and stores it.
// Workgroups of the same part are neighbours, so that an XCD's CUs still walk the same columns of shared rows (ranges that
// begin anywhere, as many as CUs, lost that: 176 left-over tiles of K 11008 took 310 us, made whole 216 us).
#include "gemm_prompt.h"

extern "C" void mp_gemm_prompt_low(const mp::GemmPrompt* a, int epi, hipStream_t stream);

namespace mp {

// a left-over tile's parts added and stored; blockIdx.y: two of a wave's eight fragments of weights, two of the eight of rows
template <int EPI>
__global__ __launch_bounds__(WideTile::THREADS) void gemm_prompt_close_kernel(GemmPrompt a) {
  typedef WideTile W;
  const int lane = threadIdx.x & 63, c16 = lane & 15, g4 = lane >> 4, r = blockIdx.x;
  const int i0 = 2 * (blockIdx.y / (W::MW / 2)), j0 = 2 * (blockIdx.y % (W::MW / 2));
  int m0, n0;
  gw_tile(a, a.full + r, m0, n0);
  const int frags = a.frags == W::MW && a.M - m0 <= W::BM / 2 ? W::MW / 2 : a.frags;
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
    if (m + 16 * j >= a.M || j0 + j >= frags) continue;
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

// stages that a part has to save: 272 tiles of K 4096 (64 stages, 16 parts) 175 -> 138 us, of K 11008 434 -> 316 us; 112
// tiles of K 4096 (2 parts, 32 saved) 81 -> 66 us
constexpr int GW_SPLIT_STAGES = 24;
// into how many parts the tiles past the last whole wave of CUs are cut (1: they are made whole like the others): where
// the stages that a CU saves are worth the parts' way through memory
static int gw_parts(int tiles, int ks) {
  const int rest = tiles % GW_CUS;
  if (!rest || ks < 8) return 1;
  const int parts = GW_CUS / rest < ks / 4 ? GW_CUS / rest : ks / 4;  // (at least four stages a part)
  return ks - (ks + parts - 1) / parts >= GW_SPLIT_STAGES ? parts : 1;
}
static int gw_tiles(int M, int N, int frags) { return (M + 32 * frags - 1) / (32 * frags) * ((N + 255) / 256); }
// How high the tiles are: what an estimate in us says.  A stage takes what is listed (a tile of 128 rows 61 % of one of 256), a
// tile 6.4 more, cut ones 14.7 and their parts' way to memory and back.  Fitted to 51 shapes and row counts whose five heights were
// timed: the height that it picks is 0.6 % slower there than the best, 256 rows 8 %.  At 45 others, of 300 to 7000 rows, 0.3 % (10 at
// the worst) and 9 %: 2100 x 4096 x 2048 42 (256 rows), 33 us (160); 4298 x 2048 x 12800 226, 177 (160); columns of 2500 x 4096 x 4096
// 82, 68 (160).
static int gw_frags(int M, int N, int K) {
  const float stage[5] = {0.77f, 0.88f, 1.00f, 1.17f, 1.27f};
  int best = 8;
  float least = 1e30f;
  for (int f = 8; f >= 4; --f) {
    const int tiles = gw_tiles(M, N, f), ks = K / 64, parts = gw_parts(tiles, ks), rest = parts > 1 ? tiles % GW_CUS : 0;
    const int turns = (tiles - rest + GW_CUS - 1) / GW_CUS;
    float t = turns * (ks * stage[f - 4] + 6.4f);
    if (rest) t += (ks + parts - 1) / parts * stage[f - 4] + 14.7f + 15.8f * rest * parts * f / (8.f * GW_CUS);
    if (t < least) least = t, best = f;
  }
  return best;
}

template <int EPI>
static void launch_prompt(const GemmPrompt& a, hipStream_t stream) {
  if (a.frags == WideTile::MW) launch_prompt<EPI, WideTile::MW>(a, stream);
  else mp_gemm_prompt_low(&a, EPI, stream);
  if (a.rest)
    hipLaunchKernelGGL((gemm_prompt_close_kernel<EPI>), dim3(a.rest, WideTile::MW * WideTile::NW / 4), dim3(WideTile::THREADS), 0,
                       stream, a);
}

}  // namespace mp

// fragments of 16 rows of a wave, half a tile's, that a product's tiles have
extern "C" int mp_gemm_prompt_frags(int M, int N, int K) { return mp::gw_frags(M, N, K); }

// fp32 elements of the workspace
extern "C" int64_t mp_gemm_prompt_ws(int M, int N, int K, int frags) {
  using namespace mp;
  const int tiles = gw_tiles(M, N, frags ? frags : gw_frags(M, N, K)), parts = gw_parts(tiles, K / 64);
  return parts > 1 ? parts * (tiles % GW_CUS) * GW_SLAB : 0;
}

extern "C" int mp_gemm_prompt(const void* x, int64_t xs, const void* w, void* out, int M, int N, int K, int epi, float limit,
                            float* ws, int frags, hipStream_t stream) {
  (void)hipGetLastError();
  using namespace mp;
  if (M < 1 || N < 16 || N % 16 || K < 64 || K % 64 || xs % 8 || (int64_t)M * xs >= (1ll << 31) || (int64_t)N * K >= (1ll << 31))
    return -1;
  if (epi == 1 && N % 32) return -2;
  if (frags == 0) frags = gw_frags(M, N, K);
  if (frags < 4 || frags > WideTile::MW) return -5;
  const int tiles = gw_tiles(M, N, frags), nt = (N + 255) / 256;
  GemmPrompt a{(const bf16_t*)x, xs, (const bf16_t*)w, (bf16_t*)out, M, N, K, limit, tiles / nt, nt, frags, 0, 0, 1, ws};
  a.parts = gw_parts(tiles, K / 64);
  a.rest = a.parts > 1 ? tiles % GW_CUS : 0;
  if (a.rest && ws == nullptr) return -3;
  a.full = tiles - a.rest;
  if (epi == 0) launch_prompt<0>(a, stream);
  else if (epi == 1) launch_prompt<1>(a, stream);
  else if (epi == 4) launch_prompt<4>(a, stream);
  else if (epi == GW_COLUMNS) launch_prompt<GW_COLUMNS>(a, stream);
  else return -4;
  return (int)hipGetLastError();
}
