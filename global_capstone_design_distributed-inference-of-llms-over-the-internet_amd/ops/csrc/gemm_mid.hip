// Products of a few dozen to a few hundred rows: the operands, epilogues and results of gemm_prompt.hip on 128 x 128 tiles of
// wide_tile.h.  They are bound by their weights' way from memory: loading [28672, 4096] alone takes 39.5 us here, [12288, 4096]
// 18.3, [4096, 4096] 6.8.  What decided:
//   * Workgroups that walk the same columns of all rows of a row-major matrix keep to a part of the memory's channels: loading
//     [28672, 4096] alone takes 224 of them 48.0 us, and 41.3 where each begins at columns of its own.  So a tile begins with a
//     stage of its own, one of the first 32, and ends with those it left out (rows x 4 KB, which all tiles read at about the
//     same time, stay in L2).  64 x 28672 x 4096 gated 53.1 -> 43.1 us, 16 x 12288 x 4096 28.0 -> 22.6.
//   * A CU loads 22 to 29 GB/s, so all of them have to: K is cut into parts, one per workgroup, whose fp32 sums lie as
//     rows for a second kernel.  How many is an estimate of stages (0.62 us, 0.72 where all CUs load) against the second kernel
//     and the sums' way (3.5 us and twice their bytes at 5 TB/s); within 6 % of the best number at 38 shapes and row counts
//     that were timed with all numbers up to 16 (at two more it picks 32).
//   * Nothing is divided on the way to the first load: the grid says tile, row tile and part.  With the divisions of a list of
//     tiles, 2 us of 13.
//   * Up to one workgroup per CU has nine slots (56 KB of weights in flight); more of them, where a small model's prompt has many
//     rows, share CUs with five each: 384 x 12288 x 4096 65, 52 us.
// us here, of the library and of the 256 x 256 tiles: 64 x 4096 x 14336 29.4, 38.9, 36.1; 192 x 4096 x 4096 19.2, 32.5, 32.1; 128 x
// 28672 x 4096 gated 49.7, 56.9, 65.3; columns of 64 x 4096 x 6144 18.7, 46.5, 26.2; 1024 x 2048 x 512 gated 8.4, 12.8, 18.3.
// From about 8192 stages of all tiles on (128 workgroups of 64) the larger tiles or the library are mostly faster: four operands' reads
// from LDS to 16 products, where the larger tiles have two to 16.
#include "act_io.h"
#include "gemm_act.h"
#include "wide_tile.h"

namespace mp {

constexpr int MID_TURN = 32;  // stages among which a tile's first one is

struct GemmMid {
  const bf16_t* x;
  int64_t xs;
  const bf16_t* w;
  bf16_t* out;
  int M, N, K;
  float limit;
  int parts, each, more;  // of K; stages of a part, parts that have one more
  float* slabs;           // [parts][M][N] where there are several
};

// one part of one tile: workgroup (weight tile, row tile, part)
template <class W, int EPI>
struct MidWork {
  typedef typename W::Source Source;
  static constexpr int STORES = W::put_stores(EPI == 1);
  static constexpr bool TURNS = true;
  static constexpr int FRAGS = W::MW;
  const GemmMid& a;
  int m0, n0, part, first, count, begin;  // its first stage, how many, the one that it begins with (from its first)
  __device__ int stages(int) const { return count; }
  __device__ int turn(int) const { return begin; }
  __device__ bool half(int) const { return a.M - m0 <= W::BM / 2; }
  __device__ void row_offsets(Source& s) const {
#pragma unroll
    for (int j = 0; j < W::PIECES; ++j) s.off[j] = (uint32_t)W::piece_row(j) * (uint32_t)(a.xs * 2) + W::piece_byte();
  }
  __device__ void weight_offsets(Source& s) const {
#pragma unroll
    for (int j = 0; j < W::PIECES; ++j)
      s.off[j] = EPI == GW_COLUMNS ? ((uint32_t)W::column_row(j) * (uint32_t)a.N + W::column_first(j)) * 2
                                   : (uint32_t)W::piece_row(j) * (uint32_t)(a.K * 2) + W::piece_byte();
  }
  __device__ void rows(int, Source& s) const {  // (the launcher checks that the bytes fit 32 bits)
    s.from(a.x + m0 * a.xs, ((uint32_t)(a.M - 1 - m0) * (uint32_t)a.xs + (uint32_t)a.K) * 2, (first + begin) * 128, 128);
  }
  __device__ void weights(int, Source& s) const {  // (columns past the last of a row are the next row's first: not stored)
    if (EPI == GW_COLUMNS)
      s.from(a.w + n0, ((uint32_t)a.N * (uint32_t)a.K - n0) * 2, (first + begin) * (uint32_t)a.N * 128, (uint32_t)a.N * 128);
    else
      s.from(a.w + (int64_t)n0 * a.K, (uint32_t)(a.N - n0) * (uint32_t)a.K * 2, (first + begin) * 128, 128);
  }
  template <int M>
  __device__ int store(int, const f32x4 (&acc)[W::NW][W::MW]) const {
    const int nw = n0 + 16 * W::NW * W::wn(), cols = EPI == 1 ? a.N / 2 : a.N;
    if (a.parts > 1) {
      const int row = m0 + 16 * M * W::wm() + (threadIdx.x & 15), col = nw + 4 * ((threadIdx.x & 63) >> 4);
      float* s = a.slabs + ((int64_t)part * a.M + row) * a.N + col;
#pragma unroll
      for (int j = 0; j < M; ++j)
#pragma unroll
        for (int i = 0; i < W::NW; ++i) {
          const f32x4 y = W::taken(acc[i][j]);
          if (row + 16 * j < a.M && nw + 16 * i < a.N) *reinterpret_cast<f32x4*>(s + (int64_t)16 * j * a.N + 16 * i) = y;
          __builtin_amdgcn_sched_barrier(0);
        }
      return 0;
    }
    auto go = [&](auto limit) {
      return W::template put<EPI == 1, M>(a.out + (int64_t)m0 * cols, cols, a.M - m0, EPI == 1 ? nw / 2 : nw, acc,
                                          [&](const f32x4& v, const f32x4& u, float(&y)[4]) { gw_act<EPI, limit.value>(a.limit, v, u, y); });
    };
    return EPI == 1 && a.limit > 0.f ? go(typename W::template Int<1>()) : go(typename W::template Int<0>());
  }
};

template <int EPI, int SLOTS>
__global__ __launch_bounds__(256, SLOTS == 5 ? 2 : 1) void gemm_mid_kernel(GemmMid a) {
  typedef TileLoop<4, SLOTS> W;
  extern __shared__ __attribute__((aligned(1024))) char smem[];
  const int n0 = blockIdx.x * W::BN, m0 = blockIdx.y * W::BM, part = blockIdx.z;
  if (n0 >= a.N) return;
  const int count = a.each + (part < a.more);
  // (a share of the part's stages that is another from tile to tile)
  const int begin = (int)(((blockIdx.x * 40503u & 0xffffu) * (uint32_t)min(count, MID_TURN)) >> 16);
  W::template run<EPI == GW_COLUMNS ? W::COLUMNS : W::ROWS>(
      smem, 1, MidWork<W, EPI>{a, m0, n0, part, part * a.each + min(part, a.more), count, begin});
}

// the parts of row blockIdx.y added, in order, and stored; a thread has 4 columns of the output
template <int EPI>
__global__ __launch_bounds__(256) void gemm_mid_close_kernel(GemmMid a) {
  const int cols = EPI == 1 ? a.N / 2 : a.N, c = (blockIdx.x * 256 + threadIdx.x) * 4, m = blockIdx.y;
  if (c >= cols) return;
  const float* s = a.slabs + (int64_t)m * a.N + (EPI == 1 ? 2 * c - (c & 15) : c);
  const int64_t step = (int64_t)a.M * a.N;
  f32x4 g = (f32x4)(0.f), u = (f32x4)(0.f);
#pragma unroll 4
  for (int p = 0; p < a.parts; ++p, s += step) {
    g += *reinterpret_cast<const f32x4*>(s);
    if (EPI == 1) u += *reinterpret_cast<const f32x4*>(s + 16);
  }
  float y[4];
  if (EPI == 1 && a.limit > 0.f) gw_act<EPI, true>(a.limit, g, u, y);
  else gw_act<EPI, false>(a.limit, g, u, y);
  st_vec<4>(a.out + (int64_t)m * cols + c, y);
}

static int gm_tiles(int M, int N) { return ((M + 127) / 128) * ((N + 127) / 128); }
// into how many parts K is cut: what an estimate in us says
static int gm_parts(int M, int N, int K) {
  const int tiles = gm_tiles(M, N), ks = K / 64;
  int best = 1;
  float least = 1e30f;
  for (int p = 1; p == 1 || (p * tiles <= 256 && 2 * p <= ks); ++p) {
    const int work = p * tiles < 256 ? p * tiles : 256;
    const float stage = fmaxf(0.62f, 0.0028f * work);
    const float t = stage * ((ks + p - 1) / p) + (p > 1 ? 3.5f + 8.f * p * M * N / 5e6f : 0.f);
    if (t < least) least = t, best = p;
  }
  return best;
}

template <int EPI, int SLOTS>
static void launch_mid(const GemmMid& a, hipStream_t stream) {
  typedef TileLoop<4, SLOTS> W;
  // (many weight tiles in eights: the row tiles and parts of one are on one XCD)
  const int nt = (a.N + W::BN - 1) / W::BN;
  const dim3 grid(nt > 64 ? (nt + 7) / 8 * 8 : nt, (a.M + W::BM - 1) / W::BM, a.parts);
  (void)hipFuncSetAttribute((const void*)gemm_mid_kernel<EPI, SLOTS>, hipFuncAttributeMaxDynamicSharedMemorySize, W::LDS);
  hipLaunchKernelGGL((gemm_mid_kernel<EPI, SLOTS>), grid, dim3(W::THREADS), W::LDS, stream, a);
  const int cols = EPI == 1 ? a.N / 2 : a.N;
  if (a.parts > 1)
    hipLaunchKernelGGL((gemm_mid_close_kernel<EPI>), dim3((cols + 1023) / 1024, a.M), dim3(256), 0, stream, a);
}

}  // namespace mp

// fp32 elements of the workspace
extern "C" int64_t mp_gemm_mid_ws(int M, int N, int K) {
  const int parts = mp::gm_parts(M, N, K);
  return parts > 1 ? (int64_t)parts * M * N : 0;
}

extern "C" int mp_gemm_mid(const void* x, int64_t xs, const void* w, void* out, int M, int N, int K, int epi, float limit, float* ws,
                         hipStream_t stream) {
  (void)hipGetLastError();
  using namespace mp;
  if (M < 1 || N < 16 || N % 16 || K < 64 || K % 64 || xs % 8 || (int64_t)M * xs >= (1ll << 31) || (int64_t)N * K >= (1ll << 31) ||
      (int64_t)(M + 64) * N >= (1ll << 31) || M > 65535)
    return -1;
  if (epi == 1 && N % 32) return -2;
  const int parts = gm_parts(M, N, K), ks = K / 64;
  if (parts > 1 && ws == nullptr) return -3;
  const GemmMid a{(const bf16_t*)x, xs, (const bf16_t*)w, (bf16_t*)out, M, N, K, limit, parts, ks / parts, ks % parts, ws};
  const bool one = gm_tiles(M, N) * parts <= 256;
#define MP_GM(E_)                         \
  if (one) launch_mid<E_, 9>(a, stream);  \
  else launch_mid<E_, 5>(a, stream);
  if (epi == 0) { MP_GM(0) }
  else if (epi == 1) { MP_GM(1) }
  else if (epi == 4) { MP_GM(4) }
  else if (epi == GW_COLUMNS) { MP_GM(GW_COLUMNS) }
  else return -4;
#undef MP_GM
  return (int)hipGetLastError();
}
