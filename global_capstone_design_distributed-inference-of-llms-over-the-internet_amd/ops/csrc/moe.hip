// Routed experts (hybrid decoders, Mixtral): router, choice, and the experts' gated feed-forwards as grouped products.
//
//   moe_router       logits[t, e] = x[t] . router[e] in 32-bit, over K slices
//   moe_choose       softmax over all experts; a group of neighbouring experts counts as its best one; the ``top``
//                    experts with the largest scores among the ``keep`` best groups; weights = scores / (sum + 1e-20)
//                    * scale.  Every choice also gets its place among its expert's rows
//   moe_place        rows sorted by expert: first row of every expert, the token of every row, the row of every choice
//   moe_order        the same, an expert's rows in the order of their tokens
//   moe_combine      every token's rows, weighed and added
//   moe_gemm_any     any shape and both element types
//   moe_gemm_rows    bf16, few rows per expert: weights stream once through registers in fragment order
//   moe_gemm_tile    bf16, many rows per expert: 128 x 128 or 256 x 256 tiles through an LDS ring
//   moe_gemm_wide    bf16, many rows per expert, K in steps of 64: 256 x 256 tiles, whole cache lines of the rows
//
// The products come in two kinds: gathered rows x gate/up weights with the clamped gated form as epilogue
// (GLU: out = g sigmoid(1.702 g) (u + 1), g <= limit, |u| <= limit; without a limit silu(g) u), and sorted rows x down
// weights.
#include "common.h"
#include "act_io.h"
#include "wide_tile.h"

namespace mp {

typedef __attribute__((ext_vector_type(8))) __bf16 bf16x8_t;
__device__ __forceinline__ f32x4 mfma_bf(const u16x8& a, const u16x8& b, const f32x4& c) {
  return __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(bf16x8_t, a), __builtin_bit_cast(bf16x8_t, b), c, 0,
                                                 0, 0);
}

constexpr float MOE_ALPHA = 1.702f;
constexpr int MOE_EXPERTS = 512;
// int32 scratch of a step: [counts E][first row E + 1][active experts E][number of active experts]
struct MoeLists {
  int32_t *cnt, *off, *act, *nact;
};
__host__ __device__ __forceinline__ MoeLists moe_lists(int32_t* p, int E) {
  return MoeLists{p, p + E, p + 2 * E + 1, p + 3 * E + 1};
}

// element offset of x[row, col], row-major (pitch xs) or packed (mt row tiles)
__device__ __forceinline__ int64_t act_at(int row, int col, int64_t xs, int mt) {
  return mt > 0 ? apk_off(row, col, mt) : (int64_t)row * xs + col;
}

__device__ __forceinline__ float moe_glu(float g, float u, float limit) {
  if (limit <= 0.f) return g / (1.f + __expf(-g)) * u;  // (uniform)
  const float a = fminf(g, limit), b = fminf(fmaxf(u, -limit), limit);
  return a / (1.f + __expf(-MOE_ALPHA * a)) * (b + 1.f);
}
__device__ __forceinline__ float moe_glu_exact(float g, float u, float limit) {
  if (limit <= 0.f) return g / (1.f + expf(-g)) * u;
  const float a = fminf(g, limit), b = fminf(fmaxf(u, -limit), limit);
  return a / (1.f + expf(-MOE_ALPHA * a)) * (b + 1.f);
}

// ------------------------------------------------------------------------------------ router
// part[s][t][e].  A workgroup: one token, four experts (a wave each), slice s of K.
template <typename T>
__global__ __launch_bounds__(256) void moe_router_any_kernel(const T* __restrict__ x, int64_t xs, int mt,
                                                             const T* __restrict__ w, float* __restrict__ part, int T_,
                                                             int E, int W, int ks, int32_t* __restrict__ cnt) {
  const int t = blockIdx.x, e = blockIdx.y * 4 + (threadIdx.x >> 6), lane = threadIdx.x & 63, s = blockIdx.z;
  if (t == 0 && s == 0 && e < E && lane == 0) cnt[e] = 0;
  if (e >= E) return;
  const int k1 = min(W, (s + 1) * ks);
  float a = 0.f;
  for (int k = s * ks + lane; k < k1; k += 64) a += to_f(x[act_at(t, k, xs, mt)]) * to_f(w[(int64_t)e * W + k]);
  a = wave_sum(a);
  if (lane == 0) part[((int64_t)s * T_ + t) * E + e] = a;
}

// 16 tokens x 16 NT experts a workgroup; the slice's 32-column steps go round the waves, U of them in flight
template <int NT, int U>
__global__ __launch_bounds__(256) void moe_router_mfma_kernel(const bf16_t* __restrict__ x, int64_t xs, int mt,
                                                              const bf16_t* __restrict__ w, float* __restrict__ part,
                                                              int T, int E, int W, int ks, int32_t* __restrict__ cnt) {
  __shared__ float red[4][16 * NT * 17];
  const int tid = threadIdx.x, lane = tid & 63, wv = tid >> 6, c16 = lane & 15, g4 = lane >> 4;
  const int t0 = blockIdx.x * 16, e0 = blockIdx.y * 16 * NT, s = blockIdx.z;
  if (blockIdx.x == 0 && s == 0 && tid < 16 * NT && e0 + tid < E) cnt[e0 + tid] = 0;
  const int row = min(t0 + c16, T - 1), k1 = min(W, (s + 1) * ks);
  f32x4 acc[NT];
  const bf16_t* wp[NT];
#pragma unroll
  for (int n = 0; n < NT; ++n) {
    acc[n] = (f32x4)(0.f);
    wp[n] = w + (int64_t)min(e0 + 16 * n + c16, E - 1) * W + 8 * g4;
  }
  for (int k = s * ks + 32 * wv; k < k1; k += 128 * U) {
    u16x8 b[U], a[U][NT];
#pragma unroll
    for (int u = 0; u < U; ++u) {
      const int kk = min(k + 128 * u, W - 32);  // (past the slice: loaded, not used)
      b[u] = *reinterpret_cast<const u16x8*>(x + act_at(row, kk + 8 * g4, xs, mt));
#pragma unroll
      for (int n = 0; n < NT; ++n) a[u][n] = *reinterpret_cast<const u16x8*>(wp[n] + kk);
    }
#pragma unroll
    for (int u = 0; u < U; ++u)
      if (k + 128 * u < k1)  // (uniform)
#pragma unroll
        for (int n = 0; n < NT; ++n) acc[n] = mfma_bf(a[u][n], b[u], acc[n]);  // rows: experts, columns: tokens
  }
#pragma unroll
  for (int n = 0; n < NT; ++n)
#pragma unroll
    for (int r = 0; r < 4; ++r) red[wv][(16 * n + 4 * g4 + r) * 17 + c16] = acc[n][r];
  __syncthreads();
  for (int i = tid; i < 256 * NT; i += 256) {
    const int t = i / (16 * NT), e = i % (16 * NT), at = e * 17 + t;
    if (t0 + t < T && e0 + e < E)
      part[((int64_t)s * T + t0 + t) * E + e0 + e] = red[0][at] + red[1][at] + red[2][at] + red[3][at];
  }
}

// ------------------------------------------------------------------------------------ choice
struct ChooseArgs {
  const float* part;  // [S][T][E]
  const int32_t* ctx;  // [T]; <= 0: a padding row, no choice
  int S, T, E, top, groups, keep;
  bool ordered;  // (more than one workgroup) moe_order follows: rows are only counted
  float scale;
  float* ew;          // [T, top]
  int32_t* idx;       // [T, top] expert, -1: none
  int32_t* slot;      // [T, top] place among its expert's rows, then (moe_place) the row
  int32_t* lists;     // moe_lists
  int32_t* tok;       // [T top] token of every row
};
struct RouteIn {  // the router's own operands, where the choice makes the logits as well
  const bf16_t *x, *w;
  int64_t xs;
  int mt, W, ks;
};

constexpr int CH_WAVES = 16;

// exclusive prefix of n <= MOE_EXPERTS counts by one wave; returns the total
__device__ __forceinline__ int moe_prefix(const int32_t* cnt, int32_t* off, int n, int lane) {
  int base = 0;
  for (int i = 0; i < n; i += 64) {
    const int v = i + lane < n ? cnt[i + lane] : 0;
    int x = v;
#pragma unroll
    for (int d = 1; d < 64; d <<= 1) {
      const int y = __shfl_up(x, d, 64);
      if (lane >= d) x += y;
    }
    if (i + lane < n) off[i + lane] = base + x - v;
    base += __shfl(x, 63, 64);
  }
  if (lane == 0) off[n] = base;
  return base;
}
// the experts that have rows, in order
__device__ __forceinline__ void moe_active(const int32_t* cnt, const MoeLists& l, int n, int lane) {
  int base = 0;
  for (int i = 0; i < n; i += 64) {
    const bool on = i + lane < n && cnt[i + lane] > 0;
    const unsigned long long m = __ballot(on);
    if (on) l.act[base + __popcll(m & ((1ull << lane) - 1))] = i + lane;
    base += __popcll(m);
  }
  if (lane == 0) *l.nact = base;
}

// ``per`` tokens a wave; ALONE: one workgroup, one token a wave, places the rows as well.  Round trips set its
// time: all slices of the logits are asked for at once, the rows are placed from registers, and up to
// 64 experts take code of an eighth the size, which is fetched cold in every launch: 12.9 -> 9.3 -> 5.2 us for 6 tokens.
// (Above that a lane has 8 logits to ask for, and 8 slices of each are enough.)
// NT > 0: up to 16 tokens and 16 NT experts, and the logits are made here, a slice of K a wave, in the sums and the order that
// the router's own launch and the choice after it have.  One CU reads the router's weights (64 to 256 KB) in 1 to 2 us,
// less than the launch and the round trip of the slices that it saves.  Two launches took 11.2 us for 6 tokens of 8 experts
// and, a branch beginning between them, 14.7 for 4 tokens of 32; this one takes 8.9 and 11.2.
template <int CH_PER, bool ALONE, int NT>
__global__ __launch_bounds__(CH_WAVES * 64) void moe_choose_kernel(ChooseArgs a, int per, RouteIn in_) {
  constexpr int AHEAD = CH_PER == 1 ? 16 : 8;
  extern __shared__ float sm[];
  const int tid = threadIdx.x, lane = tid & 63, wv = tid >> 6, E = a.E, gs = E / a.groups;
  const int nw = blockDim.x >> 6;
  int32_t* hist = (int32_t*)sm;                // [E]
  int32_t* base = hist + E;                    // [E + 1]
  float* z = sm + 2 * E + 1 + wv * 2 * E;      // this wave's logits
  float* gz = z + E;                           // and its groups' best
  const MoeLists l = moe_lists(a.lists, E);
  for (int e = tid; e < E; e += blockDim.x) hist[e] = 0;
  float* logit = sm + 2 * E + 1 + nw * 2 * E;  // (NT) [S][16 NT][17]
  if constexpr (NT > 0) {
    constexpr int U = NT == 1 ? 8 : 4;
    const int c16 = lane & 15, g4 = lane >> 4, row = min(c16, a.T - 1), k1 = min(in_.W, (wv + 1) * in_.ks);
    if (wv < a.S) {  // (uniform)
      f32x4 acc[4][NT];  // a quarter of the slice's 32-column steps each, as the router's four waves
      const bf16_t* wp[NT];
#pragma unroll
      for (int n = 0; n < NT; ++n) {
#pragma unroll
        for (int q = 0; q < 4; ++q) acc[q][n] = (f32x4)(0.f);
        wp[n] = in_.w + (int64_t)min(16 * n + c16, E - 1) * in_.W + 8 * g4;
      }
      for (int k = wv * in_.ks; k < k1; k += 32 * U) {
        u16x8 b[U], w[U][NT];
#pragma unroll
        for (int u = 0; u < U; ++u) {
          const int kk = min(k + 32 * u, in_.W - 32);  // (past the slice: loaded, not used)
          b[u] = *reinterpret_cast<const u16x8*>(in_.x + act_at(row, kk + 8 * g4, in_.xs, in_.mt));
#pragma unroll
          for (int n = 0; n < NT; ++n) w[u][n] = *reinterpret_cast<const u16x8*>(wp[n] + kk);
        }
#pragma unroll
        for (int u = 0; u < U; ++u)
          if (k + 32 * u < k1)  // (uniform)
#pragma unroll
            for (int n = 0; n < NT; ++n) acc[u & 3][n] = mfma_bf(w[u][n], b[u], acc[u & 3][n]);
      }
#pragma unroll
      for (int n = 0; n < NT; ++n)
#pragma unroll
        for (int r = 0; r < 4; ++r)
          logit[(wv * 16 * NT + 16 * n + 4 * g4 + r) * 17 + c16] = acc[0][n][r] + acc[1][n][r] + acc[2][n][r] + acc[3][n][r];
    }
  }
  __syncthreads();
  const int t0 = (blockIdx.x * nw + wv) * per;
  // the next token's logits are on their way while this one's experts are ranked
  float nx[CH_PER];
  auto fetch = [&](int t) {
#pragma unroll
    for (int j = 0; j < CH_PER; ++j) {
      const int e = lane + 64 * j;
      nx[j] = 0.f;
      if constexpr (NT > 0) {
        for (int s = 0; s < a.S; ++s) nx[j] += logit[(s * 16 * NT + min(e, E - 1)) * 17 + min(t, 15)];
      } else if (64 * j < E) {  // (uniform)
        for (int s = 0; s < a.S; s += AHEAD) {  // so many slices' loads in flight, added in order
          float p[AHEAD];
#pragma unroll
          for (int i = 0; i < AHEAD; ++i)
            p[i] = a.part[((int64_t)min(s + i, a.S - 1) * a.T + min(t, a.T - 1)) * E + min(e, E - 1)];
#pragma unroll
          for (int i = 0; i < AHEAD; ++i) nx[j] += s + i < a.S ? p[i] : 0.f;
        }
      }
    }
  };
  fetch(t0);
  int pick[CH_PER], place[CH_PER];  // (ALONE: a wave's one token's choices, until their rows are known)
#pragma unroll
  for (int j = 0; j < CH_PER; ++j) pick[j] = -1;
  for (int i = 0; i < per; ++i) {
    const int t = t0 + i;
    const bool live = t < a.T && a.ctx[t] > 0;
    float cur[CH_PER];
#pragma unroll
    for (int j = 0; j < CH_PER; ++j) cur[j] = nx[j];
    if (i + 1 < per) fetch(t + 1);
    if (t < a.T && !live)
      for (int k = lane; k < a.top; k += 64) a.idx[t * a.top + k] = a.slot[t * a.top + k] = -1, a.ew[t * a.top + k] = 0.f;
    if (live) {
      float v[CH_PER], mx = -INFINITY;
#pragma unroll
      for (int j = 0; j < CH_PER; ++j) {
        const int e = lane + 64 * j;
        v[j] = -INFINITY;
        if (e < E) {
          v[j] = fmaxf(cur[j], -3e38f);  // (not a number: last, so that every rank is taken once)
          z[e] = v[j];
          mx = fmaxf(mx, v[j]);
        }
      }
      mx = wave_max(mx);
      float sum = 0.f;
#pragma unroll
      for (int j = 0; j < CH_PER; ++j) sum += lane + 64 * j < E ? expf(v[j] - mx) : 0.f;
      sum = wave_sum(sum);
      __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
      __builtin_amdgcn_wave_barrier();
      for (int g = lane; g < a.groups; g += 64) {
        float b = z[g * gs];
#pragma unroll 8
        for (int j = 1; j < gs; ++j) b = fmaxf(b, z[g * gs + j]);
        gz[g] = b;
      }
      __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
      __builtin_amdgcn_wave_barrier();
      // an expert of a group that is not kept leaves the contest (a group's rank: how many are better)
      bool in[CH_PER];
#pragma unroll
      for (int j = 0; j < CH_PER; ++j) {
        const int e = lane + 64 * j, g = min(e, E - 1) / gs;
        int better = 0;
        if (e < E)
#pragma unroll 8
          for (int q = 0; q < a.groups; ++q) better += gz[q] > gz[g] || (gz[q] == gz[g] && q < g);
        in[j] = e < E && better < a.keep;
      }
      __builtin_amdgcn_wave_barrier();
#pragma unroll
      for (int j = 0; j < CH_PER; ++j)
        if (lane + 64 * j < E && !in[j]) z[lane + 64 * j] = -INFINITY;
      __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
      __builtin_amdgcn_wave_barrier();
      float s[CH_PER], cs = 0.f;
      int rank[CH_PER];
#pragma unroll
      for (int j = 0; j < CH_PER; ++j) {
        const int e = lane + 64 * j;
        rank[j] = a.top;
        s[j] = 0.f;
        if (in[j]) {
          int better = 0;
#pragma unroll 8
          for (int q = 0; q < E; ++q) better += z[q] > v[j] || (z[q] == v[j] && q < e);
          rank[j] = better;
          if (better < a.top) s[j] = expf(v[j] - mx) / sum;
        }
        cs += s[j];
      }
      cs = wave_sum(cs);
#pragma unroll
      for (int j = 0; j < CH_PER; ++j)
        if (rank[j] < a.top) {
          const int e = lane + 64 * j, at = t * a.top + rank[j];
          a.ew[at] = s[j] / (cs + 1e-20f) * a.scale;
          a.idx[at] = e;
          const int n = atomicAdd(&hist[e], 1);
          if (ALONE) pick[j] = rank[j], place[j] = n;
          else a.slot[at] = n;
        }
    }
  }
  __syncthreads();
  if constexpr (!ALONE) {  // places become places among all workgroups' rows
    for (int e = tid; e < E; e += blockDim.x) base[e] = hist[e] > 0 ? atomicAdd(&l.cnt[e], hist[e]) : 0;
    if (a.ordered) return;
    __syncthreads();
    for (int i = lane; i < per * a.top; i += 64) {
      const int t = t0 + i / a.top, at = t0 * a.top + i;
      if (t < a.T && a.idx[at] >= 0) a.slot[at] += base[a.idx[at]];
    }
    return;
  }
  if (wv == 0) {
    moe_prefix(hist, base, E, lane);
    moe_active(hist, l, E, lane);
  }
  __syncthreads();
  for (int e = tid; e < E; e += blockDim.x) l.cnt[e] = hist[e];
  for (int e = tid; e <= E; e += blockDim.x) l.off[e] = base[e];
#pragma unroll
  for (int j = 0; j < CH_PER; ++j)
    if (pick[j] >= 0) {
      const int r = base[lane + 64 * j] + place[j];
      a.slot[t0 * a.top + pick[j]] = r;
      a.tok[r] = t0;
    }
}

__global__ __launch_bounds__(256) void moe_place_kernel(ChooseArgs a) {
  __shared__ int32_t off[MOE_EXPERTS + 1];
  const MoeLists l = moe_lists(a.lists, a.E);
  if (threadIdx.x < 64) {
    moe_prefix(l.cnt, off, a.E, threadIdx.x);
    if (blockIdx.x == 0) moe_active(l.cnt, l, a.E, threadIdx.x);
  }
  __syncthreads();
  if (blockIdx.x == 0)
    for (int e = threadIdx.x; e <= a.E; e += 256) l.off[e] = off[e];
  const int i = blockIdx.x * 256 + threadIdx.x;
  if (i < a.T * a.top && a.idx[i] >= 0) {
    const int r = off[a.idx[i]] + a.slot[i];
    a.slot[i] = r;
    a.tok[r] = i / a.top;
  }
}

// A workgroup has an expert, its waves the choices in order, 64 at a time: once to count, once to place.  Rows in the order of
// their tokens are for experts whose last tiles moe_gemm_wide cuts in K: a row's place then decides whether it is one sum or
// two, and with places by atomics the same prompt of 2700 tokens had other last bits (0.002 of its size) in each pass.  Router,
// choice and places of 2700 tokens of two of 8 experts: 19.6 us by atomics, 20.0 in order; 8192 tokens of four of 32, whose
// products are not cut: 31 and 39.
__global__ __launch_bounds__(1024) void moe_order_kernel(ChooseArgs a) {
  constexpr int U = 8;
  __shared__ int32_t off[MOE_EXPERTS + 1], part[16];
  const MoeLists l = moe_lists(a.lists, a.E);
  const int e = blockIdx.x, lane = threadIdx.x & 63, wv = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int n = a.T * a.top, per = (n + 1023) / 1024 * 64, i0 = wv * per, i1 = min(n, i0 + per);
  int v[U], count = 0;
  auto fetch = [&](int i) {
#pragma unroll
    for (int u = 0; u < U; ++u) v[u] = i + 64 * u + lane < i1 ? a.idx[i + 64 * u + lane] : -1;
  };
  for (int i = i0; i < i1; i += 64 * U) {
    fetch(i);
#pragma unroll
    for (int u = 0; u < U; ++u) count += __popcll(__ballot(v[u] == e));
  }
  if (lane == 0) part[wv] = count;
  if (wv == 0) {
    moe_prefix(l.cnt, off, a.E, lane);
    if (e == 0) moe_active(l.cnt, l, a.E, lane);
  }
  __syncthreads();
  if (e == 0)
    for (int x = threadIdx.x; x <= a.E; x += 1024) l.off[x] = off[x];
  int row = off[e];
  for (int w = 0; w < wv; ++w) row += part[w];
  for (int i = i0; i < i1; i += 64 * U) {
    if (per > 64 * U) fetch(i);  // (else they are there)
#pragma unroll
    for (int u = 0; u < U; ++u) {
      const unsigned long long m = __ballot(v[u] == e);
      if (v[u] == e) {
        const int at = i + 64 * u + lane, r = row + __popcll(m & ((1ull << lane) - 1));
        a.slot[at] = r;
        a.tok[r] = at / a.top;
      }
      row += __popcll(m);
    }
  }
}

// ------------------------------------------------------------------------------------ products
struct MoeGemm {
  const void* x;       // rows: x[tok[r]] (gathered; row-major or packed) or x[r]
  int64_t xs;
  int mt;
  const int32_t* tok;  // null: sorted rows
  const int32_t* lists;
  const void* w;       // [E, N, K] row-major, or fragment order [E, N / 16, K / 32, 64, 8]
  void* out;           // [rows, N] or (GLU) [rows, N / 2]
  int E, N, K, block;  // block: rows of a gate / up block
  float limit;
};

// 32 rows x 32 outputs a workgroup
template <typename T, bool GLU>
__global__ __launch_bounds__(256) void moe_gemm_any_kernel(MoeGemm a) {
  __shared__ float xa[32][33], wa[2][32][33];
  const MoeLists l = moe_lists(const_cast<int32_t*>(a.lists), a.E);
  if ((int)blockIdx.y >= *l.nact) return;
  const int e = l.act[blockIdx.y], r0 = l.off[e], n = l.cnt[e], O = GLU ? a.N / 2 : a.N, o0 = blockIdx.x * 32;
  const int tid = threadIdx.x, tr = tid >> 3, tc = tid & 7;
  const T* w = (const T*)a.w + (int64_t)e * a.N * a.K;
  for (int m0 = 0; m0 < n; m0 += 32) {
    float acc[2][4] = {};
    for (int k0 = 0; k0 < a.K; k0 += 32) {
      __syncthreads();
      for (int i = tid; i < 1024; i += 256) {
        const int r = i >> 5, k = k0 + (i & 31);
        const int m = r0 + min(m0 + r, n - 1), row = a.tok ? a.tok[m] : m;
        xa[r][i & 31] = k < a.K ? to_f(((const T*)a.x)[act_at(row, k, a.xs, a.mt)]) : 0.f;
        const int o = min(o0 + r, O - 1);
#pragma unroll
        for (int h = 0; h < (GLU ? 2 : 1); ++h) {
          const int wr = GLU ? o / a.block * 2 * a.block + h * a.block + o % a.block : o;
          wa[h][r][i & 31] = k < a.K ? to_f(w[(int64_t)wr * a.K + k]) : 0.f;
        }
      }
      __syncthreads();
      for (int k = 0; k < 32; ++k)
#pragma unroll
        for (int c = 0; c < 4; ++c) {
          acc[0][c] += xa[tr][k] * wa[0][tc + 8 * c][k];
          if (GLU) acc[1][c] += xa[tr][k] * wa[1][tc + 8 * c][k];
        }
    }
    if (m0 + tr < n)
#pragma unroll
      for (int c = 0; c < 4; ++c) {
        const int o = o0 + tc + 8 * c;
        if (o >= O) continue;
        const int64_t at = (int64_t)(r0 + m0 + tr) * O + o;
        if (GLU) from_f(moe_glu_exact(acc[0][c], acc[1][c], a.limit), ((T*)a.out)[at]);
        else ((float*)a.out)[at] = acc[0][c];
      }
  }
}

// Few rows per expert.  A workgroup makes 32 weight rows' outputs (two fragment tiles: one gate / up pair) for up to 64
// rows at a time; its four waves take the 32-column steps in turn, so that together they stream 4 KiB runs of packed
// weights, and their sums meet in LDS.  D = W x^T: a lane owns one row and four neighbouring outputs.
template <bool GLU, int NR, int U, bool ONCE>
__device__ __forceinline__ void moe_rows_pass(const MoeGemm& a, const bf16_t* __restrict__ w0, const bf16_t* __restrict__ w1,
                                              int r0, int m0, int n, int o0, int nt1, float* red) {
  const int tid = threadIdx.x, lane = tid & 63, c16 = lane & 15, g4 = lane >> 4;
  const int wv = __builtin_amdgcn_readfirstlane(tid >> 6), ks = a.K >> 5;
  const bf16_t* xp[NR];
  int64_t xstep;  // elements from one 32-column step to the next
  {
    xstep = a.mt > 0 ? (int64_t)a.mt * 512 : 32;
#pragma unroll
    for (int i = 0; i < NR; ++i) {
      const int m = r0 + min(m0 + 16 * i + c16, n - 1), row = a.tok ? a.tok[m] : m;
      xp[i] = (const bf16_t*)a.x + act_at(row, 8 * g4, a.xs, a.mt);
    }
  }
  f32x4 acc[NR][2];
#pragma unroll
  for (int i = 0; i < NR; ++i) acc[i][0] = acc[i][1] = (f32x4)(0.f);
  u16x8 wf[U][2], xf[U][NR];
  const int mine = (ks - wv + 3) >> 2;  // this wave's steps
  auto load = [&](int u, int s) {
    const int64_t st = wv + 4 * min(s, mine - 1);  // (past the end: loaded, not used)
    const u16x8 *p0 = reinterpret_cast<const u16x8*>(w0 + st * 512 + lane * 8), *p1 = reinterpret_cast<const u16x8*>(w1 + st * 512 + lane * 8);
    wf[u][0] = ONCE ? __builtin_nontemporal_load(p0) : *p0;
    wf[u][1] = ONCE ? __builtin_nontemporal_load(p1) : *p1;
#pragma unroll
    for (int i = 0; i < NR; ++i) xf[u][i] = *reinterpret_cast<const u16x8*>(xp[i] + st * xstep);
  };
  auto sum = [&](int u) {
#pragma unroll
    for (int i = 0; i < NR; ++i)
#pragma unroll
      for (int h = 0; h < 2; ++h) acc[i][h] = mfma_bf(wf[u][h], xf[u][i], acc[i][h]);
  };
  if (mine > 0) {
#pragma unroll
    for (int u = 0; u < U; ++u) load(u, u);
    int s = 0;
    for (; s + U < mine; s += U)
#pragma unroll
      for (int u = 0; u < U; ++u) {
        sum(u);
        load(u, s + U + u);
        __builtin_amdgcn_sched_barrier(0);
      }
#pragma unroll
    for (int u = 0; u < U; ++u)
      if (s + u < mine) sum(u);  // (uniform)
  }
  __syncthreads();  // (the previous pass has read its sums)
#pragma unroll
  for (int i = 0; i < NR; ++i)
#pragma unroll
    for (int h = 0; h < 2; ++h) *reinterpret_cast<f32x4*>(red + ((((wv * NR + i) * 2 + h) * 64) + lane) * 4) = acc[i][h];
  __syncthreads();
  for (int q = tid; q < 128 * NR; q += 256) {  // (row tile, half, lane)
    const int i = q >> 7, h = (q >> 6) & 1, ln = q & 63, m = m0 + 16 * i + (ln & 15);
    if (GLU && h) continue;
    f32x4 v[2];
#pragma unroll
    for (int k = 0; k < 2; ++k) {
      v[k] = (f32x4)(0.f);
      if (GLU || k == h)
#pragma unroll
        for (int w = 0; w < 4; ++w) v[k] += *reinterpret_cast<const f32x4*>(red + ((((w * NR + i) * 2 + k) * 64) + ln) * 4);
    }
    if (m >= n) continue;
    if (GLU) {
      float y[4];
#pragma unroll
      for (int r = 0; r < 4; ++r) y[r] = moe_glu(v[0][r], v[1][r], a.limit);
      st_vec<4>((bf16_t*)a.out + (int64_t)(r0 + m) * (a.N / 2) + o0 / 2 + 4 * (ln >> 4), y);
    } else if (h == 0 || nt1) {
      *reinterpret_cast<f32x4*>((float*)a.out + (int64_t)(r0 + m) * a.N + o0 + 16 * h + 4 * (ln >> 4)) = v[h];
    }
  }
}

// ONCE: the weights come past the caches (non-temporal), in a single pass of up to 64 rows.  Two of 8 experts for 6 tokens of
// width 4096, 14336 columns: up 268 -> 238 us (6.9 TB/s), down 140 -> 125.  Experts of more rows read their weights again, from
// cache: past it 100 rows took 934 us instead of 832.
template <bool GLU, bool ONCE>
__device__ __forceinline__ void moe_rows(const MoeGemm& a, const bf16_t* __restrict__ w0, const bf16_t* __restrict__ w1, int r0,
                                         int n, int o0, int nt1, float* red) {
  for (int m0 = 0; m0 < n; m0 += 64) {
    const int left = n - m0;
    if (left <= 16) moe_rows_pass<GLU, 1, 6, ONCE>(a, w0, w1, r0, m0, n, o0, nt1, red);
    else if (left <= 32) moe_rows_pass<GLU, 2, 4, ONCE>(a, w0, w1, r0, m0, n, o0, nt1, red);
    else moe_rows_pass<GLU, 4, 4, ONCE>(a, w0, w1, r0, m0, n, o0, nt1, red);
  }
}
template <bool GLU, bool ONCE>
__global__ __launch_bounds__(256) void moe_gemm_rows_kernel(MoeGemm a) {
  __shared__ __attribute__((aligned(16))) float red[4 * 4 * 2 * 64 * 4];
  const MoeLists l = moe_lists(const_cast<int32_t*>(a.lists), a.E);
  if ((int)blockIdx.y >= *l.nact) return;
  const int e = l.act[blockIdx.y], r0 = l.off[e], n = l.cnt[e], nt = a.N / 16, t0 = 2 * blockIdx.x, t1 = min(t0 + 1, nt - 1);
  const int64_t tile = (int64_t)a.K * 16;
  const bf16_t *w = (const bf16_t*)a.w + (int64_t)e * a.N * a.K, *w0 = w + t0 * tile, *w1 = w + t1 * tile;
  if (ONCE && n <= 64) moe_rows<GLU, true>(a, w0, w1, r0, n, 16 * t0, t1 > t0, red);
  else moe_rows<GLU, false>(a, w0, w1, r0, n, 16 * t0, t1 > t0, red);
}

// Many rows per expert: WM x WN waves of MW x NW fragment tiles (rows x weight rows), 32 columns a stage.  Both operands
// arrive in LDS in fragment order (global_load_lds, 1 KiB a wave: packed weights as they lie, rows gathered by lane)
// through a ring of MG_P slots, MG_P - 1 of them in flight.
constexpr int MG_BAND = 8;
constexpr int MG_P = 4;

__device__ __forceinline__ int moe_tile_count(const MoeLists& l, int E, int i, int lane, int bm) {
  return i + lane < E ? (l.cnt[i + lane] + bm - 1) / bm : 0;
}

// which tile this workgroup makes (one wave): experts' row tiles in order, an expert's tiles in bands of MG_BAND row tiles, a
// band's by weight rows, then rows; a contiguous run of them per XCD, whose 32 CUs then share few rows and few weights.  pick: expert (-1: none), weight tile, row tile
__device__ __forceinline__ void moe_pick(const MoeLists& l, int E, int ntn, int bm, int* pick) {
  const int lane = threadIdx.x & 63;
  int total = 0;
  for (int i = 0; i < E; i += 64) total += moe_tile_count(l, E, i, lane, bm);
#pragma unroll
  for (int d = 32; d > 0; d >>= 1) total += __shfl_xor(total, d, 64);
  const int all = total * ntn, per = (all + 7) / 8;
  const int id = ((int)blockIdx.x & 7) * per + ((int)blockIdx.x >> 3);
  const bool on = ((int)blockIdx.x >> 3) < per && id < all;
  if (lane == 0) pick[0] = -1;
  int base = 0;
  for (int i = 0; i < E && on; i += 64) {
    const int c = moe_tile_count(l, E, i, lane, bm);
    int x = c;
#pragma unroll
    for (int d = 1; d < 64; d <<= 1) {
      const int y = __shfl_up(x, d, 64);
      if (lane >= d) x += y;
    }
    const int lo = (base + x - c) * ntn, hi = (base + x) * ntn;
    if (id >= lo && id < hi) {
      const int q = id - lo, band = q / (MG_BAND * ntn), h = min(MG_BAND, c - MG_BAND * band), r = q - band * MG_BAND * ntn;
      pick[0] = i + lane;
      pick[1] = r / h;
      pick[2] = MG_BAND * band + r % h;
    }
    base += __shfl(x, 63, 64);
  }
}

template <bool GLU, typename TO, int MW, int NW, int WM, int WN>
__global__ __launch_bounds__(WM * WN * 64) void moe_gemm_tile_kernel(MoeGemm a) {
  constexpr int BM = 16 * MW * WM, BN = 16 * NW * WN, FX = BM / 16, J = (BM + BN) / 16 / (WM * WN), SLOT = (BM + BN) * 64;
  static_assert((BM + BN) / 16 % (WM * WN) == 0, "whole fragments a wave");
  extern __shared__ __attribute__((aligned(1024))) char smem[];
  __shared__ int pick[4];
  const MoeLists l = moe_lists(const_cast<int32_t*>(a.lists), a.E);
  const int tid = threadIdx.x, lane = tid & 63, c16 = lane & 15, g4 = lane >> 4;
  const int wv = __builtin_amdgcn_readfirstlane(tid >> 6);
  if (wv == 0) moe_pick(l, a.E, (a.N + BN - 1) / BN, BM, pick);
  __syncthreads();
  const int e = pick[0];
  if (e < 0) return;
  const int n0 = pick[1] * BN, m0 = pick[2] * BM, r0 = l.off[e], n = l.cnt[e], nt = a.N / 16, ks = a.K / 32;
  const bf16_t* w = (const bf16_t*)a.w + (int64_t)e * a.N * a.K;
  const bf16_t* fp[J];  // this wave's fragments of a stage, and their step to the next one
  int fs[J];
#pragma unroll
  for (int j = 0; j < J; ++j) {
    const int f = wv * J + j;
    if (f < FX) {
      const int m = r0 + min(m0 + 16 * f + c16, n - 1), row = a.tok ? a.tok[m] : m;
      fp[j] = (const bf16_t*)a.x + (int64_t)row * a.xs + 8 * g4;
      fs[j] = 32;
    } else {
      fp[j] = w + (int64_t)min(n0 / 16 + f - FX, nt - 1) * a.K * 16 + lane * 8;
      fs[j] = 512;
    }
  }
  typedef __attribute__((address_space(3))) void* lptr_t;
  typedef __attribute__((address_space(1))) const void* gptr_t;
  auto issue = [&](int st) {
    char* b = smem + (st & (MG_P - 1)) * SLOT + wv * J * 1024;
    const int k = min(st, ks - 1);  // (past the end: a slot that is not read)
#pragma unroll
    for (int j = 0; j < J; ++j)
      __builtin_amdgcn_global_load_lds((gptr_t)(fp[j] + (int64_t)k * fs[j]), (lptr_t)(b + j * 1024), 16, 0, 0);
  };
  const int wm = wv % WM, wn = wv / WM;
  f32x4 acc[NW][MW];
#pragma unroll
  for (int i = 0; i < NW; ++i)
#pragma unroll
    for (int j = 0; j < MW; ++j) acc[i][j] = (f32x4)(0.f);
#pragma unroll
  for (int p = 0; p < MG_P - 1; ++p) issue(p);
  for (int st = 0; st < ks; ++st) {
    asm volatile("s_waitcnt vmcnt(%0)" ::"n"(J * (MG_P - 2)) : "memory");
    lds_wait_barrier();  // stage st has landed for all waves, and all have read stage st - 1
    issue(st + MG_P - 1);
    const char* b = smem + (st & (MG_P - 1)) * SLOT + lane * 16;
    u16x8 xf[MW], wf[NW];
#pragma unroll
    for (int j = 0; j < MW; ++j) xf[j] = *reinterpret_cast<const u16x8*>(b + (MW * wm + j) * 1024);
#pragma unroll
    for (int i = 0; i < NW; ++i) wf[i] = *reinterpret_cast<const u16x8*>(b + (FX + NW * wn + i) * 1024);
#pragma unroll
    for (int i = 0; i < NW; ++i)
#pragma unroll
      for (int j = 0; j < MW; ++j) acc[i][j] = mfma_bf(wf[i], xf[j], acc[i][j]);
  }
  asm volatile("s_waitcnt vmcnt(0)" ::: "memory");  // (the ring's last loads end before the workgroup does)
#pragma unroll
  for (int j = 0; j < MW; ++j) {
    const int m = m0 + 16 * (MW * wm + j) + c16;
    if (m >= n) continue;
#pragma unroll
    for (int i = 0; i < NW; i += GLU ? 2 : 1) {
      const int o = n0 + 16 * (NW * wn + i);
      if (o >= a.N) continue;
      float y[4];
#pragma unroll
      for (int r = 0; r < 4; ++r) y[r] = GLU ? moe_glu(acc[i][j][r], acc[GLU ? i + 1 : i][j][r], a.limit) : acc[i][j][r];
      st_vec<4>((TO*)a.out + (int64_t)(r0 + m) * (GLU ? a.N / 2 : a.N) + (GLU ? o / 2 : o) + 4 * g4, y);
    }
  }
}

// Many rows per expert, K in steps of 64: 256 x 256 tiles (wide_tile.h) of gathered rows and packed weights.
// On the ring of 32-column stages, with tiles of eight waves, and so: 2700 tokens of two of eight 14336-wide experts of width 4096 up
// 1502, 1106, 1048 us, down (with the halves added) 803, 651, 568; 4298 tokens of four of 32 1408-wide ones of 2048 up 260, 209,
// 197, down 151, 121, 112 (the last two in turn, means of five draws).
//
// A tile of up to 128 rows makes half the products but loads as much: 0.78 to 0.86 of the time of one of more, 256 of either at once
// (8 experts of 8192 x 1024, weights in the 256 MB cache: 28.2, 36.0 us; of 8192 x 4096, from HBM: 105, 125).  Every XCD gets an
// eighth of the whole tiles and an eighth of the half ones, each a run in order, whose CUs then share few rows and few weights.
// Its G workgroups take whole tiles in turn; those that the r left over do not reach take two half ones first (one
// first: within 1 %, but for down products of 1500 tokens, 4 % more), and the other half ones go round.  Where all that
// is left fits one half round, and a workspace is there, the r are cut at the middle of K instead: a workgroup makes a
// half, and moe_gemm_close_kernel adds the two.  A workgroup's half tiles lie between its whole ones, sooner in some than
// in others: their weights come from HBM a second time, and all at once that bound them.
// Lane k of a wave knows tile k of up to 64 of them: the experts' tile counts are summed over the lanes, then every lane
// looks for its own tile among them.
constexpr int MW_SPLIT = 16;  // whole tiles an XCD cuts at most (twice as many fill 32 workgroups)
struct MoeDeal {
  int f0, q, r, h0, halves;  // whole tiles from f0 on: q a workgroup, r left over; half ones from h0 on
  bool split;
  __device__ MoeDeal(const MoeLists& l, int E, int ntn, int xcd, int G, bool can_split) {
    const int lane = threadIdx.x & 63;
    int f = 0, h = 0;
    for (int i = lane; i < E; i += 64) f += (l.cnt[i] + 127) >> 8, h += ((l.cnt[i] + 255) >> 8) - ((l.cnt[i] + 127) >> 8);
#pragma unroll
    for (int d = 32; d > 0; d >>= 1) f += __shfl_xor(f, d, 64), h += __shfl_xor(h, d, 64);
    const int64_t F = (int64_t)__builtin_amdgcn_readfirstlane(f) * ntn, H = (int64_t)__builtin_amdgcn_readfirstlane(h) * ntn;
    f0 = (int)(F * xcd >> 3), h0 = (int)(H * xcd >> 3);
    const int run = (int)(F * (xcd + 1) >> 3) - f0;
    halves = (int)(H * (xcd + 1) >> 3) - h0, q = run / G, r = run % G;
    split = can_split && r > 0 && r <= MW_SPLIT && 2 * r + halves <= G;
  }
};
// per lane: expert, weight tile and row tile of whole or half tile ``id``
__device__ __forceinline__ void moe_find(const MoeLists& l, int E, int ntn, bool half, int id, int& e, int& nt, int& mt) {
  const int lane = threadIdx.x & 63;
  int fb = 0, hb = 0;
  e = nt = mt = 0;
  for (int i = 0; i < E; i += 64) {
    const int c = i + lane < E ? l.cnt[i + lane] : 0, f = (c + 127) >> 8, h = ((c + 255) >> 8) - f;
    int fs = f, hs = h;
#pragma unroll
    for (int d = 1; d < 64; d <<= 1) {
      const int y = __shfl_up(fs, d, 64), z = __shfl_up(hs, d, 64);
      if (lane >= d) fs += y, hs += z;
    }
    for (int g = 0; g < min(64, E - i); ++g) {
      const int fe = __builtin_amdgcn_readlane(f, g), he = __builtin_amdgcn_readlane(h, g);
      const int ce = half ? he : fe;
      const int first = (half ? hb + __builtin_amdgcn_readlane(hs, g) - he : fb + __builtin_amdgcn_readlane(fs, g) - fe) * ntn;
      if (id >= first && id < first + ce * ntn) {
        const int s = id - first, band = s / (MG_BAND * ntn), n = min(MG_BAND, ce - MG_BAND * band), u = s - band * MG_BAND * ntn;
        e = i + g, nt = u / n;
        mt = half ? fe : MG_BAND * band + u % n;
      }
    }
    fb += __builtin_amdgcn_readlane(fs, 63), hb += __builtin_amdgcn_readlane(hs, 63);
  }
}

template <bool GLU, typename TO>
struct MoeWork {
  static constexpr int STORES = WideTile::put_stores(GLU);
  static constexpr bool TURNS = false;
  typedef WideTile W;
  static constexpr int FRAGS = W::MW;
  const MoeGemm& a;
  const MoeLists& l;
  float* ws;
  int en, mt, pt;  // lane k: expert and weight tile (10 bits and the others), row tile of tile k; 0, or its place in ws + 1
  __device__ int part(int k) const { return __builtin_amdgcn_readlane(pt, k); }
  __device__ int first(int k) const { return part(k) && !(part(k) & 1) ? (a.K / 64 + 1) / 2 : 0; }  // its first stage
  __device__ int expert(int k) const { return __builtin_amdgcn_readlane(en, k) & 1023; }
  __device__ int n0(int k) const { return (__builtin_amdgcn_readlane(en, k) >> 10) * W::BN; }
  __device__ int m0(int k) const { return __builtin_amdgcn_readlane(mt, k) * W::BM; }
  __device__ int stages(int k) const { return !part(k) ? a.K / 64 : (a.K / 64 + (part(k) & 1)) / 2; }
  __device__ void row_offsets(W::Source&) const {}
  __device__ void weight_offsets(W::Source& s) const {
#pragma unroll
    for (int j = 0; j < W::PIECES; ++j) s.off[j] = (uint32_t)W::packed_tile(j) * (uint32_t)(a.K * 32) + W::packed_byte(j);
  }
  __device__ void rows(int k, W::Source& s) const {
    const int e = expert(k), m = m0(k), r0 = l.off[e], n = l.cnt[e];
    s.from(a.x, 0xffffffffu, 128 * first(k), 128);
#pragma unroll
    for (int j = 0; j < W::PIECES; ++j) {  // (the launcher checks that they fit)
      const int q = r0 + min(m + W::piece_row(j), n - 1), row = a.tok ? a.tok[q] : q;
      s.off[j] = (uint32_t)row * (uint32_t)(a.xs * 2) + W::piece_byte();
    }
  }
  __device__ void weights(int k, W::Source& s) const {
    s.from((const bf16_t*)a.w + ((int64_t)expert(k) * a.N + n0(k)) * a.K, (uint32_t)(a.N - n0(k)) * (uint32_t)a.K * 2,
           2048 * first(k), 2048);
  }
  __device__ bool half(int k) const { return l.cnt[expert(k)] - m0(k) <= W::BM / 2; }
  // (a lane's sums as they lie, 16 bytes each: whoever adds the parts has the same lanes)
  static __device__ __forceinline__ f32x4* kept(float* ws, int place) {
    return reinterpret_cast<f32x4*>(ws) + ((int64_t)place * 4 + W::wave()) * W::NW * W::MW * 64 + (threadIdx.x & 63);
  }
  template <int M>
  __device__ int store(int k, const f32x4 (&acc)[W::NW][W::MW]) const {
    const int lane = threadIdx.x & 63;
    if (!GLU && part(k)) {  // (of a whole tile)
      f32x4* to = kept(ws, part(k) - 1);
#pragma unroll
      for (int i = 0; i < W::NW; ++i)
#pragma unroll
        for (int j = 0; j < M; ++j) {
          to[(i * W::MW + j) * 64] = W::taken(acc[i][j]);
          __builtin_amdgcn_sched_barrier(0);
        }
      return STORES * M / W::MW;
    }
    const int e = expert(k), m = m0(k), o = n0(k) + 16 * W::NW * W::wn(), n = l.cnt[e];
    const int cols = GLU ? a.N / 2 : a.N;
    TO* out = (TO*)a.out + (int64_t)(l.off[e] + m) * cols;
    if constexpr (sizeof(TO) == 2) {
      auto go = [&](float limit) {
        return W::put<GLU, M>(out, cols, n - m, GLU ? o / 2 : o, acc, [&](const f32x4& v, const f32x4& u, float(&y)[4]) {
#pragma unroll
          for (int r = 0; r < 4; ++r) y[r] = GLU ? moe_glu(v[r], u[r], limit) : v[r];
        });
      };
      return GLU && a.limit > 0.f ? go(a.limit) : go(0.f);
    } else {
      const int r = 16 * M * W::wm() + (lane & 15);
#pragma unroll
      for (int j = 0; j < M; ++j)
#pragma unroll
        for (int i = 0; i < W::NW; ++i) {
          const f32x4 y = W::taken(acc[i][j]);
          if (m + r + 16 * j < n && o + 16 * i < a.N)
            *reinterpret_cast<f32x4*>(out + (int64_t)(r + 16 * j) * cols + o + 16 * i + 4 * (lane >> 4)) = y;
          __builtin_amdgcn_sched_barrier(0);
        }
      return 0;
    }
  }
};

template <bool GLU, typename TO>
__global__ __launch_bounds__(WideTile::THREADS, 1) void moe_gemm_wide_kernel(MoeGemm a, float* ws) {
  extern __shared__ __attribute__((aligned(1024))) char smem[];
  const MoeLists l = moe_lists(const_cast<int32_t*>(a.lists), a.E);
  const int lane = threadIdx.x & 63, ntn = (a.N + WideTile::BN - 1) / WideTile::BN;
  const int G = gridDim.x >> 3, at = blockIdx.x >> 3, xcd = blockIdx.x & 7;
  const MoeDeal d(l, a.E, ntn, xcd, G, !GLU && ws != nullptr);
  const int free = d.r > 0 && !d.split ? G - d.r : 0, early = min(d.halves, 2 * free);  // half tiles of those the r do not reach
  const int mine = at - d.r;
  const int whole = d.q + (!d.split && at < d.r);
  const int n1 = free > 0 && mine >= 0 && early > mine ? (early - mine + free - 1) / free : 0;
  const int rest = (d.split ? 2 * d.r + d.halves : d.halves - early) - at;
  const int halves = n1 + (rest > 0 ? (rest + G - 1) / G : 0), n = whole + halves;
  const int shift = n * at / G;
  for (int first = 0; first < n; first += 64) {
    const int count = min(64, n - first), k = first + min(lane, count - 1);
    const int before = (k * halves + shift) / n;  // half tiles ahead of tile k
    bool half = ((k + 1) * halves + shift) / n > before;
    int id = d.f0 + at + (k - before) * G, pt = 0;
    if (half) {
      id = before < n1 ? mine + before * free : early + at + (before - n1) * G;
      if (d.split && id < 2 * d.r) {
        pt = 1 + 2 * (xcd * MW_SPLIT + (id >> 1)) + (id & 1);
        id = d.f0 + d.q * G + (id >> 1);
        half = false;
      } else {
        id += d.h0 - (d.split ? 2 * d.r : 0);
      }
    }
    int e, nt, mt;
    moe_find(l, a.E, ntn, half, id, e, nt, mt);
    if (first) __syncthreads();  // (the last tiles' operands have been read)
    WideTile::run<WideTile::PACKED>(smem, count, MoeWork<GLU, TO>{a, l, ws, e + (nt << 10), mt, pt});
  }
}

// The cut tiles' two sums added, rounded and stored; workgroup (XCD, tile of it), two of a wave's eight fragments of weights
// and two of the eight of rows.  Bound by the 64 MB at most that they lie in.
__global__ __launch_bounds__(WideTile::THREADS) void moe_gemm_close_kernel(MoeGemm a, float* ws, int G) {
  typedef WideTile W;
  typedef MoeWork<false, bf16_t> Work;
  const MoeLists l = moe_lists(const_cast<int32_t*>(a.lists), a.E);
  const int lane = threadIdx.x & 63, ntn = (a.N + W::BN - 1) / W::BN, xcd = blockIdx.x & 7, at = blockIdx.x >> 3;
  const int i0 = 2 * (blockIdx.y / (W::MW / 2)), j0 = 2 * (blockIdx.y % (W::MW / 2));
  const MoeDeal d(l, a.E, ntn, xcd, G, true);
  if (!d.split || at >= d.r) return;
  int e, nt, mt;
  moe_find(l, a.E, ntn, false, d.f0 + d.q * G + at, e, nt, mt);
  e = __builtin_amdgcn_readfirstlane(e), nt = __builtin_amdgcn_readfirstlane(nt), mt = __builtin_amdgcn_readfirstlane(mt);
  const int place = 2 * (xcd * MW_SPLIT + at);
  const f32x4 *p = Work::kept(ws, place), *q = Work::kept(ws, place + 1);
  const int m = mt * W::BM + 16 * (W::MW * W::wm() + j0) + (lane & 15), o = nt * W::BN + 16 * (W::NW * W::wn() + i0);
  bf16_t* out = (bf16_t*)a.out + ((int64_t)l.off[e] + m) * a.N + o + 4 * (lane >> 4);
#pragma unroll
  for (int j = 0; j < 2; ++j)
#pragma unroll
    for (int i = 0; i < 2; ++i) {
      if (m + 16 * j >= l.cnt[e] || o + 16 * i >= a.N) continue;
      const int f = ((i0 + i) * W::MW + j0 + j) * 64;
      const f32x4 s = p[f] + q[f];
      const float y[4] = {s[0], s[1], s[2], s[3]};
      st_vec<4>(out + (int64_t)16 * j * a.N + 16 * i, y);
    }
}

template <bool GLU, typename TO>
static int launch_moe_wide(const MoeGemm& a, int rows, int act, float* ws, hipStream_t stream) {
  const int tiles = (rows / WideTile::BM + act) * ((a.N + WideTile::BN - 1) / WideTile::BN), per = (tiles + 7) / 8 + 1;
  const int G = per < WideTile::CUS / 8 ? per : WideTile::CUS / 8;  // (whole and half tiles are shared out apart: one more)
  (void)hipFuncSetAttribute((const void*)moe_gemm_wide_kernel<GLU, TO>, hipFuncAttributeMaxDynamicSharedMemorySize,
                            WideTile::LDS);
  hipLaunchKernelGGL((moe_gemm_wide_kernel<GLU, TO>), dim3(8 * G), dim3(WideTile::THREADS), WideTile::LDS, stream, a, ws);
  if constexpr (!GLU && sizeof(TO) == 2)
    if (ws) hipLaunchKernelGGL(moe_gemm_close_kernel, dim3(8 * MW_SPLIT, WideTile::MW * WideTile::NW / 4),
                               dim3(WideTile::THREADS), 0, stream, a, ws, G);
  return (int)hipGetLastError();
}

// out[t] = sum over its choices of weight * row; a token without choices: 0.  A thread has 8 columns of a token; the rows of
// its choices are read at once.  Bound by the rows' bytes in prompts (2700 tokens of two 4096-wide rows: 18 us for 66 MB) and
// by its launch in decode steps (4.7 us, where one add per expert took 8 x 6).
template <typename T>
__global__ __launch_bounds__(256) void moe_combine_kernel(const T* __restrict__ y, const float* __restrict__ ew,
                                                          const int32_t* __restrict__ slot, bf16_t* __restrict__ out, int top,
                                                          int H, int64_t n) {
  const int64_t i = (int64_t)blockIdx.x * 256 + threadIdx.x;
  if (i >= n) return;
  const int64_t t = i / (H / 8);
  const int c = (int)(i % (H / 8)) * 8;
  float acc[8] = {};
  for (int k = 0; k < top; k += 4) {
    float v[4][8], w[4];
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      const int32_t r = slot[t * top + min(k + j, top - 1)];
      w[j] = k + j < top && r >= 0 ? ew[t * top + k + j] : 0.f;
      ld_vec<8>(y + (int64_t)max(r, 0) * H + c, v[j]);
    }
#pragma unroll
    for (int j = 0; j < 4; ++j)
#pragma unroll
      for (int e = 0; e < 8; ++e) acc[e] += w[j] == 0.f ? 0.f : w[j] * v[j][e];  // (rows never written are not counted)
  }
  st_vec<8>(out + t * H + c, acc);
}

template <bool GLU, typename TO, int MW, int NW, int WM, int WN>
static int launch_moe_tile(const MoeGemm& a, int rows, int act, hipStream_t stream) {
  constexpr int BM = 16 * MW * WM, BN = 16 * NW * WN, LDS = MG_P * (BM + BN) * 64;
  // (row tiles: at most one more than full ones per expert that has rows)
  const int tiles = (rows / BM + act) * ((a.N + BN - 1) / BN);
  (void)hipFuncSetAttribute((const void*)moe_gemm_tile_kernel<GLU, TO, MW, NW, WM, WN>,
                            hipFuncAttributeMaxDynamicSharedMemorySize, LDS);
  hipLaunchKernelGGL((moe_gemm_tile_kernel<GLU, TO, MW, NW, WM, WN>), dim3((tiles + 7) / 8 * 8), dim3(WM * WN * 64), LDS,
                     stream, a);
  return (int)hipGetLastError();
}

}  // namespace mp

// int32 elements of ``lists``
extern "C" int64_t mp_moe_lists(int E) { return 3 * (int64_t)E + 2; }

// K slices of the router's product over T rows
extern "C" int mp_moe_router_splits(int T, int W, int E, int f32) {
  if (f32) return 1;
  const int tiles = ((T + 15) / 16) * ((E + 63) / 64);
  int s = 256 / (tiles > 0 ? tiles : 1);
  if (s > W / 256) s = W / 256;
  return s < 1 ? 1 : s > 16 ? 16 : s;
}

extern "C" int mp_moe_route(const void* x, int64_t xs, int mt, const void* w, const int32_t* ctx, float* part, int S,
                            float* ew, int32_t* idx, int32_t* slot, int32_t* lists, int32_t* tok, int T, int E, int W,
                            int top, int groups, int keep, float scale, int f32, int ordered, hipStream_t stream) {
  using namespace mp;
  (void)hipGetLastError();
  if (T == 0) return 0;
  if (E > MOE_EXPERTS || E < 1 || groups < 1 || E % groups || keep > groups || top > E) return -1;
  const MoeLists l = moe_lists(lists, E);
  int ks = (W + S - 1) / S;
  ks = (ks + 31) / 32 * 32;
  const bool mfma = !f32 && W % 32 == 0 && (mt > 0 || xs % 8 == 0);
  // few tokens and experts: one launch (E > 32: a single CU would read 512 KB of weights and more)
  const int fused = mfma && T <= CH_WAVES && S <= CH_WAVES && E <= 32 ? (E + 15) / 16 : 0;
  if (fused) {
  } else if (mfma) {
#define MP_RT(NT_, U_)                                                                                                  \
  hipLaunchKernelGGL((moe_router_mfma_kernel<NT_, U_>), dim3((T + 15) / 16, (E + 16 * NT_ - 1) / (16 * NT_), S),        \
                     dim3(256), 0, stream, (const bf16_t*)x, xs, mt, (const bf16_t*)w, part, T, E, W, ks, l.cnt)
    if (E <= 16) MP_RT(1, 8);
    else if (E <= 32) MP_RT(2, 8);
    else MP_RT(4, 4);
#undef MP_RT
  } else {
    const dim3 grid(T, (E + 3) / 4, S);
    if (f32)
      hipLaunchKernelGGL(moe_router_any_kernel<float>, grid, dim3(256), 0, stream, (const float*)x, xs, mt,
                         (const float*)w, part, T, E, W, ks, l.cnt);
    else
      hipLaunchKernelGGL(moe_router_any_kernel<bf16_t>, grid, dim3(256), 0, stream, (const bf16_t*)x, xs, mt,
                         (const bf16_t*)w, part, T, E, W, ks, l.cnt);
  }
  const RouteIn in{(const bf16_t*)x, (const bf16_t*)w, xs, mt, W, ks};
  const ChooseArgs a{part, ctx, S, T, E, top, groups, keep, ordered != 0, scale, ew, idx, slot, lists, tok};
  const int nw = E <= 256 ? CH_WAVES : CH_WAVES / 2;  // (LDS: 8 E bytes a wave)
  const size_t lds = (2 * E + 1 + nw * 2 * E + fused * S * 16 * 17) * sizeof(float);
  // one token a wave as long as that fills no more than the chip; a single workgroup also places the rows
  const int per = (T + 256 * nw - 1) / (256 * nw), nb = (T + nw * per - 1) / (nw * per);
  auto choose = [&](auto kern) { hipLaunchKernelGGL(kern, dim3(nb), dim3(nw * 64), lds, stream, a, per, in); };
  if (fused) fused == 1 ? choose(moe_choose_kernel<1, true, 1>) : choose(moe_choose_kernel<1, true, 2>);
  else if (E <= 64) nb > 1 ? choose(moe_choose_kernel<1, false, 0>) : choose(moe_choose_kernel<1, true, 0>);
  else nb > 1 ? choose(moe_choose_kernel<MOE_EXPERTS / 64, false, 0>) : choose(moe_choose_kernel<MOE_EXPERTS / 64, true, 0>);
  if (nb > 1 && ordered) hipLaunchKernelGGL(moe_order_kernel, dim3(E), dim3(1024), 0, stream, a);
  else if (nb > 1) hipLaunchKernelGGL(moe_place_kernel, dim3((T * top + 255) / 256), dim3(256), 0, stream, a);
  return (int)hipGetLastError();
}

extern "C" int mp_moe_combine(const void* y, int f32, const float* ew, const int32_t* slot, void* out, int64_t T, int top,
                              int H, hipStream_t stream) {
  using namespace mp;
  (void)hipGetLastError();
  if (H % 8 || top < 1) return -1;
  if (T == 0) return 0;
  const int64_t n = T * (H / 8);
  const dim3 g((unsigned)((n + 255) / 256));
  if (f32)
    hipLaunchKernelGGL((moe_combine_kernel<float>), g, dim3(256), 0, stream, (const float*)y, ew, slot, (bf16_t*)out, top, H, n);
  else
    hipLaunchKernelGGL((moe_combine_kernel<bf16_t>), g, dim3(256), 0, stream, (const bf16_t*)y, ew, slot, (bf16_t*)out, top, H, n);
  return (int)hipGetLastError();
}

// floats of the workspace that lets form 3 cut the tiles of its last round (bf16 down products): from K = 4096 on, half a
// tile is 45 us and more, and adding the halves 15
extern "C" int64_t mp_moe_gemm_ws(int form, int K) {
  return form == 3 && K % 64 == 0 && K >= 4096 ? 8ll * mp::MW_SPLIT * 2 * mp::WideTile::BM * mp::WideTile::BN : 0;
}

// form 0: any shape, 1: few rows per expert, 2: many, 3: very many
extern "C" int mp_moe_gemm(int form, int glu, const void* x, int64_t xs, int mt, const int32_t* tok,
                           const int32_t* lists, const void* w, void* out, int out_f32, int rows, int E, int N, int K,
                           int block, float limit, int f32, float* ws, hipStream_t stream) {
  using namespace mp;
  (void)hipGetLastError();
  if (rows == 0) return 0;
  const MoeGemm a{x, xs, mt, tok, lists, w, out, E, N, K, block, limit};
  const int act = rows < E ? rows : E, O = glu ? N / 2 : N;
  const dim3 grid((O + 31) / 32, act);
  if (form) {
    if (f32 || N % 16 || K % 32 || (glu && (N % 32 || block != 16))) return -1;
    if (form == 1) {
      if (!glu && !out_f32) return -1;
      const dim3 g((N / 16 + 1) / 2, act);
      // past the caches from 64 MB of experts on (each of a layer's two products for itself).  Both products of a layer, past the caches
      // over from them, 6 and 64 rows: up products of 64 MB and more 0.90 to 0.94 wherever the model's experts are more than the 256
      // MB of cache, 0.90 to 1.07 where they are fewer (2 layers); 32 and 48 MB 0.93 to 0.97 from 8 layers on, up to 1.09 with
      // fewer; 16 MB 0.98 to 1.02 with 16 layers, 1.02 to 1.12 with fewer, whose weights are still there in the next step
      const bool once = (int64_t)E * N * K * 2 >= 64ll << 20;
      auto launch = [&](auto kern) { hipLaunchKernelGGL(kern, g, dim3(256), 0, stream, a); };
      if (glu) once ? launch(moe_gemm_rows_kernel<true, true>) : launch(moe_gemm_rows_kernel<true, false>);
      else once ? launch(moe_gemm_rows_kernel<false, true>) : launch(moe_gemm_rows_kernel<false, false>);
      return (int)hipGetLastError();
    }
    if (mt > 0) return -1;
    // 256 x 256 tiles from 128 rows an expert on (ops/moe.py expert_form); where K is not in steps of 64, or a piece's
    // byte offset does not fit 32 bits, the ring of 32-column stages: its 256 x 256 form from 384 rows on, else 128 x 128
    const bool wide = form == 3 && K % 64 == 0 && (int64_t)rows * xs < (1ll << 31) && (int64_t)N * K < (1ll << 31) &&
                      (uintptr_t)out % 4 == 0;
    const bool big = form == 3 && rows >= 384 * E;
#define MP_MT(GLU_, TO_)                                                        \
  return wide  ? launch_moe_wide<GLU_, TO_>(a, rows, act, GLU_ || sizeof(TO_) != 2 ? nullptr : ws, stream) \
         : big ? launch_moe_tile<GLU_, TO_, 4, 8, 4, 2>(a, rows, act, stream) \
               : launch_moe_tile<GLU_, TO_, 4, 4, 2, 2>(a, rows, act, stream);
    if (glu) MP_MT(true, bf16_t)
    if (out_f32) MP_MT(false, float)
    MP_MT(false, bf16_t)
#undef MP_MT
  }
  if (!glu && !out_f32) return -1;
  if (f32) {
    if (glu) hipLaunchKernelGGL((moe_gemm_any_kernel<float, true>), grid, dim3(256), 0, stream, a);
    else hipLaunchKernelGGL((moe_gemm_any_kernel<float, false>), grid, dim3(256), 0, stream, a);
  } else {
    if (glu) hipLaunchKernelGGL((moe_gemm_any_kernel<bf16_t, true>), grid, dim3(256), 0, stream, a);
    else hipLaunchKernelGGL((moe_gemm_any_kernel<bf16_t, false>), grid, dim3(256), 0, stream, a);
  }
  return (int)hipGetLastError();
}
