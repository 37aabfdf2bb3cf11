// Gated recurrences over prompts (gated.h has the equations), gfx950, bf16 activations.  Tokens are taken 16 at a time.  With
// P(a, b] the product of the decays of tokens a < t <= b per key channel, S the state ahead of a block and everything below a
// matrix over the block's tokens:
//
//   U = MU V - W S        what is written: DELTA solves (I + A) U = diag(beta) (V - KG S), A_ij = beta_i k_i . k_j P(j, i] below
//                         the diagonal, so MU = (I + A)^-1 diag(beta), W = MU KG, KG_t = k_t P(-1, t];  GLA U = V;  SSD U = us V
//   O = MO V + Q S        DELTA with B_ij = q_i . k_j P(j, i] up to the diagonal: MO = B MU, Q = QG - MO KG;  GLA MO = B, Q = QG
//   S <- gc S + K^T U     K_t = k_t P(t, 15], gc = P(-1, 15]
//
// Only S goes from block to block.  The rest is made for all blocks at once and then streamed:
//
//   short_conv_kernel       convolution and silu of every row, and the reciprocal norms of DELTA's q and k
//   gated_operands_kernel   GLA, DELTA: a workgroup per (block, head), fp32.  Decay products are only ever products of decays
//                           <= 1.  A and B split by the highest bit in which two positions differ: with L = 8, 4, 2, 1 and m
//                           the start of the upper half of their common 2 L positions, P(j, i] = P(j, m - 1] P(m - 1, i],
//                           so one table per level gives all its pairs as a product.
//   ssd_operands_kernel     SSD: a workgroup per (block, group); decays are scalars, C B^T is made once for a group's heads
//   gated_blocks_kernel     the recurrence: NW waves per (sequence, head, 16 NV NW value columns), S in their MFMA accumulators.
//                           S is the next product's operand as it lies there (the other operand's columns come in the order
//                           in which the accumulators hold them), and so is U.  The blocks' operands lie in memory in fragment
//                           order, 1 KB a fragment, and arrive in LDS through a ring (global_load_lds), each slot filled
//                           again as soon as it has been read.  32-bit operands enter as hi + lo bf16 pairs; where 16 tokens are summed over, the 32 terms
//                           of a product hold both: {hi, lo} times {x, x}.
#include "gated.h"

#include <type_traits>

namespace mp {

typedef __attribute__((ext_vector_type(8))) __bf16 bf16x8_g;
__device__ __forceinline__ f32x4 mfma_k32(const u16x8& a, const u16x8& b, const f32x4& c) {
  return __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(bf16x8_g, a), __builtin_bit_cast(bf16x8_g, b), c, 0, 0, 0);
}
__device__ __forceinline__ f32x4 mfma_f(float a, float b, const f32x4& c) {
  return __builtin_amdgcn_mfma_f32_16x16x4f32(a, b, c, 0, 0, 0);
}

constexpr int GB = 16;  // tokens of a block
constexpr float LOG2E_G = 1.44269504088896340736f, LN2_G = 0.69314718055994530942f;

__device__ __forceinline__ void split4(const f32x4& x, u16x4& hi, u16x4& lo) {
#pragma unroll
  for (int j = 0; j < 4; ++j) {
    hi[j] = f2bf(x[j]);
    lo[j] = f2bf(x[j] - bf2f(hi[j]));
  }
}

__device__ __forceinline__ u16x8 cat4(const u16x4& x, const u16x4& y) {
  return (u16x8){x[0], x[1], x[2], x[3], y[0], y[1], y[2], y[3]};
}
// a lane's 16 bytes of a fragment
__device__ __forceinline__ void put_frag(bf16_t* frag, int lane, const u16x4& x, const u16x4& y) {
  *reinterpret_cast<u16x8*>(frag + lane * 8) = cat4(x, y);
}

__device__ __forceinline__ float sigmoid_g(float x) { return __builtin_amdgcn_rcpf(1.f + __builtin_amdgcn_exp2f(-LOG2E_G * x)); }
// log2(1 + exp(x)) for x <= 0, to a relative error of some units in the last place also where exp(x) is small
__device__ __forceinline__ float log2_1p_exp(float x) {
  const float e = __builtin_amdgcn_exp2f(x * LOG2E_G), w = 1.f + e;
  return w == 1.f ? e * LOG2E_G : __builtin_amdgcn_logf(w) * (e * __builtin_amdgcn_rcpf(w - 1.f));
}

// Fragments (1 KB: 64 lanes, 16 bytes each) of a block's operands for DF 32-column slices of key channels, in this order:
//   per (block, head)   Q hi, Q lo, W hi, W lo (DELTA): [DF] A operands, the columns of a slice in the order 4 g4 + r, 16 + 4 g4 + r
//                       K [2 DF]: A operands of 16 channels, 4 tokens hi | lo;  MO, MU (DELTA): A operands, hi | lo
//                       gc: fp32 [channel];  V [ceil(tiles / 2)]: B operands, two tiles of 16 columns, 8 bytes a lane
//   SSD                 per (block, group) Q [DF] (exact), K [DF]: two tiles of 16 channels, 8 bytes a lane;  per (block, head)
//                       MO, scalars (qs [16], us [16], gc), V
constexpr int FRAG = 512;  // bf16 elements of a fragment
template <int KIND>
struct Operands {
  static __host__ __device__ constexpr int shared(int DF) { return KIND == SSD ? 2 * DF : 0; }
  static __host__ __device__ constexpr int q(int DF) { return 0; }
  static __host__ __device__ constexpr int w(int DF) { return 2 * DF; }
  static __host__ __device__ constexpr int k(int DF) { return KIND == SSD ? DF : KIND == DELTA ? 4 * DF : 2 * DF; }
  // from here on per head; SSD: counted without the shared ones in memory
  static __host__ __device__ constexpr int mo(int DF) { return KIND == SSD ? 0 : k(DF) + 2 * DF; }
  static __host__ __device__ constexpr int mu(int DF) { return mo(DF) + 1; }
  static __host__ __device__ constexpr int gc(int DF) { return mo(DF) + (KIND == DELTA ? 2 : 1); }
  static __host__ __device__ constexpr int v(int DF) { return gc(DF) + 1; }
  static __host__ __device__ constexpr int size(int DF, int tiles) { return v(DF) + (tiles + 1) / 2; }
};

// ------------------------------------------------------------------------------------ convolution
// A wave takes one head's channels (DELTA: q and k heads with their norms, value heads; SSD: value heads, B and C groups) of a
// block's tokens.  chunks [2, n]: first token, tokens.
constexpr int CONV_TAPS = 16, CONV_CH = 8;  // channels of a lane at most

// PAIR: a lane's channels are neighbours two by two (4-byte accesses).  ROWS rows are on their way while as many are worked on: bound by
// memory, where one row ahead was a chain of round trips.  4298 rows of 6144 channels 35.6 -> 27.0 us, of 12288 (two times 106 MB) 78.6 -> 53.2 us.
template <int NCH, int TAPS, bool PAIR>
__global__ __launch_bounds__(256) void short_conv_kernel(GatedArgs a, int kind, int zcol, const int32_t* __restrict__ chunks,
                                                         int nchunk, bf16_t* __restrict__ out, float* __restrict__ unit) {
  const int lane = threadIdx.x & 63, head = blockIdx.y * 4 + (threadIdx.x >> 6), G = a.G, H = a.H, D = a.D, V = a.V;
  const int C = conv_channels(H, G, D, V), taps = TAPS > 0 ? TAPS : a.taps;
  if (head >= 2 * G + H) return;
  // DELTA [q | k | v], SSD [x | B | C]
  const bool key = kind == DELTA ? head < 2 * G : head >= H;
  const int n = key ? D : V, c0 = kind == DELTA ? (key ? head * D : 2 * G * D + (head - 2 * G) * V) : (key ? H * V + (head - H) * D : head * V);
  const int tok0 = chunks[blockIdx.x], ntok = chunks[nchunk + blockIdx.x];
  const int seq = a.q_seq[tok0], p0 = a.q_ctx[tok0] - 1;
  const bf16_t* z = (const bf16_t*)a.z + zcol + c0;
  const float* ring = a.ring + (int64_t)seq * a.taps * C + c0;
  constexpr int TM = TAPS > 0 ? TAPS : CONV_TAPS, ST = PAIR ? 2 : 1, ROWS = NCH > 4 ? 2 : NCH > 2 ? 4 : 8;
  float x[NCH][TM], w[NCH][TM], b[NCH];  // the last inputs, oldest first
  int ch[NCH];
  bool on[NCH];
#pragma unroll
  for (int k = 0; k < NCH; ++k) {
    const int c = PAIR ? 2 * lane + (k & 1) + 128 * (k >> 1) : lane + 64 * k;
    on[k] = c < n;
    ch[k] = PAIR ? min(c & ~1, n - 2) + (c & 1) : min(c, n - 1);  // (PAIR: n is even)
  }
  auto row = [&](int t, bf16_t (&v)[NCH]) {
    const bf16_t* p = z + (int64_t)t * a.zs;
#pragma unroll
    for (int k = 0; k < NCH; k += ST) {
      if constexpr (PAIR) {
        const u16x2 y = *reinterpret_cast<const u16x2*>(p + ch[k]);
        v[k] = y[0], v[k + 1] = y[1];
      } else {
        v[k] = p[ch[k]];
      }
    }
  };
  bf16_t nx[ROWS][NCH];  // the rows that come next, on their way
#pragma unroll
  for (int j = 0; j < ROWS; ++j) row(tok0 + min(j, ntok - 1), nx[j]);
  const bool inside = tok0 > 0 && a.q_seq[max(tok0 - 1, 0)] == seq;  // (then the 16 rows before are this sequence's too)
#pragma unroll
  for (int i = 0; i < TM; ++i) {
    const int back = taps - 1 - i;  // x[i] is position p0 - back's input (i = taps - 1: the token's own)
#pragma unroll
    for (int k = 0; k < NCH; ++k) {
      x[k][i] = 0.f;
      w[k][i] = i < taps ? a.conv[(int64_t)i * C + c0 + ch[k]] : 0.f;
      if (!inside && i < taps - 1 && back <= p0) x[k][i] = ring[(int64_t)((p0 - back) % a.taps) * C + ch[k]];
    }
  }
  if (inside) {
    bf16_t v[TM][NCH];
#pragma unroll
    for (int i = 0; i < TM; ++i) row(max(tok0 - max(taps - 1 - i, 0), 0), v[i]);
#pragma unroll
    for (int i = 0; i < TM; ++i)
#pragma unroll
      for (int k = 0; k < NCH; ++k)
        if (i < taps - 1) x[k][i] = bf2f(v[i][k]);
  }
#pragma unroll
  for (int k = 0; k < NCH; ++k) b[k] = a.conv_b != nullptr ? a.conv_b[c0 + ch[k]] : 0.f;
  auto token = [&](int t, const bf16_t (&in)[NCH]) {
    float ss = 0.f;
    bf16_t o[NCH];
#pragma unroll
    for (int k = 0; k < NCH; ++k)
#pragma unroll
      for (int i = 0; i < TM; ++i)
        if (i == taps - 1) x[k][i] = bf2f(in[k]);
#pragma unroll
    for (int k = 0; k < NCH; ++k) {
      float y = b[k];
#pragma unroll
      for (int i = 0; i < TM; ++i) y += w[k][i] * x[k][i];
      y *= sigmoid_g(y);
#pragma unroll
      for (int i = 0; i < TM - 1; ++i) x[k][i] = x[k][i + 1];
      o[k] = f2bf(y);
      ss += on[k] ? bf2f(o[k]) * bf2f(o[k]) : 0.f;
    }
    bf16_t* p = out + (int64_t)(tok0 + t) * C + c0;
#pragma unroll
    for (int k = 0; k < NCH; k += ST) {
      if (!on[k]) continue;
      if constexpr (PAIR) *reinterpret_cast<u16x2*>(p + ch[k]) = (u16x2){o[k], o[k + ST - 1]};
      else p[ch[k]] = o[k];
    }
    if (kind == DELTA && key) {
      ss = wave_sum(ss);
      if (lane == 0) unit[(int64_t)(tok0 + t) * 2 * G + head] = (head < G ? a.qs : 1.f) / sqrtf(ss + UNIT_EPS);
    }
  };
  for (int t0 = 0; t0 < ntok; t0 += ROWS) {
    bf16_t in[ROWS][NCH];
#pragma unroll
    for (int j = 0; j < ROWS; ++j)
#pragma unroll
      for (int k = 0; k < NCH; ++k) in[j][k] = nx[j][k];
    if (t0 + ROWS < ntok)
#pragma unroll
      for (int j = 0; j < ROWS; ++j) row(tok0 + min(t0 + ROWS + j, ntok - 1), nx[j]);
#pragma unroll
    for (int j = 0; j < ROWS; ++j)
      if (t0 + j < ntok) token(t0 + j, in[j]);
  }
}

// ------------------------------------------------------------------------------------ operands
struct ChunkIn {
  const bf16_t *q, *k, *dec;       // rows' first column of head 0, [T, ..]
  int64_t qs, ks, ds;              // row pitches
  const bf16_t* v;                 // rows' first value column of head 0
  int64_t vs;
  const bf16_t* beta;              // DELTA: [T, ..] column of head 0
  int64_t bs;
  const float* unit;               // DELTA: [T, 2 G]
  const int32_t* chunks;
  int nchunk;
  bf16_t* ops;
};

// LDS: the levels' tables, then in their place Q, K rows from the block's start and the pairs
template <int KIND, int DF>
struct OperandLds {
  static constexpr int DC = 32 * DF, DP = DC + 4;
  static constexpr int KR = KIND == DELTA ? 16 : 8;  // rows of a level's key table (GLA: lower tokens only)
  static constexpr int KT = 0, QT = 4 * KR, TABLES = QT + 32, QG = 0, KG = 16, GATED = KIND == DELTA ? 32 : 16;  // rows
  static constexpr int PAIR = 16 * 20, PAIRS = (KIND == DELTA ? 8 : 4) * PAIR;
  static constexpr int FIRST = TABLES * DP, SECOND = GATED * DP + PAIRS, REST = FIRST > SECOND ? FIRST : SECOND;  // floats
  static constexpr size_t BYTES = (REST + 48 + 64) * 4;
};

// sum over the 32 lanes of a wave's half, valid in the half's last 16 lanes
__device__ __forceinline__ float half_sum(float v) {
  v += dppf<0xB1>(v, 0.f);
  v += dppf<0x4E>(v, 0.f);
  v += dppf<0x141>(v, 0.f);
  v += dppf<0x140>(v, 0.f);
  v += dppf<0x142, 0xA>(v, 0.f);  // row_bcast15 into rows 1, 3
  return v;
}

template <int KIND, int DF>
__global__ __launch_bounds__(256, DF > 4 ? 1 : 3) void gated_operands_kernel(GatedArgs a, ChunkIn in) {
  typedef OperandLds<KIND, DF> L;
  typedef Operands<KIND> Op;
  constexpr int DC = L::DC, DP = L::DP, NC = DC > 128 ? 2 : 1;
  extern __shared__ __attribute__((aligned(16))) float sm[];
  float(*tab)[DP] = reinterpret_cast<float(*)[DP]>(sm);
  float* pairs = sm + L::GATED * DP;
  float(*pq)[16][20] = reinterpret_cast<float(*)[16][20]>(pairs);                // q k pairs of the levels
  float(*pk)[16][20] = reinterpret_cast<float(*)[16][20]>(pairs + 4 * L::PAIR);  // DELTA: k k pairs
  float* sc = sm + L::REST;                                                      // rq [16], rk [16], beta [16]
  float(*dgs)[16] = reinterpret_cast<float(*)[16]>(sc + 48);                     // [4] q k of a token, a wave's channels
  const int tid = threadIdx.x, lane = tid & 63, c16 = lane & 15, g4 = lane >> 4;
  const int w = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int h = blockIdx.y, D = a.D, gh = h / (a.H / a.G);
  const int tok0 = in.chunks[blockIdx.x], nb = in.chunks[in.nchunk + blockIdx.x];
  const int tiles = (a.V + 15) >> 4;
  bf16_t* ops = in.ops + ((int64_t)blockIdx.x * a.H + h) * Op::size(DF, tiles) * FRAG;

  // lanes 0..31 of a wave take tokens 0..7 of 32 channels, the others tokens 8..15 of the same
  const int half = lane >> 5, ch0 = 32 * w + (lane & 31), r0 = 8 * half;
  bf16_t rq[NC][8], rk[NC][8], rd[NC][8];
  float bias[NC];
#pragma unroll
  for (int kk = 0; kk < NC; ++kk) {
    const int cc = min(ch0 + 128 * kk, D - 1);
#pragma unroll
    for (int t = 0; t < 8; ++t) {
      const int64_t r = tok0 + min(r0 + t, nb - 1);
      rq[kk][t] = in.q[r * in.qs + gh * D + cc];
      rk[kk][t] = in.k[r * in.ks + gh * D + cc];
      rd[kk][t] = in.dec[r * in.ds + h * D + cc];
    }
    bias[kk] = KIND == DELTA ? a.dt_bias[h * D + cc] : a.a2_b[h * D + cc];
  }
  if (tid < 16) {
    const int t = tok0 + min(tid, nb - 1);
    const bool ok = tid < nb;
    sc[tid] = KIND == DELTA ? in.unit[(int64_t)t * 2 * a.G + gh] : a.qs;
    sc[16 + tid] = KIND == DELTA ? in.unit[(int64_t)t * 2 * a.G + a.G + gh] : 1.f;
    if constexpr (KIND == DELTA) sc[32 + tid] = ok ? sigmoid_g(bf2f(in.beta[(int64_t)t * in.bs + h])) : 0.f;
  }
  for (int e = tid; e < tiles * 64; e += 256) {  // V as B operands
    const int col = min((e >> 6) * 16 + (e & 15), a.V - 1), t0 = ((e >> 4) & 3) * 4;
    u16x4 x;
#pragma unroll
    for (int j = 0; j < 4; ++j) x[j] = in.v[(int64_t)(tok0 + min(t0 + j, nb - 1)) * in.vs + h * a.V + col];
    *reinterpret_cast<u16x4*>(ops + (Op::v(DF) + (e >> 7)) * FRAG + ((e >> 6) & 1) * 256 + (e & 63) * 4) = x;
  }
  __syncthreads();
  float dg[8], qg[NC][8], kg[NC][8];  // q k of a token; q and k times the decays from the block's start
#pragma unroll
  for (int t = 0; t < 8; ++t) dg[t] = 0.f;
  if (ch0 < DC) {  // (uniform: a wave's channels are all in or out)
#pragma unroll
    for (int kk = 0; kk < NC; ++kk) {
      const int ch = ch0 + 128 * kk;
      float q[8], f[8], k[8];
      const float rate = KIND == DELTA ? a.decay[h] : a.inv_tau;
#pragma unroll
      for (int t = 0; t < 8; ++t) {
        const bool ok = ch < D && r0 + t < nb;  // past the end: f = 1, k = 0, q = 0
        q[t] = ok ? bf2f(rq[kk][t]) : 0.f;
        k[t] = ok ? bf2f(rk[kk][t]) : 0.f;
        const float x = bf2f(rd[kk][t]) + bias[kk];
        // log2 of the decay: GLA log2(sigmoid(x)) / tau, DELTA -A log2(e) softplus(x)
        const float l = log2_1p_exp(-fabsf(x));
        const float e = KIND == DELTA ? -rate * LOG2E_G * (fmaxf(x, 0.f) + l * LN2_G) : rate * (fminf(x, 0.f) * LOG2E_G - l);
        f[t] = ok ? __builtin_amdgcn_exp2f(e) : 1.f;
      }
      auto level = [&](int ti, auto lc) {
        constexpr int N = decltype(lc)::value;
#pragma unroll
        for (int base = 0; base < 8; base += 2 * N) {
          float p = 1.f;
#pragma unroll
          for (int t = base + N - 1; t >= base; --t) {
            tab[L::KT + ti * L::KR + (KIND == DELTA ? r0 + t : (r0 + base) / 2 + t - base)][ch] = k[t] * p;
            p *= f[t];
          }
          p = 1.f;
#pragma unroll
          for (int t = base + N; t < base + 2 * N; ++t) {
            p *= f[t];
            if constexpr (KIND == DELTA) tab[L::KT + ti * L::KR + r0 + t][ch] = k[t] * p;
            tab[L::QT + ti * 8 + (r0 + base) / 2 + t - base - N][ch] = q[t] * p;
          }
        }
      };
      level(1, std::integral_constant<int, 4>());
      level(2, std::integral_constant<int, 2>());
      level(3, std::integral_constant<int, 1>());
      // products within the half: fw[t] = P up to and with t, bw[t] = P after t
      float fw[8], bw[8];
      fw[0] = f[0];
      bw[7] = 1.f;
#pragma unroll
      for (int t = 1; t < 8; ++t) {
        fw[t] = fw[t - 1] * f[t];
        bw[7 - t] = bw[8 - t] * f[8 - t];
      }
      const float other = __shfl_xor(fw[7], 32, 64);  // the other half's
      const float fp = half ? other : 1.f, bp = half ? 1.f : other;
      u16x8 kx[2];  // tokens r0 .. r0 + 3 and r0 + 4 ..: hi | lo
#pragma unroll
      for (int t = 0; t < 8; ++t) {
        dg[t] += q[t] * k[t];
        if (half) {  // level 8: upper tokens forward, lower ones backward
          tab[L::QT + t][ch] = q[t] * fw[t];
          if constexpr (KIND == DELTA) tab[L::KT + 8 + t][ch] = k[t] * fw[t];
        } else {
          tab[L::KT + t][ch] = k[t] * bw[t];
        }
        qg[kk][t] = q[t] * fw[t] * fp;
        kg[kk][t] = k[t] * fw[t] * fp;
        const float x = k[t] * bw[t] * bp * sc[16 + r0 + t];
        const bf16_t hi = f2bf(x);
        kx[t >> 2][t & 3] = hi;
        kx[t >> 2][4 + (t & 3)] = f2bf(x - bf2f(hi));
      }
      bf16_t* kp = ops + (Op::k(DF) + (ch >> 4)) * FRAG + ((r0 >> 2) * 16 + (ch & 15)) * 8;
      *reinterpret_cast<u16x8*>(kp) = kx[0];
      *reinterpret_cast<u16x8*>(kp + 128) = kx[1];
      if (half == 0) reinterpret_cast<float*>(ops + Op::gc(DF) * FRAG)[ch] = fw[7] * other;
    }
  }
#pragma unroll
  for (int t = 0; t < 8; ++t) {
    const float x = half_sum(dg[t]);
    if ((lane & 31) == 31) dgs[w][r0 + t] = x;
  }
  __syncthreads();
  // pairs of level w (2 L positions, L = 8 >> w); of the diagonal a wave's channels
  const int lw = 3 - w;
  f32x4 q2 = (f32x4)(0.f), k2 = (f32x4)(0.f);
  {
    const int low = ((c16 >> (lw + 1)) << lw) | (c16 & ((1 << lw) - 1));  // place of token c16 among its level's halves
    const float* kt = tab[L::KT + w * L::KR + (KIND == DELTA ? c16 : low)] + 4 * g4;
    const float* qt = tab[L::QT + 8 * w + low] + 4 * g4;
#pragma unroll
    for (int m = 0; m < 2 * DF; ++m) {
      const f32x4 x = *reinterpret_cast<const f32x4*>(kt + 16 * m), y = *reinterpret_cast<const f32x4*>(qt + 16 * m);
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        q2 = mfma_f(y[r], x[r], q2);
        if constexpr (KIND == DELTA) k2 = mfma_f(x[r], x[r], k2);
      }
    }
  }
  __syncthreads();  // (the tables have been read)
  if (ch0 < DC) {
#pragma unroll
    for (int kk = 0; kk < NC; ++kk)
#pragma unroll
      for (int t = 0; t < 8; ++t) {
        tab[L::QG + r0 + t][ch0 + 128 * kk] = qg[kk][t];
        if constexpr (KIND == DELTA) tab[L::KG + r0 + t][ch0 + 128 * kk] = kg[kk][t];
      }
  }
#pragma unroll
  for (int r = 0; r < 4; ++r) {
    const int i = 4 * g4 + r, j = c16;
    const bool pair = (i >> (lw + 1)) == (j >> (lw + 1)) && ((i >> lw) & 1) && !((j >> lw) & 1);
    const float s = sc[16 + j];
    pq[w][i][j] = (pair ? q2[r] : i == j ? dgs[w][i] : 0.f) * sc[i] * s;
    if constexpr (KIND == DELTA) pk[w][i][j] = pair ? k2[r] * sc[32 + i] * sc[16 + i] * s : 0.f;
  }
  __syncthreads();
  if constexpr (KIND == DELTA) {
    const int i = tid >> 4, j = tid & 15;  // (from here A, MU, MO lie in pk[0], [1], [2], B in pq[0]; an element is one thread's)
    pk[0][i][j] += pk[1][i][j] + pk[2][i][j] + pk[3][i][j];
    pq[0][i][j] += pq[1][i][j] + pq[2][i][j] + pq[3][i][j];
    __syncthreads();
    if (w == 0) {
      // MU = X diag(beta), X = (I + A)^-1 in halves of 8: X11, X22 column by column, top down; X21 = -X22 A21 X11
      const int hb = (lane >> 3) & 1, jc = lane & 7;
      float x[8];
#pragma unroll
      for (int r = 0; r < 8; ++r) {
        float y = r == jc ? 1.f : 0.f;
#pragma unroll
        for (int l = 0; l < 8; l += 4) {
          if (l >= r) continue;
          const f32x4 v = *reinterpret_cast<const f32x4*>(&pk[0][8 * hb + r][8 * hb + l]);
#pragma unroll
          for (int e = 0; e < 4; ++e)
            if (l + e < r) y -= v[e] * x[l + e];
        }
        x[r] = y;
      }
      if (lane < 16) {
        const float be = sc[32 + 8 * hb + jc];
#pragma unroll
        for (int r = 0; r < 8; ++r) {
          pk[1][8 * hb + r][8 * hb + jc] = x[r] * be;
          if (hb) {
            pk[3][r][jc] = x[r];
            pk[1][r][8 + jc] = 0.f;
          }
        }
      }
      __builtin_amdgcn_wave_barrier();  // (LDS operations of a wave are in order)
      const int xi = lane >> 3, xj = lane & 7;
      float y = 0.f;
#pragma unroll
      for (int l = 0; l < 8; ++l) y += pk[0][8 + xi][l] * pk[1][l][xj];
      pk[3][8 + xi][xj] = y;
      __builtin_amdgcn_wave_barrier();
      y = 0.f;
#pragma unroll
      for (int l = 0; l < 8; ++l) y -= pk[3][xi][l] * pk[3][8 + l][xj];
      pk[1][8 + xi][xj] = y;
      __builtin_amdgcn_wave_barrier();
      f32x4 mo = (f32x4)(0.f);  // MO = B MU
      const f32x4 b = *reinterpret_cast<const f32x4*>(&pq[0][c16][4 * g4]);
#pragma unroll
      for (int r = 0; r < 4; ++r) mo = mfma_f(b[r], pk[1][4 * g4 + r][c16], mo);
#pragma unroll
      for (int r = 0; r < 4; ++r) pk[2][4 * g4 + r][c16] = mo[r];
    }
    __syncthreads();
    const float rqc = sc[c16];
    // W = MU KG and Q = QG - MO KG, made as their transposes: a lane holds four neighbouring channels of token c16
    f32x4 mu = *reinterpret_cast<const f32x4*>(&pk[1][c16][4 * g4]), mo = *reinterpret_cast<const f32x4*>(&pk[2][c16][4 * g4]);
    if (w < 2) {
      u16x4 hi, lo;
      split4(w ? mu : mo, hi, lo);
      put_frag(ops + (w ? Op::mu(DF) : Op::mo(DF)) * FRAG, lane, hi, lo);
    }
    const f32x4 s = *reinterpret_cast<const f32x4*>(&sc[16 + 4 * g4]);
    mu *= s, mo *= s;
    for (int f = w; f < DF; f += 4) {
      u16x4 xh[2], xl[2], yh[2], yl[2];
#pragma unroll
      for (int e = 0; e < 2; ++e) {
        const int m = 2 * f + e;
        f32x4 x = (f32x4)(0.f), y = (f32x4)(0.f);
#pragma unroll
        for (int r = 0; r < 4; ++r) {
          const float kv = tab[L::KG + 4 * g4 + r][16 * m + c16];
          x = mfma_f(kv, mu[r], x);
          y = mfma_f(kv, mo[r], y);
        }
        const f32x4 qv = *reinterpret_cast<const f32x4*>(&tab[L::QG + c16][16 * m + 4 * g4]);
        split4(x, xh[e], xl[e]);
        split4(qv * rqc - y, yh[e], yl[e]);
      }
      put_frag(ops + (Op::w(DF) + f) * FRAG, lane, xh[0], xh[1]);
      put_frag(ops + (Op::w(DF) + DF + f) * FRAG, lane, xl[0], xl[1]);
      put_frag(ops + (Op::q(DF) + f) * FRAG, lane, yh[0], yh[1]);
      put_frag(ops + (Op::q(DF) + DF + f) * FRAG, lane, yl[0], yl[1]);
    }
  } else {
    if (w == 3) {
      f32x4 mo = *reinterpret_cast<const f32x4*>(&pq[0][c16][4 * g4]);
#pragma unroll
      for (int l = 1; l < 4; ++l) mo += *reinterpret_cast<const f32x4*>(&pq[l][c16][4 * g4]);
      u16x4 hi, lo;
      split4(mo, hi, lo);
      put_frag(ops + Op::mo(DF) * FRAG, lane, hi, lo);
    }
    for (int f = w; f < DF; f += 4) {
      u16x4 yh[2], yl[2];
#pragma unroll
      for (int e = 0; e < 2; ++e)
        split4(*reinterpret_cast<const f32x4*>(&tab[L::QG + c16][16 * (2 * f + e) + 4 * g4]) * sc[c16], yh[e], yl[e]);
      put_frag(ops + (Op::q(DF) + f) * FRAG, lane, yh[0], yh[1]);
      put_frag(ops + (Op::q(DF) + DF + f) * FRAG, lane, yl[0], yl[1]);
    }
  }
}

// grid (blocks, groups).  x [T, C] convolved rows [x | B | C]; dt: column of head 0; kt: the shared fragments
template <int DF>
__global__ __launch_bounds__(256) void ssd_operands_kernel(GatedArgs a, const bf16_t* __restrict__ x, const bf16_t* __restrict__ dt,
                                                           const int32_t* __restrict__ chunks, int nchunk, bf16_t* __restrict__ ops,
                                                           bf16_t* __restrict__ kt) {
  typedef Operands<SSD> Op;
  __shared__ float cb[16][17];
  __shared__ float sg[4][2][16];  // a head per wave: cumulated log2 decay, dt
  const int tid = threadIdx.x, lane = tid & 63, c16 = lane & 15, g4 = lane >> 4;
  const int w = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int g = blockIdx.y, H = a.H, G = a.G, D = a.D, V = a.V, rep = H / G, C = conv_channels(H, G, D, V), tiles = (V + 15) >> 4;
  const int tok0 = chunks[blockIdx.x], nb = chunks[nchunk + blockIdx.x];
  const bf16_t* B = x + (int64_t)tok0 * C + H * V + g * D;
  const bf16_t* Cq = B + G * D;
  bf16_t* sh = kt + ((int64_t)blockIdx.x * G + g) * Op::shared(DF) * FRAG;
  bf16_t* hd = ops + ((int64_t)blockIdx.x * H + g * rep) * Op::size(DF, tiles) * FRAG;
  if (w == 0) {
    f32x4 y = (f32x4)(0.f);
    const int64_t r = (int64_t)min(c16, nb - 1) * C;
#pragma unroll
    for (int f = 0; f < DF; ++f) {
      u16x8 u, v;  // (both in the accumulators' column order)
#pragma unroll
      for (int j = 0; j < 8; ++j) {
        const int d = 32 * f + 16 * (j >> 2) + 4 * g4 + (j & 3);
        u[j] = d < D ? Cq[r + d] : (bf16_t)0;
        v[j] = d < D ? B[r + d] : (bf16_t)0;
      }
      *reinterpret_cast<u16x8*>(sh + f * FRAG + lane * 8) = u;
      y = mfma_k32(u, v, y);
    }
#pragma unroll
    for (int j = 0; j < 4; ++j) cb[4 * g4 + j][c16] = y[j];
  }
  for (int e = tid; e < 2 * DF * 64; e += 256) {  // B^T: lane (channel, four tokens) of a tile of 16 channels
    const int d = (e >> 6) * 16 + (e & 15), t0 = ((e >> 4) & 3) * 4;
    u16x4 v;
#pragma unroll
    for (int j = 0; j < 4; ++j) v[j] = d < D && t0 + j < nb ? B[(int64_t)min(t0 + j, nb - 1) * C + d] : (bf16_t)0;
    *reinterpret_cast<u16x4*>(sh + (Op::k(DF) + (e >> 7)) * FRAG + ((e >> 6) & 1) * 256 + (e & 63) * 4) = v;
  }
  for (int e = tid; e < rep * tiles * 64; e += 256) {  // V as B operands
    const int hh = e / (tiles * 64), y = e - hh * tiles * 64, col = min((y >> 6) * 16 + (y & 15), V - 1), t0 = ((y >> 4) & 3) * 4;
    u16x4 v;
#pragma unroll
    for (int j = 0; j < 4; ++j) v[j] = x[(int64_t)(tok0 + min(t0 + j, nb - 1)) * C + (g * rep + hh) * V + col];
    *reinterpret_cast<u16x4*>(hd + ((int64_t)hh * Op::size(DF, tiles) + Op::v(DF) + (y >> 7)) * FRAG + ((y >> 6) & 1) * 256 +
                              (y & 63) * 4) = v;
  }
  __syncthreads();
  for (int hh = w; hh < rep; hh += 4) {
    const int h = g * rep + hh;
    bf16_t* op = hd + (int64_t)hh * Op::size(DF, tiles) * FRAG;
    const float xx = bf2f(dt[(int64_t)(tok0 + min(c16, nb - 1)) * a.zs + h]) + a.dt_bias[h];
    const float s = c16 < nb ? fmaxf(xx, 0.f) + LN2_G * log2_1p_exp(-fabsf(xx)) : 0.f;
    float l = -a.decay[h] * LOG2E_G * s;
#pragma unroll
    for (int k = 1; k < 16; k <<= 1) {
      const float o = __shfl_up(l, k, 16);
      if (c16 >= k) l += o;
    }
    const float end = __shfl(l, 15, 16);
    if (g4 == 0) {
      sg[w][0][c16] = l;
      sg[w][1][c16] = s;
      float* fl = reinterpret_cast<float*>(op + Op::gc(DF) * FRAG);
      fl[c16] = __builtin_amdgcn_exp2f(l);
      fl[16 + c16] = s * __builtin_amdgcn_exp2f(end - l);
      if (c16 == 0) fl[32] = __builtin_amdgcn_exp2f(end);
    }
    __builtin_amdgcn_wave_barrier();  // (a wave's own row: LDS operations of a wave are in order)
    u16x4 hi, lo;
    f32x4 m;
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      const int jj = 4 * g4 + j;
      m[j] = jj <= c16 ? cb[c16][jj] * __builtin_amdgcn_exp2f(l - sg[w][0][jj]) * sg[w][1][jj] : 0.f;
      if (jj == c16) m[j] += a.skip[h];
    }
    split4(m, hi, lo);
    put_frag(op + Op::mo(DF) * FRAG, lane, hi, lo);
    __builtin_amdgcn_wave_barrier();
  }
}

// ------------------------------------------------------------------------------------ recurrence
// A long sequence of GLA or SSD, whose decays act on S alone, may be cut into parts: with F the product of a part's gc and L
// what it makes of a state of zeros, S <- F S + L.  LOCAL makes F and L of every part but the last, then PARTS runs all of them
// at once, each from what those ahead of it leave.
enum { WHOLE = 0, LOCAL = 1, PARTS = 2 };

template <int KIND, int DF, int NV, int NW, int MODE>
struct Ring {
  static constexpr int VF = (NV * NW + 1) / 2;  // value fragments of a workgroup
  static constexpr int SKIP = MODE == LOCAL ? Operands<KIND>::k(DF) : 0;  // (no reading: Q stays away)
  static constexpr int HEAD = Operands<KIND>::v(DF), SHARED = Operands<KIND>::shared(DF), N = SHARED + HEAD + VF - SKIP;
  static constexpr int J = (N + NW - 1) / NW;  // loads of a wave
  static constexpr int SLOTS = N <= 40 ? 4 : 3;
  static constexpr size_t BYTES = (size_t)SLOTS * N * 1024;
  // memory operations that follow a block's loads until they are waited for: the later blocks' and their stores
  static constexpr int NEWER = (J + (MODE == LOCAL ? 0 : 4 * NV)) * (SLOTS - 2), WAIT = NEWER > 63 ? 63 : NEWER;
};

// seqs [4, nseq]: first token, tokens, first block, blocks; with parts [5, nseq], a part's number in its sequence last.  starts
// [nseq, H, D, V]: the state ahead of a first part, the L of the part before for the others;  fade [nseq, H, D]: F (SSD: the
// first of D).  out fp32 [T + 1, H V]: lanes past the end store into the last row, so
// that every wave has as many memory operations under way.  Workgroups of the value slices of one (sequence, head) lie on one XCD.
template <int KIND, int DF, int NV, int NW, int MODE>
__global__ __launch_bounds__(NW * 64, DF > 4 ? 1 : 2) void gated_blocks_kernel(GatedArgs a, const int32_t* __restrict__ seqs, int nseq,
                                                                 const bf16_t* __restrict__ ops, const bf16_t* __restrict__ kt,
                                                                 float* __restrict__ out, int T, float* __restrict__ starts,
                                                                 float* __restrict__ fade) {
  static_assert(MODE == WHOLE || KIND != DELTA, "the delta rule's parts are no F S + L with a diagonal F");
  constexpr int DT = 2 * DF;
  typedef Operands<KIND> Op;
  typedef Ring<KIND, DF, NV, NW, MODE> R;
  extern __shared__ __attribute__((aligned(1024))) char smem[];
  typedef __attribute__((address_space(3))) void* lptr_t;
  typedef __attribute__((address_space(1))) const void* gptr_t;
  const int lane = threadIdx.x & 63, c16 = lane & 15, g4 = lane >> 4;
  const int w = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int H = a.H, D = a.D, V = a.V, tiles = (V + 15) >> 4;
  const int per = (tiles + NV * NW - 1) / (NV * NW);  // workgroups of a (sequence, head)
  const int y = blockIdx.x >> 3, grp = (blockIdx.x & 7) + 8 * (y / per), t0 = (y % per) * NV * NW;
  if (grp >= nseq * H) return;
  const int s = grp / H, h = grp - s * H, gh = h / (H / a.G);
  const int tok0 = seqs[s], ntok = seqs[nseq + s], blk0 = seqs[2 * nseq + s], nblk = seqs[3 * nseq + s];
  const int64_t row = a.q_seq[tok0];
  const bool fresh = a.q_ctx[tok0] <= 1;
  float* state = a.state + (row * H + h) * (int64_t)D * V;
  const int part = MODE == WHOLE ? 0 : seqs[4 * nseq + s];
  const bool last = MODE == WHOLE || s + 1 == nseq || seqs[4 * nseq + s + 1] == 0;
  if (MODE == LOCAL && last) return;
  const int64_t spitch = (int64_t)H * D * V;  // of a part in starts
  float* start = MODE == WHOLE ? nullptr : starts + s * spitch + (int64_t)h * D * V;
  float* fd = MODE == WHOLE ? nullptr : fade + ((int64_t)s * H + h) * D;

  // this wave's fragments of a block, and their step to the next one (bytes)
  const int64_t hstep = (int64_t)H * Op::size(DF, tiles) * 1024, gstep = (int64_t)a.G * R::SHARED * 1024;
  const char* fp[R::J];
  bool of_head[R::J];
#pragma unroll
  for (int j = 0; j < R::J; ++j) {
    const int f = R::SKIP + min(w + NW * j, R::N - 1);  // (one too many: the last one again)
    of_head[j] = f >= R::SHARED;
    const int hf = f - R::SHARED;
    if (!of_head[j]) fp[j] = (const char*)kt + (((int64_t)blk0 * a.G + gh) * R::SHARED + f) * 1024;
    else fp[j] = (const char*)ops + (((int64_t)blk0 * H + h) * Op::size(DF, tiles) +
                                     (hf < R::HEAD ? hf : min(Op::v(DF) + t0 / 2 + hf - R::HEAD, Op::size(DF, tiles) - 1))) * 1024;
    fp[j] += lane * 16;
  }
  auto issue = [&](int b) {
    const int64_t k = min(b, nblk - 1);  // (past the end: a slot that is not read)
    char* slot = smem + (b % R::SLOTS) * R::N * 1024;
#pragma unroll
    for (int j = 0; j < R::J; ++j)
      __builtin_amdgcn_global_load_lds((gptr_t)(fp[j] + k * (of_head[j] ? hstep : gstep)),
                                       (lptr_t)(slot + min(w + NW * j, R::N - 1) * 1024), 16, 0, 0);
  };
#pragma unroll
  for (int b = 0; b < R::SLOTS; ++b) issue(b);

  int col[NV];
#pragma unroll
  for (int n = 0; n < NV; ++n) col[n] = (t0 + w * NV + n) * 16 + c16;
  f32x4 S[DT][NV];
#pragma unroll
  for (int m = 0; m < DT; ++m)
#pragma unroll
    for (int n = 0; n < NV; ++n)
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        const int d = 16 * m + 4 * g4 + r;
        const bool ok = d < D && col[n] < V;
        const int64_t at = (int64_t)d * V + col[n];
        float x = 0.f;
        if (MODE == WHOLE || (part == 0 && (MODE == LOCAL || last))) {
          x = !fresh && ok ? state[at] : 0.f;
          if (MODE == LOCAL && ok) start[at] = x;
        } else if (MODE == PARTS) {
          x = ok ? start[at - (part > 0 ? part - 1 : 0) * spitch] : 0.f;
        }
        S[m][n][r] = x;
      }
  if constexpr (MODE == PARTS) {
    for (int j = 2; j <= part; ++j) {  // S <- F S + L
      const float *f = fd + (int64_t)(j - 1 - part) * H * D, *l = start - (part - j) * spitch;
#pragma unroll
      for (int m = 0; m < DT; ++m)
#pragma unroll
        for (int r = 0; r < 4; ++r) {
          const int d = min(16 * m + 4 * g4 + r, D - 1);
          const float fx = f[KIND == SSD ? 0 : d];
#pragma unroll
          for (int n = 0; n < NV; ++n) S[m][n][r] = S[m][n][r] * fx + l[(int64_t)d * V + min(col[n], V - 1)];
        }
    }
  }
  f32x4 F[MODE == LOCAL ? (KIND == SSD ? 1 : DT) : 1];
#pragma unroll
  for (int m = 0; m < (MODE == LOCAL && KIND != SSD ? DT : 1); ++m) F[m] = (f32x4)(1.f);
  // S and the next block's Q and W as operands: made and read while the block before it is finished
  u16x8 sh[DF][NV], sl[DF][NV], qh[DF], ql[KIND == SSD ? 1 : DF], wh[KIND == DELTA ? DF : 1], wl[KIND == DELTA ? DF : 1];
  auto split = [&](int f) {
#pragma unroll
    for (int n = 0; n < NV; ++n) {
      u16x4 h0, l0, h1, l1;
      split4(S[2 * f][n], h0, l0);
      split4(S[2 * f + 1][n], h1, l1);
      sh[f][n] = cat4(h0, h1);
      sl[f][n] = cat4(l0, l1);
    }
  };
  auto read_q = [&](int b) {
    const bf16_t* L = reinterpret_cast<const bf16_t*>(smem + (b % R::SLOTS) * R::N * 1024);
#pragma unroll
    for (int f = 0; f < DF; ++f) {
      qh[f] = *reinterpret_cast<const u16x8*>(L + (Op::q(DF) + f) * FRAG + lane * 8);
      if constexpr (KIND != SSD) ql[f] = *reinterpret_cast<const u16x8*>(L + (Op::q(DF) + DF + f) * FRAG + lane * 8);
      if constexpr (KIND == DELTA) {
        wh[f] = *reinterpret_cast<const u16x8*>(L + (Op::w(DF) + f) * FRAG + lane * 8);
        wl[f] = *reinterpret_cast<const u16x8*>(L + (Op::w(DF) + DF + f) * FRAG + lane * 8);
      }
    }
  };
  asm volatile("s_waitcnt vmcnt(0)" ::: "memory");  // (later waits count the stores of the blocks before)
  lds_wait_barrier();
  if constexpr (MODE != LOCAL) {
    read_q(0);
#pragma unroll
    for (int f = 0; f < DF; ++f) split(f);
  }
  for (int b = 0; b < nblk; ++b) {
    const bf16_t* L = reinterpret_cast<const bf16_t*>(smem + (b % R::SLOTS) * R::N * 1024);
    auto head = [&](int f) { return L + (R::SHARED - R::SKIP + f) * FRAG; };
    u16x8 vv[NV];  // {V, V}
#pragma unroll
    for (int n = 0; n < NV; ++n) {
      const int x = NV * NW == 1 ? t0 & 1 : w * NV + n;
      const u16x4 v = *reinterpret_cast<const u16x4*>(head(R::HEAD + (x >> 1)) + (x & 1) * 256 + lane * 4);
      vv[n] = cat4(v, v);
    }
    const u16x8 mo = *reinterpret_cast<const u16x8*>(head(Op::mo(DF)) + lane * 8);
    u16x8 mu;
    if constexpr (KIND == DELTA) mu = *reinterpret_cast<const u16x8*>(head(Op::mu(DF)) + lane * 8);
    const float* gcp = reinterpret_cast<const float*>(head(Op::gc(DF)));
    f32x4 fq, fu;
    if constexpr (KIND == SSD) {
      fq = *reinterpret_cast<const f32x4*>(gcp + 4 * g4);
      fu = *reinterpret_cast<const f32x4*>(gcp + 16 + 4 * g4);
    }
    u16x8 k[DT];
    f32x4 gc[KIND == SSD ? 1 : DT];
    if constexpr (KIND == SSD) gc[0] = (f32x4)(gcp[32]);
#pragma unroll
    for (int m = 0; m < DT; ++m) {
      if constexpr (KIND == SSD) {
        const u16x4 x = *reinterpret_cast<const u16x4*>(L + (Op::k(DF) - R::SKIP + (m >> 1)) * FRAG + (m & 1) * 256 + lane * 4);
        k[m] = cat4(x, x);
      } else {
        k[m] = *reinterpret_cast<const u16x8*>(L + (Op::k(DF) - R::SKIP + m) * FRAG + lane * 8);
        gc[m] = *reinterpret_cast<const f32x4*>(gcp + 16 * m + 4 * g4);
      }
    }
    f32x4 O[NV], U[NV], O2[NV], U2[NV];  // (two chains each: large and small terms)
#pragma unroll
    for (int n = 0; n < NV; ++n) O[n] = U[n] = O2[n] = U2[n] = (f32x4)(0.f);
#pragma unroll
    for (int f = 0; f < (MODE == LOCAL ? 0 : DF); ++f)
#pragma unroll
      for (int n = 0; n < NV; ++n) {
        if constexpr (KIND == DELTA) {
          U[n] = mfma_k32(wh[f], sh[f][n], U[n]);
          U2[n] = mfma_k32(wl[f], sh[f][n], U2[n]);
          U2[n] = mfma_k32(wh[f], sl[f][n], U2[n]);
        }
        O[n] = mfma_k32(qh[f], sh[f][n], O[n]);
        if constexpr (KIND != SSD) O2[n] = mfma_k32(ql[f], sh[f][n], O2[n]);
        O2[n] = mfma_k32(qh[f], sl[f][n], O2[n]);
      }
    asm volatile("s_waitcnt vmcnt(%0)" ::"n"(R::WAIT) : "memory");  // block b + 1 has landed
    lds_wait_barrier();                                            // for all waves, and all have read block b
    issue(b + R::SLOTS);
    if constexpr (MODE != LOCAL) read_q(b + 1);
    u16x8 uu[NV], uv[NV];  // what K meets: SSD {hi, lo}; DELTA {hi, hi}, {lo, lo}; GLA {V, V}
#pragma unroll
    for (int n = 0; n < NV; ++n) {
      O[n] += O2[n];
      u16x4 hi, lo;
      if constexpr (KIND == SSD) {
        O[n] *= fq;
        f32x4 x;
#pragma unroll
        for (int j = 0; j < 4; ++j) x[j] = bf2f(vv[n][j]) * fu[j];
        split4(x, hi, lo);
        uu[n] = cat4(hi, lo);
      }
      if constexpr (KIND == DELTA) {
        split4(mfma_k32(mu, vv[n], -(U[n] + U2[n])), hi, lo);
        uu[n] = cat4(hi, hi);
        uv[n] = cat4(lo, lo);
      }
      if constexpr (KIND == GLA) uu[n] = vv[n];
      if constexpr (MODE != LOCAL) O[n] = mfma_k32(mo, vv[n], O[n]);
    }
#pragma unroll
    for (int m = 0; m < DT; ++m) {
#pragma unroll
      for (int n = 0; n < NV; ++n) {
        S[m][n] *= gc[KIND == SSD ? 0 : m];
        if constexpr (KIND == DELTA) S[m][n] = mfma_k32(k[m], uv[n], S[m][n]);
        S[m][n] = mfma_k32(k[m], uu[n], S[m][n]);
      }
      if (MODE != LOCAL && (m & 1)) split(m >> 1);
      if (MODE == LOCAL && (m == 0 || KIND != SSD)) F[KIND == SSD ? 0 : m] *= gc[KIND == SSD ? 0 : m];
    }
#pragma unroll
    for (int n = 0; n < (MODE == LOCAL ? 0 : NV); ++n)
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        const int t = 16 * b + 4 * g4 + r;
        const bool ok = t < ntok && col[n] < V;
        out[(int64_t)(ok ? tok0 + t : T) * H * V + h * V + (ok ? col[n] : 0)] = O[n][r];
      }
  }
  asm volatile("s_waitcnt vmcnt(0)" ::: "memory");  // (the ring's last loads end before the workgroup does)
#pragma unroll
  for (int m = 0; m < DT; ++m)
#pragma unroll
    for (int n = 0; n < NV; ++n)
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        const int d = 16 * m + 4 * g4 + r;
        float* to = MODE == LOCAL ? start + spitch : state;
        if (last != (MODE == LOCAL) && d < D && col[n] < V) to[(int64_t)d * V + col[n]] = S[m][n][r];
      }
  if constexpr (MODE == LOCAL) {
    if (t0 + w == 0 && c16 == 0) {  // (the same in every column)
#pragma unroll
      for (int m = 0; m < (KIND == SSD ? 1 : DT); ++m)
#pragma unroll
        for (int r = 0; r < 4; ++r)
          if (const int d = 16 * m + 4 * g4 + r; d < (KIND == SSD ? 1 : D)) fd[d] = F[m][r];
    }
  }
}

static int chunk_df(int D) { return D <= 32 ? 1 : D <= 64 ? 2 : D <= 128 ? 4 : 8; }

#define MP_DF(D_, M_)          \
  switch (chunk_df(D_)) {      \
    case 1: M_(1) break;       \
    case 2: M_(2) break;       \
    case 4: M_(4) break;       \
    default: M_(8) break;      \
  }

template <int KIND>
static int launch_operands(const GatedArgs& a, const ChunkIn& in, hipStream_t stream) {
#define MP_GO(DF_)                                                                                                      \
  {                                                                                                                     \
    constexpr size_t lds = OperandLds<KIND, DF_>::BYTES;                                                                \
    if (lds > 65536)                                                                                                    \
      (void)hipFuncSetAttribute((const void*)gated_operands_kernel<KIND, DF_>, hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds); \
    hipLaunchKernelGGL((gated_operands_kernel<KIND, DF_>), dim3(in.nchunk, a.H), dim3(256), lds, stream, a, in);        \
  }
  MP_DF(a.D, MP_GO)
#undef MP_GO
  return (int)hipGetLastError();
}

struct Seqs {
  const int32_t* p;  // [4, n], or with parts [5, n]
  int n;
  float *starts, *fade;  // of parts
};

template <int KIND, int DF, int NV, int NW, int MODE>
static int launch_blocks_as(const GatedArgs& a, const Seqs& q, const bf16_t* ops, const bf16_t* kt, float* out, int T,
                            hipStream_t stream) {
  typedef Ring<KIND, DF, NV, NW, MODE> R;
  static_assert(R::BYTES <= 160 * 1024, "the ring fits LDS");
  const int tiles = (a.V + 15) / 16, per = (tiles + NV * NW - 1) / (NV * NW);
  const int64_t grid = 8 * (((int64_t)q.n * a.H + 7) / 8) * per;
  if (grid > 0x7fffffff) return -1;
  (void)hipFuncSetAttribute((const void*)gated_blocks_kernel<KIND, DF, NV, NW, MODE>, hipFuncAttributeMaxDynamicSharedMemorySize, (int)R::BYTES);
  hipLaunchKernelGGL((gated_blocks_kernel<KIND, DF, NV, NW, MODE>), dim3((unsigned)grid), dim3(64 * NW), R::BYTES, stream, a, q.p, q.n, ops,
                     kt, out, T, q.starts, q.fade);
  return (int)hipGetLastError();
}

// few sequences: a wave per workgroup, to have as many as there are CUs; else a workgroup takes up to 128 value columns
template <int KIND, int DF, int MODE>
static int launch_blocks_of(const GatedArgs& a, const Seqs& q, const bf16_t* ops, const bf16_t* kt, float* out, int T,
                            hipStream_t stream) {
  const int tiles = (a.V + 15) / 16;
  if constexpr (DF <= 4) {
    if ((int64_t)q.n * a.H * tiles > 512) {
      if (tiles > 4) return launch_blocks_as<KIND, DF, 1, 8, MODE>(a, q, ops, kt, out, T, stream);
      if (tiles > 2) return launch_blocks_as<KIND, DF, 1, 4, MODE>(a, q, ops, kt, out, T, stream);
      if (tiles > 1) return launch_blocks_as<KIND, DF, 1, 2, MODE>(a, q, ops, kt, out, T, stream);
    }
  }
  return launch_blocks_as<KIND, DF, 1, 1, MODE>(a, q, ops, kt, out, T, stream);
}

template <int KIND>
static int launch_blocks(const GatedArgs& a, const Seqs& q, const bf16_t* ops, const bf16_t* kt, float* out, int T, hipStream_t stream) {
  if constexpr (KIND != DELTA) {
    if (q.starts != nullptr) {
#define MP_GB(DF_)                                                                              \
  {                                                                                             \
    const int rc = launch_blocks_of<KIND, DF_, LOCAL>(a, q, ops, kt, out, T, stream);            \
    return rc ? rc : launch_blocks_of<KIND, DF_, PARTS>(a, q, ops, kt, out, T, stream);          \
  }
      MP_DF(a.D, MP_GB)
#undef MP_GB
    }
  }
#define MP_GB(DF_) return launch_blocks_of<KIND, DF_, WHOLE>(a, q, ops, kt, out, T, stream);
  MP_DF(a.D, MP_GB)
#undef MP_GB
}

}  // namespace mp

// bf16 elements of a (block, head)'s operands, and (SSD) of a (block, group)'s
extern "C" int64_t mp_gated_operands(int kind, int D, int V) {
  using namespace mp;
  const int df = chunk_df(D), tiles = (V + 15) / 16;
  return (int64_t)FRAG * (kind == DELTA ? Operands<DELTA>::size(df, tiles)
                                        : kind == GLA ? Operands<GLA>::size(df, tiles) : Operands<SSD>::size(df, tiles));
}
extern "C" int64_t mp_gated_shared(int D) { return (int64_t)mp::FRAG * mp::Operands<mp::SSD>::shared(mp::chunk_df(D)); }

// convolution of z's columns from zcol on into out [T, C]; unit [T, 2 G] (DELTA)
extern "C" int mp_short_conv(int kind, const mp::GatedArgs* args, int zcol, const int32_t* chunks, int nchunk, void* out, float* unit,
                             hipStream_t stream) {
  using namespace mp;
  (void)hipGetLastError();
  if (nchunk == 0) return 0;
  const GatedArgs& a = *args;
  const int most = a.D > a.V ? a.D : a.V;
  if (a.taps > CONV_TAPS || most > 64 * CONV_CH || (kind == DELTA && unit == nullptr)) return -1;
  const dim3 grid(nchunk, (2 * a.G + a.H + 3) / 4);
  const bool pair = a.D % 2 == 0 && a.V % 2 == 0 && a.zs % 2 == 0 && (zcol & 1) == 0 && (uintptr_t)a.z % 4 == 0;
#define MP_SC(N_, P_)                                                                                                        \
  {                                                                                                                         \
    if (a.taps == 4) hipLaunchKernelGGL((short_conv_kernel<N_, 4, P_>), grid, dim3(256), 0, stream, a, kind, zcol, chunks, nchunk, (bf16_t*)out, unit); \
    else hipLaunchKernelGGL((short_conv_kernel<N_, 0, P_>), grid, dim3(256), 0, stream, a, kind, zcol, chunks, nchunk, (bf16_t*)out, unit);             \
  }
  if (pair) {
    if (most <= 128) MP_SC(2, true) else if (most <= 256) MP_SC(4, true) else MP_SC(8, true)
  } else {
    if (most <= 64) MP_SC(1, false) else if (most <= 256) MP_SC(4, false) else MP_SC(8, false)
  }
#undef MP_SC
  return (int)hipGetLastError();
}

// Blocks' operands, then the recurrence: out fp32 [T + 1, H V].  q, k, v: rows' first columns of head 0 (SSD: v the convolved rows
// x); dec: GLA, DELTA [T, H D] inputs of the decays; beta: DELTA's beta, SSD's dt, column of head 0 in a row of z.  starts, fade
// (or null): GLA and SSD have their sequences in parts, seqs [5, nseq]
extern "C" int mp_gated_chunk(int kind, const mp::GatedArgs* args, const void* q, const void* k, const void* v, int64_t rs,
                              const void* dec, int64_t ds, const void* beta, const float* unit, const int32_t* chunks, int nchunk,
                              const int32_t* seqs, int nseq, float* starts, float* fade, void* ops, void* kt, float* out, int T,
                              hipStream_t stream) {
  using namespace mp;
  (void)hipGetLastError();
  if (nchunk == 0 || nseq == 0) return 0;
  const Seqs sq{seqs, nseq, starts, fade};
  const GatedArgs& a = *args;
  if (a.D > 256 || a.H > 65535 || a.G < 1 || a.H % a.G) return -1;
  const bf16_t* vp = (const bf16_t*)v;
  bf16_t *op = (bf16_t*)ops, *kp = (bf16_t*)kt;
  int rc;
  if (kind == SSD) {
#define MP_SO(DF_)                                                                                                              \
  hipLaunchKernelGGL((ssd_operands_kernel<DF_>), dim3(nchunk, a.G), dim3(256), 0, stream, a, vp, (const bf16_t*)beta, chunks, nchunk, \
                     op, kp);
    MP_DF(a.D, MP_SO)
#undef MP_SO
    rc = (int)hipGetLastError();
    return rc ? rc : launch_blocks<SSD>(a, sq, op, kp, out, T, stream);
  }
  const ChunkIn in{(const bf16_t*)q, (const bf16_t*)k, (const bf16_t*)dec, rs, rs, ds, vp, rs, (const bf16_t*)beta, a.zs, unit, chunks,
                   nchunk, op};
  rc = kind == DELTA ? launch_operands<DELTA>(a, in, stream) : launch_operands<GLA>(a, in, stream);
  if (rc) return rc;
  return kind == DELTA ? launch_blocks<DELTA>(a, sq, op, nullptr, out, T, stream)
                       : launch_blocks<GLA>(a, sq, op, nullptr, out, T, stream);
}
