// Kernels of the stateless fine-tuning path (runtime/autograd_stage.py): causal attention over whole sequences with its
// gradients, the norm, rotary and silu-gate steps between the projections and their gradients.
//
// The reference's server recomputes the span's forward with autograd and differentiates it
// (petals/server/block_functions.py:84-141).  Here the frozen weights' blocks are differentiated by hand, so nothing of
// size [heads, T, T] exists: a block's forward keeps its input, q / k / v, the fp32 attention output, one number per
// (token, head) and the gate / up rows.
//
// Attention.  All products are 16x16x32 bf16 MFMA over exact bf16 operands (q, k, v, and the incoming gradient), their
// accumulators fp32.  What is fp32 in between - probabilities P and score gradients dS - enters the next product as
// three bf16 terms, 8 significant bits each, whose sum is the fp32 number: no step is held in fewer bits than 32-bit
// products of 32-bit operands would.  (With two terms, 16 bits, the output was 7 to 11 times as far from 64-bit attention
// as with those, for 10 to 15 % less time.)
// Orientation: a wave makes scores with the dimension it reduces over LATER in the accumulator's rows; P and dS are then
// operands of the next product as they lie in the registers (k order permuted: 4 rows of one 16-row subtile, 4 of the
// next), the other operand comes from the same row-major LDS tile through the transposing LDS read, and the outputs have
// 4 consecutive columns a lane.
#include "common.h"

namespace mp {

typedef __attribute__((ext_vector_type(8))) __bf16 bf16x8_t;
typedef short s16x4_t __attribute__((ext_vector_type(4)));

__device__ __forceinline__ f32x4 mfma16(const u16x8& a, const u16x8& b, const f32x4& c) {
  return __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(bf16x8_t, a), __builtin_bit_cast(bf16x8_t, b), c, 0, 0,
                                                 0);
}
// each group of 16 lanes reads 4 rows x 16 columns and gets them transposed: lane i column i, 4 rows
__device__ __forceinline__ u16x4 tr_read(const unsigned char* p) {
  const s16x4_t v = __builtin_amdgcn_ds_read_tr16_b64_v4i16(
      (__attribute__((address_space(3))) s16x4_t*)(const_cast<unsigned char*>(p)));
  return __builtin_bit_cast(u16x4, v);
}

struct TrainAttn {
  const bf16_t* qkv;   // [B T, ld]: q heads, k heads, v heads, q and k turned
  int64_t ld;
  int T, nh, nkv;
  float scale;
  bf16_t* out;         // forward: [B T, nh D]
  float* out32;        // the same in fp32, or nullptr
  float* lse;          // [B, nh, T] log2 of the softmax's denominator, or nullptr
  const bf16_t* dout;  // backward: gradient of ``out``
  float* delta;        // [B, nh, T] sum over d of dout out
  const float* cs;     // [T, D] cos (first half), sin of the rotary angles
  bf16_t* dqkv;        // [B T, ld]
  float* part;         // [2, B T, nh, D] keys' and values' gradients per query head
};

constexpr int TPAD = 16;  // bytes after an LDS row: 16 rows' 16-byte chunks fall into 16 different bank groups

// rows r0 .. r0 + ROWS - 1 of a [T, D] matrix (row stride ``ld``) on their way into an LDS tile: fetched into registers a
// step ahead, rows past T as zeros
template <int D, int ROWS>
struct Tile {
  static constexpr int LD = 2 * D + TPAD, BYTES = ROWS * LD, CH = D / 8, N = ROWS * CH / 256;
  static_assert(ROWS * CH % 256 == 0, "whole chunks per thread");
  u16x8 v[N];
  __device__ __forceinline__ void fetch(const bf16_t* p, int64_t ld, int r0, int T) {
    const char* base = reinterpret_cast<const char*>(p + (int64_t)r0 * ld);
    const int last = min(ROWS, T - r0) - 1;
#pragma unroll
    for (int j = 0; j < N; ++j) {
      const int c = threadIdx.x + 256 * j;
      v[j] = *reinterpret_cast<const u16x8*>(base + (uint32_t)min(c / CH, last) * (uint32_t)(ld * 2) + (c % CH) * 16);
    }
  }
  // ``rows`` of them are the matrix's, the others zeros
  __device__ __forceinline__ void stash(unsigned char* lds, int rows) {
    if (rows < ROWS) {
#pragma unroll
      for (int j = 0; j < N; ++j)
        if ((int)(threadIdx.x + 256 * j) / CH >= rows) v[j] = (u16x8)(0);
    }
#pragma unroll
    for (int j = 0; j < N; ++j) {
      const int c = threadIdx.x + 256 * j;
      *reinterpret_cast<u16x8*>(lds + (c / CH) * LD + (c % CH) * 16) = v[j];
    }
  }
};

// 16 rows' operand (row = lane % 16, 8 columns from 32 s + 8 (lane / 16)) of a row-major LDS tile
template <int D>
__device__ __forceinline__ u16x8 row_frag(const unsigned char* t, int row0, int s) {
  const int lane = threadIdx.x & 63;
  return *reinterpret_cast<const u16x8*>(t + (row0 + (lane & 15)) * Tile<D, 64>::LD + 64 * s + 16 * (lane >> 4));
}
// the same tile transposed: operand rows are columns 16 dt + lane % 16, its k order rows row0 + 4 g .. + 3 and
// row0 + 16 + 4 g .. + 3 (g = lane / 16)
template <int D>
__device__ __forceinline__ u16x8 col_frag(const unsigned char* t, int row0, int dt) {
  const int lane = threadIdx.x & 63, g = lane >> 4, i = lane & 15;
  const unsigned char* p = t + (row0 + 4 * g + (i >> 2)) * Tile<D, 64>::LD + 32 * dt + 8 * (i & 3);
  const u16x4 a = tr_read(p), b = tr_read(p + 16 * Tile<D, 64>::LD);
  return (u16x8){a[0], a[1], a[2], a[3], b[0], b[1], b[2], b[3]};
}
// 8 fp32 (two subtiles' 4) as three operands; the remainders are exact, so is their sum
__device__ __forceinline__ void split8(const f32x4& a, const f32x4& b, u16x8 (&t)[3]) {
#pragma unroll
  for (int j = 0; j < 8; ++j) {
    float r = j < 4 ? a[j & 3] : b[j & 3];
#pragma unroll
    for (int i = 0; i < 3; ++i) {
      t[i][j] = f2bf(r);
      r -= bf2f(t[i][j]);
    }
  }
}

// Forward and dQ: a workgroup has 64 queries of one head, 16 a wave, and walks the keys 64 at a time.
// Bound by the chain of a tile's steps, so three workgroups share a CU: one LDS buffer, the next tile's rows in registers
// (two buffers of 70 KB let two workgroups in).  2 x 777 tokens, 32 heads of 128 (8 kv heads): forward 59 -> 46 us, dQ, dK and dV
// together 179 -> 144.  The fp32 batched products, softmax passes and copies that it replaced were most of 12.3 ms for two
// blocks' forward and backward requests.
template <int D, bool GRAD>
__global__ __launch_bounds__(256, 3) void train_attn_q_kernel(TrainAttn a) {
  constexpr int KS = D / 32, DT = D / 16;
  typedef Tile<D, 64> KTile;
  __shared__ __attribute__((aligned(16))) unsigned char smem[2][KTile::BYTES];  // [K | V]
  const int lane = threadIdx.x & 63, w = threadIdx.x >> 6, g = lane >> 4;
  const int h = blockIdx.y, b = blockIdx.z, kvh = h / (a.nh / a.nkv);
  const int q0 = (gridDim.x - 1 - blockIdx.x) * 64;  // longest context first
  const int q = q0 + 16 * w + (lane & 15);
  const bool live = q < a.T;
  const int64_t row = (int64_t)b * a.T + min(q, a.T - 1);
  const bf16_t* base = a.qkv + (int64_t)b * a.T * a.ld;
  const bf16_t *kp = base + (a.nh + kvh) * D, *vp = base + (a.nh + a.nkv + kvh) * D;
  const int64_t stat = ((int64_t)b * a.nh + h) * a.T + min(q, a.T - 1);
  const float c2 = a.scale * 1.4426950408889634f;

  u16x8 qf[KS], gf[KS];
  float delta = 0.f, lse = 0.f;
#pragma unroll
  for (int s = 0; s < KS; ++s) {
    qf[s] = live ? *reinterpret_cast<const u16x8*>(a.qkv + row * a.ld + h * D + 32 * s + 8 * g) : (u16x8)(0);
    if (GRAD) {
      const int64_t at = (row * a.nh + h) * D + 32 * s + 8 * g;
      gf[s] = live ? *reinterpret_cast<const u16x8*>(a.dout + at) : (u16x8)(0);
      const f32x4 o0 = *reinterpret_cast<const f32x4*>(a.out32 + at), o1 = *reinterpret_cast<const f32x4*>(a.out32 + at + 4);
#pragma unroll
      for (int j = 0; j < 4; ++j) delta += bf2f(gf[s][j]) * o0[j] + bf2f(gf[s][j + 4]) * o1[j];
    }
  }
  if (GRAD) {
    delta += __shfl_xor(delta, 16, 64);
    delta += __shfl_xor(delta, 32, 64);
    lse = a.lse[stat];
    if (live && g == 0) a.delta[stat] = delta;
  }
  f32x4 o[DT];
#pragma unroll
  for (int dt = 0; dt < DT; ++dt) o[dt] = (f32x4)(0.f);
  float m = -INFINITY, l = 0.f;

  KTile kt, vt;
  const int end = min(q0 + 64, a.T);
  kt.fetch(kp, a.ld, 0, a.T), vt.fetch(vp, a.ld, 0, a.T);
  for (int k0 = 0; k0 < end; k0 += 64) {
    kt.stash(smem[0], a.T - k0), vt.stash(smem[1], a.T - k0);
    __syncthreads();
    if (k0 + 64 < end) kt.fetch(kp, a.ld, k0 + 64, a.T), vt.fetch(vp, a.ld, k0 + 64, a.T);
    const unsigned char *K = smem[0], *V = smem[1];
    if (k0 <= q0 + 16 * w + 15) {
      f32x4 s[4], dp[4];
#pragma unroll
      for (int st = 0; st < 4; ++st) {
        s[st] = dp[st] = (f32x4)(0.f);
#pragma unroll
        for (int ks = 0; ks < KS; ++ks) {
          s[st] = mfma16(row_frag<D>(K, 16 * st, ks), qf[ks], s[st]);
          if (GRAD) dp[st] = mfma16(row_frag<D>(V, 16 * st, ks), gf[ks], dp[st]);
        }
      }
      if (k0 + 63 > q0 + 16 * w) {  // the diagonal
#pragma unroll
        for (int st = 0; st < 4; ++st)
#pragma unroll
          for (int j = 0; j < 4; ++j)
            if (k0 + 16 * st + 4 * g + j > q) s[st][j] = -INFINITY;
      }
      if (GRAD) {
#pragma unroll
        for (int st = 0; st < 4; ++st)
#pragma unroll
          for (int j = 0; j < 4; ++j) {
            const float p = __builtin_amdgcn_exp2f(__builtin_fmaf(s[st][j], c2, -lse));
            s[st][j] = p == 0.f ? 0.f : p * (dp[st][j] - delta) * a.scale;  // (0 times an infinite dp: not seen)
          }
      } else {
        float top = -INFINITY;
#pragma unroll
        for (int st = 0; st < 4; ++st)
#pragma unroll
          for (int j = 0; j < 4; ++j) top = fmaxf(top, s[st][j]);
        top = fmaxf(top, __shfl_xor(top, 16, 64));
        top = fmaxf(top, __shfl_xor(top, 32, 64)) * c2;
        const float mn = fmaxf(m, top), mu = mn == -INFINITY ? 0.f : mn;
        const float alpha = __builtin_amdgcn_exp2f(m - mu);
        m = mn;
        if (__any(alpha != 1.f)) {  // (most tiles leave every maximum where it was)
          l *= alpha;
#pragma unroll
          for (int dt = 0; dt < DT; ++dt) o[dt] *= alpha;
        }
#pragma unroll
        for (int st = 0; st < 4; ++st)
#pragma unroll
          for (int j = 0; j < 4; ++j) {
            s[st][j] = __builtin_amdgcn_exp2f(__builtin_fmaf(s[st][j], c2, -mu));
            l += s[st][j];
          }
      }
      const unsigned char* R = GRAD ? K : V;
#pragma unroll
      for (int half = 0; half < 2; ++half) {
        u16x8 t[3];
        split8(s[2 * half], s[2 * half + 1], t);
#pragma unroll
        for (int dt = 0; dt < DT; ++dt) {
          const u16x8 f = col_frag<D>(R, 32 * half, dt);
#pragma unroll
          for (int i = 2; i >= 0; --i) o[dt] = mfma16(f, t[i], o[dt]);
        }
      }
    }
    __syncthreads();
  }
  if (!live) return;
  if (GRAD) {  // dQ turned back: entry d pairs with d + D / 2, which lies DT / 2 accumulators on
    const float* cs = a.cs + (int64_t)q * D;
    bf16_t* y = a.dqkv + row * a.ld + h * D;
#pragma unroll
    for (int dt = 0; dt < DT / 2; ++dt) {
      u16x4 u, v;
#pragma unroll
      for (int j = 0; j < 4; ++j) {
        const int d = 16 * dt + 4 * g + j;
        const float c = cs[d], s = cs[D / 2 + d];
        u[j] = f2bf(o[dt][j] * c + o[dt + DT / 2][j] * s);
        v[j] = f2bf(o[dt + DT / 2][j] * c - o[dt][j] * s);
      }
      *reinterpret_cast<u16x4*>(y + 16 * dt + 4 * g) = u;
      *reinterpret_cast<u16x4*>(y + D / 2 + 16 * dt + 4 * g) = v;
    }
    return;
  }
  l += __shfl_xor(l, 16, 64);
  l += __shfl_xor(l, 32, 64);
  const float inv = 1.f / l;
  const int64_t at = (row * a.nh + h) * D + 4 * g;
#pragma unroll
  for (int dt = 0; dt < DT; ++dt) {
    o[dt] *= inv;
    u16x4 u;
#pragma unroll
    for (int j = 0; j < 4; ++j) u[j] = f2bf(o[dt][j]);
    *reinterpret_cast<u16x4*>(a.out + at + 16 * dt) = u;
    if (a.out32 != nullptr) *reinterpret_cast<f32x4*>(a.out32 + at + 16 * dt) = o[dt];
  }
  if (a.lse != nullptr && g == 0) a.lse[stat] = m + __builtin_amdgcn_logf(l);
}

// dK and dV: a workgroup has 64 keys of one query head, 16 a wave, and walks the queries from the diagonal on, 32 at a
// time.  A query head's part goes out in fp32; the heads of a group are added by train_kv_close_kernel: a workgroup per
// kv head would leave most CUs idle (13 x 8 blocks a sequence of 777 tokens) and atomics would make the sum's order,
// and so its bits, change from run to run.  Two workgroups to a CU: with the registers of three it spills (142 us where two
// take 81, both gradients of 700 tokens).
template <int D>
__global__ __launch_bounds__(256, 2) void train_attn_kv_kernel(TrainAttn a) {
  constexpr int KS = D / 32, DT = D / 16;
  typedef Tile<D, 32> QTile;
  __shared__ __attribute__((aligned(16))) unsigned char smem[2][2][QTile::BYTES];  // [buffer][Q | dO]
  __shared__ float stats[2][2][32];                                                // [buffer][lse | delta]
  const int lane = threadIdx.x & 63, w = threadIdx.x >> 6, g = lane >> 4;
  const int h = blockIdx.y, b = blockIdx.z, kvh = h / (a.nh / a.nkv);
  const int k0 = blockIdx.x * 64, key = k0 + 16 * w + (lane & 15);
  const int64_t row = (int64_t)b * a.T + min(key, a.T - 1);
  const bf16_t* qp = a.qkv + (int64_t)b * a.T * a.ld + h * D;
  const bf16_t* gp = a.dout + ((int64_t)b * a.T * a.nh + h) * D;
  const float *lp = a.lse + ((int64_t)b * a.nh + h) * a.T, *dp_ = a.delta + ((int64_t)b * a.nh + h) * a.T;
  const float c2 = a.scale * 1.4426950408889634f;

  u16x8 kf[KS], vf[KS];
#pragma unroll
  for (int s = 0; s < KS; ++s) {
    const bf16_t* p = a.qkv + row * a.ld + (a.nh + kvh) * D + 32 * s + 8 * g;
    kf[s] = key < a.T ? *reinterpret_cast<const u16x8*>(p) : (u16x8)(0);
    vf[s] = key < a.T ? *reinterpret_cast<const u16x8*>(p + a.nkv * D) : (u16x8)(0);
  }
  f32x4 dk[DT], dv[DT];
#pragma unroll
  for (int dt = 0; dt < DT; ++dt) dk[dt] = dv[dt] = (f32x4)(0.f);

  QTile qt, gt;
  float st_ = 0.f;
  auto fetch = [&](int r0) {
    qt.fetch(qp, a.ld, r0, a.T), gt.fetch(gp, (int64_t)a.nh * D, r0, a.T);
    if (threadIdx.x < 64) {  // a query past T: weight 0
      const int r = r0 + (threadIdx.x & 31);
      st_ = threadIdx.x < 32 ? (r < a.T ? lp[r] : INFINITY) : (r < a.T ? dp_[r] : 0.f);
    }
  };
  auto stash = [&](int buf, int r0) {
    qt.stash(smem[buf][0], a.T - r0), gt.stash(smem[buf][1], a.T - r0);
    if (threadIdx.x < 64) stats[buf][threadIdx.x >> 5][threadIdx.x & 31] = st_;
  };
  fetch(k0);
  stash(0, k0);
  __syncthreads();
  for (int r0 = k0, cur = 0; r0 < a.T; r0 += 32, cur ^= 1) {
    const bool more = r0 + 32 < a.T;
    if (more) fetch(r0 + 32);
    const unsigned char *Q = smem[cur][0], *G = smem[cur][1];
    if (r0 + 31 >= k0 + 16 * w) {
      f32x4 p[2], ds[2];
#pragma unroll
      for (int st = 0; st < 2; ++st) {
        f32x4 s = (f32x4)(0.f), dp = (f32x4)(0.f);
#pragma unroll
        for (int ks = 0; ks < KS; ++ks) {
          s = mfma16(row_frag<D>(Q, 16 * st, ks), kf[ks], s);
          dp = mfma16(row_frag<D>(G, 16 * st, ks), vf[ks], dp);
        }
        const f32x4 lse = *reinterpret_cast<const f32x4*>(&stats[cur][0][16 * st + 4 * g]);
        const f32x4 del = *reinterpret_cast<const f32x4*>(&stats[cur][1][16 * st + 4 * g]);
#pragma unroll
        for (int j = 0; j < 4; ++j) {
          const float e = __builtin_amdgcn_exp2f(__builtin_fmaf(s[j], c2, -lse[j]));
          p[st][j] = r0 + 16 * st + 4 * g + j >= key ? e : 0.f;
          ds[st][j] = p[st][j] == 0.f ? 0.f : p[st][j] * (dp[j] - del[j]) * a.scale;
        }
      }
      u16x8 pt[3], st[3];
      split8(p[0], p[1], pt);
      split8(ds[0], ds[1], st);
#pragma unroll
      for (int dt = 0; dt < DT; ++dt) {
        const u16x8 gc = col_frag<D>(G, 0, dt), qc = col_frag<D>(Q, 0, dt);
#pragma unroll
        for (int i = 2; i >= 0; --i) {
          dv[dt] = mfma16(gc, pt[i], dv[dt]);
          dk[dt] = mfma16(qc, st[i], dk[dt]);
        }
      }
    }
    if (more) stash(cur ^ 1, r0 + 32);
    __syncthreads();
  }
  if (key >= a.T) return;
  float* y = a.part + (row * a.nh + h) * D + 4 * g;
  const int64_t half = (int64_t)gridDim.z * a.T * a.nh * D;
#pragma unroll
  for (int dt = 0; dt < DT; ++dt) {
    *reinterpret_cast<f32x4*>(y + 16 * dt) = dk[dt];
    *reinterpret_cast<f32x4*>(y + half + 16 * dt) = dv[dt];
  }
}

// the query heads' parts of a kv head added, keys turned back, both into their columns of dqkv; a thread has 4 pairs
template <int D>
__global__ __launch_bounds__(256) void train_kv_close_kernel(TrainAttn a, int64_t rows) {
  constexpr int C = D / 8;
  const int64_t i = (int64_t)blockIdx.x * 256 + threadIdx.x, n = rows * a.nkv * C;
  if (i >= n) return;
  const int c = (int)(i % C) * 4, kvh = (int)(i / C % a.nkv), rep = a.nh / a.nkv;
  const int64_t row = i / C / a.nkv;
  f32x4 k0 = (f32x4)(0.f), k1 = k0, v0 = k0, v1 = k0;
  for (int r = 0; r < rep; ++r) {
    const float* p = a.part + (row * a.nh + kvh * rep + r) * D + c;
    const float* pv = p + rows * a.nh * D;
    k0 += *reinterpret_cast<const f32x4*>(p), k1 += *reinterpret_cast<const f32x4*>(p + D / 2);
    v0 += *reinterpret_cast<const f32x4*>(pv), v1 += *reinterpret_cast<const f32x4*>(pv + D / 2);
  }
  const float* cs = a.cs + (row % a.T) * D + c;
  u16x4 y[4];
#pragma unroll
  for (int j = 0; j < 4; ++j) {
    y[0][j] = f2bf(k0[j] * cs[j] + k1[j] * cs[D / 2 + j]);
    y[1][j] = f2bf(k1[j] * cs[j] - k0[j] * cs[D / 2 + j]);
    y[2][j] = f2bf(v0[j]), y[3][j] = f2bf(v1[j]);
  }
  bf16_t* o = a.dqkv + row * a.ld + (a.nh + kvh) * D + c;
  *reinterpret_cast<u16x4*>(o) = y[0], *reinterpret_cast<u16x4*>(o + D / 2) = y[1];
  o += a.nkv * D;
  *reinterpret_cast<u16x4*>(o) = y[2], *reinterpret_cast<u16x4*>(o + D / 2) = y[3];
}

// cos, then sin of the angles t inv[d] in 64 bits, rounded once: [T, 2 n].  The host's table took two copies that waited for
// all work on the device and left it idle until the host had caught up, for the request and again for its gradients: both
// together take 4.34 ms at 1554 tokens of four blocks with this kernel, 4.53 ms with the copies.
__global__ __launch_bounds__(256) void train_angles_kernel(const double* __restrict__ inv, float* __restrict__ out, int n,
                                                           int64_t total) {
  const int64_t i = (int64_t)blockIdx.x * 256 + threadIdx.x;
  if (i >= total) return;
  const int d = (int)(i % n);
  const int64_t t = i / n;
  double s, c;
  sincos((double)t * inv[d], &s, &c);
  out[t * 2 * n + d] = (float)c, out[t * 2 * n + n + d] = (float)s;
}

// q and k heads of the fused projection turned in place; a thread has 8 pairs (entry d and d + D / 2)
__global__ __launch_bounds__(256) void train_rope_kernel(bf16_t* x, int64_t ld, const float* __restrict__ cs, int T, int heads,
                                                         int D, int64_t n) {
  const int C = D / 16;
  const int64_t i = (int64_t)blockIdx.x * 256 + threadIdx.x;
  if (i >= n) return;
  const int c = (int)(i % C) * 8, h = (int)(i / C % heads);
  const int64_t row = i / C / heads;
  bf16_t* p = x + row * ld + (int64_t)h * D + c;
  const float* t = cs + (row % T) * D + c;
  u16x8 u = *reinterpret_cast<u16x8*>(p), v = *reinterpret_cast<u16x8*>(p + D / 2);
#pragma unroll
  for (int j = 0; j < 8; ++j) {
    const float x0 = bf2f(u[j]), x1 = bf2f(v[j]), co = t[j], si = t[D / 2 + j];
    u[j] = f2bf(x0 * co - x1 * si), v[j] = f2bf(x1 * co + x0 * si);
  }
  *reinterpret_cast<u16x8*>(p) = u, *reinterpret_cast<u16x8*>(p + D / 2) = v;
}

// Norm of a row of the stream, a workgroup a row, the row in registers (one read).  Forward: sum = x + y (y may be
// absent) + the block's deep prompt in a sequence's first P rows, each sum rounded, out = sum / rms(sum) w.  (At
// 1554 rows of 4096 8.5 us without a prompt, 8.7 with one; the prompt in launches of its own 16.5.)  Backward: out = res + d sum of (norm's gradient ``y``): rms and the row's dot product
// are made again from ``x``, which is read anyway.
template <int NC, bool GRAD>
__global__ __launch_bounds__(256) void train_norm_kernel(const bf16_t* __restrict__ x, const bf16_t* __restrict__ y,
                                                         const bf16_t* __restrict__ w, bf16_t* sum, bf16_t* out, int H,
                                                         float eps, const bf16_t* __restrict__ deep, int P, int T,
                                                         int64_t apart) {
  __shared__ float red[16], red2[16];
  const int64_t at = (int64_t)blockIdx.x * H;
  const int nch = H >> 3;
  const int b = GRAD || deep == nullptr ? 0 : blockIdx.x / T, t0 = GRAD || deep == nullptr ? 0 : blockIdx.x - b * T;
  const bool prompted = !GRAD && deep != nullptr && t0 < P;
  const bf16_t* dp = deep + b * apart + (int64_t)t0 * H;
  u16x8 xv[NC], yv[NC], wv[NC], rv[NC];
#pragma unroll
  for (int k = 0; k < NC; ++k) {
    const int c = 8 * min((int)threadIdx.x + 256 * k, nch - 1);
    xv[k] = *reinterpret_cast<const u16x8*>(x + at + c);
    if (y != nullptr) yv[k] = *reinterpret_cast<const u16x8*>(y + at + c);
    wv[k] = *reinterpret_cast<const u16x8*>(w + c);
    if (GRAD) rv[k] = *reinterpret_cast<const u16x8*>(sum + at + c);
    else if (prompted) rv[k] = *reinterpret_cast<const u16x8*>(dp + c);
  }
  float ss = 0.f, dot = 0.f;
#pragma unroll
  for (int k = 0; k < NC; ++k) {
    const int c = threadIdx.x + 256 * k;
    if (c >= nch) continue;
    if (!GRAD && sum != nullptr) {
      if (y != nullptr)
#pragma unroll
        for (int j = 0; j < 8; ++j) xv[k][j] = f2bf(bf2f(xv[k][j]) + bf2f(yv[k][j]));
      if (prompted)
#pragma unroll
        for (int j = 0; j < 8; ++j) xv[k][j] = f2bf(bf2f(xv[k][j]) + bf2f(rv[k][j]));
      *reinterpret_cast<u16x8*>(sum + at + 8 * c) = xv[k];
    }
#pragma unroll
    for (int j = 0; j < 8; ++j) {
      const float f = bf2f(xv[k][j]);
      ss += f * f;
      if (GRAD) dot += f * bf2f(wv[k][j]) * bf2f(yv[k][j]);
    }
  }
  const float r = rsqrtf(block_sum(ss, red) / (float)H + eps);
  const float t = GRAD ? block_sum(dot, red2) * r * r / (float)H : 0.f;
#pragma unroll
  for (int k = 0; k < NC; ++k) {
    const int c = threadIdx.x + 256 * k;
    if (c >= nch) continue;
    u16x8 o;
#pragma unroll
    for (int j = 0; j < 8; ++j) {
      const float f = bf2f(xv[k][j]), g = bf2f(wv[k][j]);
      o[j] = GRAD ? f2bf(bf2f(rv[k][j]) + r * (g * bf2f(yv[k][j]) - f * t)) : f2bf(f * r * g);
    }
    *reinterpret_cast<u16x8*>(out + at + 8 * c) = o;
  }
}

// gate / up rows in alternating blocks of 16 -> their gradients in the same places, from the activation's gradient
__global__ __launch_bounds__(256) void train_glu_grad_kernel(bf16_t* gu, const bf16_t* __restrict__ da, int64_t n, int F) {
  for (int64_t i = (int64_t)blockIdx.x * 256 + threadIdx.x; i < n; i += (int64_t)gridDim.x * 256) {
    const int64_t row = i / (F / 8);
    const int c = (int)(i % (F / 8)) * 8;
    bf16_t* p = gu + row * 2 * F + (c >> 4) * 32 + (c & 15);
    u16x8 gv = *reinterpret_cast<u16x8*>(p), uv = *reinterpret_cast<u16x8*>(p + 16);
    const u16x8 dv = *reinterpret_cast<const u16x8*>(da + row * F + c);
#pragma unroll
    for (int j = 0; j < 8; ++j) {
      const float g = bf2f(gv[j]), u = bf2f(uv[j]), d = bf2f(dv[j]);
      const float s = 1.f / (1.f + expf(-g));
      gv[j] = f2bf(d * u * s * (1.f + g * (1.f - s)));
      uv[j] = f2bf(d * g * s);
    }
    *reinterpret_cast<u16x8*>(p) = gv, *reinterpret_cast<u16x8*>(p + 16) = uv;
  }
}

}  // namespace mp

extern "C" int mp_train_attn(const void* qkv, int64_t ld, int B, int T, int nh, int nkv, int D, float scale, void* out,
                             float* out32, float* lse, hipStream_t stream) {
  (void)hipGetLastError();
  using namespace mp;
  TrainAttn a{};
  a.qkv = (const bf16_t*)qkv, a.ld = ld, a.T = T, a.nh = nh, a.nkv = nkv, a.scale = scale;
  a.out = (bf16_t*)out, a.out32 = out32, a.lse = lse;
  const dim3 grid((T + 63) / 64, nh, B);
  if (D == 128) hipLaunchKernelGGL((train_attn_q_kernel<128, false>), grid, dim3(256), 0, stream, a);
  else if (D == 64) hipLaunchKernelGGL((train_attn_q_kernel<64, false>), grid, dim3(256), 0, stream, a);
  else return -1;
  return (int)hipGetLastError();
}

extern "C" int mp_train_attn_grad(const void* qkv, int64_t ld, int B, int T, int nh, int nkv, int D, float scale,
                                  const float* out32, const float* lse, const void* dout, float* delta, const float* cs,
                                  float* part, void* dqkv, hipStream_t stream) {
  (void)hipGetLastError();
  using namespace mp;
  TrainAttn a{};
  a.qkv = (const bf16_t*)qkv, a.ld = ld, a.T = T, a.nh = nh, a.nkv = nkv, a.scale = scale;
  a.out32 = const_cast<float*>(out32), a.lse = const_cast<float*>(lse), a.dout = (const bf16_t*)dout, a.delta = delta;
  a.cs = cs, a.part = part, a.dqkv = (bf16_t*)dqkv;
  const dim3 grid((T + 63) / 64, nh, B);
  const int64_t rows = (int64_t)B * T;
  const dim3 close((unsigned)((rows * nkv * (D / 8) + 255) / 256));
  if (D == 128) {
    hipLaunchKernelGGL((train_attn_q_kernel<128, true>), grid, dim3(256), 0, stream, a);
    hipLaunchKernelGGL((train_attn_kv_kernel<128>), grid, dim3(256), 0, stream, a);
    hipLaunchKernelGGL((train_kv_close_kernel<128>), close, dim3(256), 0, stream, a, rows);
  } else if (D == 64) {
    hipLaunchKernelGGL((train_attn_q_kernel<64, true>), grid, dim3(256), 0, stream, a);
    hipLaunchKernelGGL((train_attn_kv_kernel<64>), grid, dim3(256), 0, stream, a);
    hipLaunchKernelGGL((train_kv_close_kernel<64>), close, dim3(256), 0, stream, a, rows);
  } else {
    return -1;
  }
  return (int)hipGetLastError();
}

extern "C" int mp_train_angles(const double* inv, float* out, int n, int64_t T, hipStream_t stream) {
  (void)hipGetLastError();
  using namespace mp;
  hipLaunchKernelGGL(train_angles_kernel, dim3((unsigned)((T * n + 255) / 256)), dim3(256), 0, stream, inv, out, n, T * n);
  return (int)hipGetLastError();
}

extern "C" int mp_train_rope(void* x, int64_t ld, const float* cs, int64_t rows, int T, int heads, int D,
                             hipStream_t stream) {
  (void)hipGetLastError();
  using namespace mp;
  const int64_t n = rows * heads * (D / 16);
  hipLaunchKernelGGL(train_rope_kernel, dim3((unsigned)((n + 255) / 256)), dim3(256), 0, stream, (bf16_t*)x, ld, cs, T,
                     heads, D, n);
  return (int)hipGetLastError();
}

extern "C" int mp_train_norm(const void* x, const void* y, const void* w, void* sum, void* out, int64_t rows, int H, float eps,
                             int grad, const void* deep, int P, int T, int64_t apart, hipStream_t stream) {
  (void)hipGetLastError();
  using namespace mp;
  if (H % 8 || H > 16384 || H < 8 || (deep != nullptr && (grad || sum == nullptr || T < 1))) return -1;
#define MP_TN(NC_, G_)                                                                                              \
  hipLaunchKernelGGL((train_norm_kernel<NC_, G_>), dim3((unsigned)rows), dim3(256), 0, stream, (const bf16_t*)x,        \
                     (const bf16_t*)y, (const bf16_t*)w, (bf16_t*)sum, (bf16_t*)out, H, eps, (const bf16_t*)deep, P, T, apart)
#define MP_TN2(NC_) \
  if (grad) MP_TN(NC_, true); else MP_TN(NC_, false)
  if (H <= 4096) { MP_TN2(2); } else if (H <= 8192) { MP_TN2(4); } else { MP_TN2(8); }
#undef MP_TN2
#undef MP_TN
  return (int)hipGetLastError();
}

extern "C" int mp_train_glu_grad(void* gu, const void* da, int64_t rows, int F, hipStream_t stream) {
  (void)hipGetLastError();
  using namespace mp;
  if (F % 16) return -1;
  const int64_t n = rows * (F / 8), blocks = (n + 255) / 256;
  hipLaunchKernelGGL(train_glu_grad_kernel, dim3((unsigned)(blocks < 8192 ? blocks : 8192)), dim3(256), 0, stream, (bf16_t*)gu,
                     (const bf16_t*)da, n, F);
  return (int)hipGetLastError();
}
