// Causal prefill attention over the paged KV cache on gfx950, FA2-style with 32x32x16 MFMA
// (survey K7 "attn_prefill: causal, MFMA 32x32x16 bf16 QK^T and PV, LDS tiling").
//
// The reference computes prefill attention as matmul -> fp32 softmax -> matmul over the whole
// [heads, T, P+T] score tensor, and without a causal mask (petals/llama/block.py:134-141,
// SURVEY §7.2).  Here one workgroup of NW waves owns 32 x NW query ROWS of one kv head and
// one sequence (row = token-major x the GQA group's HB heads: row r is token tok0 + r / HB,
// head hbase + r % HB), and streams the causal context in 64-token steps:
//
//   * K and V tiles [64 tok][128 d] are staged once per step for all NW waves through two LDS slots
//     each (256-B rows, 16-B chunks XOR-swizzled by the row so both the row reads of K and the
//     transposed reads of V are bank-conflict-free).  Loads go straight to LDS, a step ahead, and
//     the page of the step behind them is looked up a step before that (one barrier per step).
//   * A step takes the softmax and O of its scores and makes the NEXT step's scores, so that the
//     exponentials have the MFMAs of K . Q^T between them and the next maximum those of V^T . P^T.
//     Bound by VALU and MFMA issue, which add up: a step of 32 rows is 1024 cycles of MFMA and about 1250
//     of VALU (512 of them exponentials), two waves a SIMD.  7995 tokens of 32 / 8 heads: 686 us with the
//     phases one after the other and tiles by way of registers, 670 with loads straight to LDS and the phases mixed,
//     641 with pages looked up ahead and the maximum exchanged without LDS.  (Measured and left: a
//     barrier for every second step 660; wave priorities 645; spills in the loop 1142, as their waits cover
//     the tiles' loads.)
//   * S^T = K . Q^T per wave: 2 x (D/16) v_mfma_f32_32x32x16_bf16 (A = K rows from LDS with
//     ds_read_b128, B = Q^T fragments held in registers for the whole kernel).  The
//     accumulator's COLUMN is the query row, so each lane owns one row and 16 of its
//     scores per 32-token subtile: the online softmax (exp2 domain, causal + context mask)
//     is lane-local plus one xor-32 shuffle for the row maximum.
//   * O^T += V^T . P^T: the exponentiated scores are the B operand straight from the S^T
//     accumulators (no LDS round trip, permuted k order), and V^T comes from the row-major
//     V tile through ds_read_b64_tr_b16, the hardware transpose read: 16 MFMAs per step.
//     O^T's column is the query row too, so the softmax rescale is a per-lane scalar.
//   * causal skipping: a wave stops computing at its own rows' context (the diagonal steps
//     of the earlier waves), workgroups are launched longest-context first.
// Splits of the context (NP > 1) write (m, l, O) partials reduced by launch_attn_reduce (attention.hip).
#include "common.h"

namespace mp {

typedef __attribute__((ext_vector_type(8))) __bf16 bf16x8_fa;
typedef short s16x4_fa __attribute__((ext_vector_type(4)));
typedef __attribute__((ext_vector_type(4))) unsigned u32x4_fa;

__device__ __forceinline__ f32x16 mfma32x16(const u16x8& a, const u16x8& b, const f32x16& c) {
  return __builtin_amdgcn_mfma_f32_32x32x16_bf16(__builtin_bit_cast(bf16x8_fa, a), __builtin_bit_cast(bf16x8_fa, b), c,
                                                 0, 0, 0);
}

// LDS image of a [rows][128 bf16] tile (16-B chunks ch = 0..15): 8-row x 32-column subtiles of
// 512 B, the chunk's 4 low bits XOR-swizzled by the row (guide T10 image (a)).  Row reads of
// the 32x32x16 A operand (ds_read_b128) and transposed 4-row reads of V (ds_read_b64_tr_b16) are
// both bank-conflict-free on it, and within a lane every read of a step differs from one of two
// base addresses by an immediate offset (no per-read address arithmetic).
__device__ __forceinline__ int fa_off(int row, int ch) {
  return 2048 * (row >> 3) + 512 * (ch >> 2) + 64 * (row & 7) + 16 * ((ch & 3) ^ ((row >> 2) & 3));
}

__device__ __forceinline__ u16x4 tr16(const unsigned char* p) {
  const s16x4_fa v = __builtin_amdgcn_ds_read_tr16_b64_v4i16(
      (__attribute__((address_space(3))) s16x4_fa*)(const_cast<unsigned char*>(p)));
  return __builtin_bit_cast(u16x4, v);
}

// two fp32 -> packed bf16 pair (v_cvt_pk_bf16_f32)
typedef __attribute__((ext_vector_type(2))) float f32x2_fa;
typedef __attribute__((ext_vector_type(2))) __bf16 bf16x2_fa;
__device__ __forceinline__ unsigned pk_bf16(float a, float b) {
  const bf16x2_fa v = __builtin_convertvector((f32x2_fa){a, b}, bf16x2_fa);
  return __builtin_bit_cast(unsigned, v);
}

constexpr float FA_RESCALE_THR = 8.f;  // log2 units: P may reach 2^8 before O / l are rescaled (T13)

template <int HB, int NW>
__global__ __launch_bounds__(NW * 64) void attn_fa_kernel(
    const bf16_t* __restrict__ q, int64_t q_stride, const bf16_t* __restrict__ kc, const bf16_t* __restrict__ vc,
    const int32_t* __restrict__ block_tables, int bt_stride, const int32_t* __restrict__ q_seq,
    const int32_t* __restrict__ q_ctx, const int32_t* __restrict__ fb_tok0, const int32_t* __restrict__ fb_ntok,
    int NBF, bf16_t* __restrict__ out, int64_t out_stride, float* __restrict__ part_o, float* __restrict__ part_ml,
    int nkv, int nh, int page_log2, int PS, int NP, float scale_log2, int pair) {
  constexpr int D = 128;
  constexpr int STEP = 64;
  constexpr int TILE = STEP * D * 2;            // bytes of one K or V tile (16 KiB)
  constexpr int NT = NW * 64;
  constexpr int CPT = (STEP * D / 8) / NT;      // 16-B chunks per thread per tile
  static_assert((STEP * D / 8) % NT == 0, "tile chunks split evenly over the threads");
  __shared__ __attribute__((aligned(16))) unsigned char smem[2 * 2 * TILE];  // [buf][K | V]

  const int tid = threadIdx.x, lane = tid & 63;
  const int w = __builtin_amdgcn_readfirstlane(tid >> 6);
  // XCD-aware order: the query blocks of one head sit on one XCD (its K / V stay in that L2),
  // longest causal context first inside a head
  // pair (causal balance for small grids): workgroup j of a head runs query block NBF-1-j, then
  // block j - every workgroup streams the same total context (a long block + its short mirror),
  // instead of the longest blocks setting the kernel time on a grid of ~2 workgroups per CU
  const int G = gridDim.x, NHG = nh / HB;
  const int NBP = pair ? (NBF + 1) / 2 : NBF;  // workgroups per head
  int lin = blockIdx.x;
  if ((G & 7) == 0) lin = (lin & 7) * (G >> 3) + (lin >> 3);
  const int hg = lin / NBP;
  const int jb = lin - hg * NBP;
  const int p = blockIdx.y;
  const int hbase = hg * HB;
  const int g = hbase / (nh / nkv);
  const int npass = pair && (NBF - 1 - jb) != jb ? 2 : 1;
  (void)NHG;
  for (int pass = 0; pass < npass; ++pass) {
  const int bx = pair ? (pass == 0 ? NBF - 1 - jb : jb) : NBF - 1 - jb;
  const int tok0 = fb_tok0[bx], ntok = fb_ntok[bx];
  const int32_t* bt = block_tables + (int64_t)q_seq[tok0] * bt_stride;
  const int page_size = 1 << page_log2;
  const int64_t page_stride = (int64_t)nkv * page_size * D;
  const int64_t head_off = (int64_t)g * page_size * D;

  // contexts are non-decreasing along a sequence's tokens: the last token's is the largest
  const int grp_ctx = q_ctx[tok0 + ntok - 1];
  const int wt_first = (32 * w) / HB, wt_last = min((32 * w + 31) / HB, ntok - 1);
  const bool wave_rows = wt_first < ntok;
  const int wave_ctx = wave_rows ? q_ctx[tok0 + wt_last] : 0;
  const int start = p * PS, end = min(start + PS, grp_ctx);
  const int wave_lim0 = wave_rows ? min(q_ctx[tok0 + wt_first], end) : 0;  // smallest limit of its rows

  const int r = lane & 31, hh = lane >> 5;
  const int my_row = 32 * w + r;
  const int my_t = my_row / HB, my_h = hbase + my_row % HB;
  const bool row_ok = my_t < ntok;
  const int my_ctx = row_ok ? q_ctx[tok0 + my_t] : 0;
  const int lim = min(my_ctx, end);

  u16x8 qf[D / 16];
#pragma unroll
  for (int s = 0; s < D / 16; ++s) {
    qf[s] = row_ok ? *reinterpret_cast<const u16x8*>(q + (int64_t)(tok0 + my_t) * q_stride + (int64_t)my_h * D +
                                                     16 * s + 8 * hh)
                   : (u16x8)(0);
  }
  f32x16 o[D / 32];
#pragma unroll
  for (int dt = 0; dt < D / 32; ++dt) o[dt] = (f32x16)(0.f);
  float m = -INFINITY, l = 0.f;  // running max (log2 units, scale applied) and sum of row r

  // A tile goes straight to LDS, two KiB a wave: 1-KiB blocks of 8 rows x 64 columns, whose lanes' rows and chunks are the
  // image's.  (Loads the compiler knows of make every transposed read wait for them; these are waited for by hand.)
  const int fr = (lane >> 2) & 7;  // row of a block
  uint32_t off[CPT];
#pragma unroll
  for (int j = 0; j < CPT; ++j) {
    const int blk = CPT * w + j, row = 8 * (blk >> 1) + fr, ch = 8 * (blk & 1) + 4 * (lane >> 5) + ((lane & 3) ^ ((row >> 2) & 3));
    off[j] = (uint32_t)(row * D + ch * 8) * 2;
  }
  auto page = [&](int s0) { return s0 < end ? bt[s0 >> page_log2] : 0; };
  auto fetch = [&](const bf16_t* from, int s0, int64_t pg, int tile) {
    const uint64_t at = (uint64_t)(uintptr_t)(from + pg * page_stride + head_off + (int64_t)(s0 & (page_size - 1)) * D);
    const u32x4_fa words = {(uint32_t)__builtin_amdgcn_readfirstlane((int)at),
                            (uint32_t)__builtin_amdgcn_readfirstlane((int)(at >> 32)) & 0xffff, (uint32_t)TILE, 0x00020000u};
#pragma unroll
    for (int j = 0; j < CPT; ++j) {
      const uint32_t to = (uint32_t)(uintptr_t)(__attribute__((address_space(3))) void*)(smem + tile * TILE + (CPT * w + j) * 1024);
      asm volatile("s_mov_b32 m0, %0\n\ts_nop 4\n\tbuffer_load_dwordx4 %1, %2, 0 offen lds" ::"s"(to), "v"(off[j]), "s"(words)
                   : "memory");
    }
  };
  // the wave's loads have landed; rows of V past the context are cleared (stale cache bytes never meet a p = 0; stale scores
  // are masked)
  auto landed = [&](int s0, int tile) {
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
    if (s0 + STEP > end)
#pragma unroll
      for (int j = 0; j < CPT; ++j)
        if (s0 + 8 * ((CPT * w + j) >> 1) + fr >= end)
          *reinterpret_cast<u16x8*>(smem + tile * TILE + (CPT * w + j) * 1024 + lane * 16) = (u16x8)(0);
  };

  // per-lane LDS bases (every read of a step is one of them + an immediate):
  //   K row read (sub, s): row 32 sub + r, chunk 2 s + hh -> kbase[s & 1] + 8192 sub + 512 (s >> 1)
  //   V transposed read (sub, s2, dt, hi): this lane feeds row q of the 4-row block at
  //   32 sub + 16 s2 + 8 hi + 4 hh, chunk 4 dt + 2 (grp & 1) + (tp >> 1), + 8 (tp & 1) bytes
  //   -> vbase[hi] + 8192 sub + 4096 s2 + 512 dt
  const int grp = lane >> 4, gi = lane & 15, tq = gi >> 2, tp = gi & 3;
  const int kbase0 = fa_off(r, hh), kbase1 = fa_off(r, 2 + hh);
  const int trc = 2 * (grp & 1) + (tp >> 1);
  const int vbase0 = fa_off(4 * hh + tq, trc) + 8 * (tp & 1);
  const int vbase1 = fa_off(8 + 4 * hh + tq, trc) + 8 * (tp & 1);

  // A step takes the softmax of its scores and its part of O, and makes the scores of the next one, S^T = K . Q^T (two
  // accumulation chains, halves of d, summed afterwards).  In groups of one MFMA, the VALU work of two scores and the LDS reads
  // of the MFMA four on, which the fences keep as written: first the exponentials beside the next scores, then the next
  // maximum beside O.
  f32x16 st[2];
  float lm;  // largest of st on this lane
  u16x8 ka[4];
  auto key = [&](const unsigned char* kt, int sub, int s) {
    return *reinterpret_cast<const u16x8*>(kt + ((s & 1) ? kbase1 : kbase0) + 8192 * sub + 512 * (s >> 1));
  };
  auto value = [&](const unsigned char* vt, int i) {  // i: 8 sub + 4 s2 + dt
    const u16x4 lo = tr16(vt + vbase0 + 4096 * (i >> 2) + 512 * (i & 3));
    const u16x4 hi = tr16(vt + vbase1 + 4096 * (i >> 2) + 512 * (i & 3));
    return (u16x8){lo[0], lo[1], lo[2], lo[3], hi[0], hi[1], hi[2], hi[3]};
  };
  auto across = [](float x) {  // the larger of a row's two lanes
    const auto y = __builtin_amdgcn_permlane32_swap(__float_as_uint(x), __float_as_uint(x), false, false);
    return fmaxf(__uint_as_float(y[0]), __uint_as_float(y[1]));
  };
  auto largest = [&](int sub) {
#pragma unroll
    for (int j = 0; j < 16; ++j) lm = fmaxf(lm, st[sub][j]);
  };
  auto step = [&](int b0, const unsigned char* kt, const unsigned char* vt) {
    // ---- online softmax of row r over this lane's 32 tokens (raw scores; the scale is
    //      folded into the exponent's FMA) ----
#pragma unroll
    for (int s = 0; s < 4; ++s) ka[s] = key(kt, 0, s);
    if (b0 + STEP > wave_lim0) {  // diagonal / last step: causal and context mask
#pragma unroll
      for (int sub = 0; sub < 2; ++sub)
#pragma unroll
        for (int j = 0; j < 16; ++j) {
          const int tk = b0 + 32 * sub + 4 * hh + (j & 3) + 8 * (j >> 2);
          st[sub][j] = tk < lim ? st[sub][j] : -INFINITY;
        }
      lm = -INFINITY;
      largest(0), largest(1);
    }
    lm = across(lm) * scale_log2;
    // rescale O and l only when some row's maximum grew by more than the threshold
    if (!__all(lm <= m + FA_RESCALE_THR)) {
      const float m_new = fmaxf(m, lm);
      const float alpha = m_new == -INFINITY ? 1.f : __builtin_amdgcn_exp2f(m - m_new);
      l *= alpha;
#pragma unroll
      for (int dt = 0; dt < D / 32; ++dt) o[dt] *= alpha;
      m = m_new;
    }
    const float mu = m == -INFINITY ? 0.f : m;  // fully masked row so far: every p is 0
    float ps = 0.f;
    unsigned pk[2][8];
    auto weigh = [&](int sub, int i) {
      const float p0 = __builtin_amdgcn_exp2f(__builtin_fmaf(st[sub][2 * i], scale_log2, -mu));
      const float p1 = __builtin_amdgcn_exp2f(__builtin_fmaf(st[sub][2 * i + 1], scale_log2, -mu));
      ps += p0 + p1;
      pk[sub][i] = pk_bf16(p0, p1);
    };
    auto pf = [&](int sub, int s2) {
      return __builtin_bit_cast(u16x8, (u32x4_fa){pk[sub][4 * s2], pk[sub][4 * s2 + 1], pk[sub][4 * s2 + 2], pk[sub][4 * s2 + 3]});
    };
    f32x16 sa[2], sb[2];
    sa[0] = sa[1] = sb[0] = sb[1] = (f32x16)(0.f);
    u16x8 va[4];
    __builtin_amdgcn_sched_barrier(0);
#pragma unroll
    for (int s = 0; s < 8; ++s) {
      sa[s >> 2] = mfma32x16(ka[s & 3], qf[s], sa[s >> 2]);
      ka[s & 3] = s < 4 ? key(kt, 0, s + 4) : key(kt, 1, s - 4);
      weigh(0, s);
      __builtin_amdgcn_sched_barrier(0);
    }
#pragma unroll
    for (int s = 0; s < 8; ++s) {
      sb[s >> 2] = mfma32x16(ka[s & 3], qf[s], sb[s >> 2]);
      if (s < 4) ka[s] = key(kt, 1, s + 4);
      else va[s - 4] = value(vt, s - 4);
      weigh(1, s);
      if (s == 3) st[0] = sa[0] + sa[1];
      __builtin_amdgcn_sched_barrier(0);
    }
    // ---- O^T += V^T . P^T: A = V^T by transposed LDS reads, B = P from registers ----
    lm = -INFINITY;
#pragma unroll
    for (int s = 0; s < 8; ++s) {
      o[s & 3] = mfma32x16(va[s & 3], pf(0, s >> 2), o[s & 3]);
      va[s & 3] = value(vt, 4 + s);
      if (s == 2) largest(0);
      if (s == 5) st[1] = sb[0] + sb[1];
      __builtin_amdgcn_sched_barrier(0);
    }
#pragma unroll
    for (int s = 0; s < 8; ++s) {
      o[s & 3] = mfma32x16(va[s & 3], pf(1, s >> 2), o[s & 3]);
      if (s < 4) va[s] = value(vt, 12 + s);
      if (s == 2) largest(1);
      __builtin_amdgcn_sched_barrier(0);
    }
    l += ps;
  };

  // tiles: K of even and odd steps, V of even and odd steps.  A step reads its V and the next one's K.
  int pg0 = page(start), pg1 = page(start + STEP), pg2 = page(start + 2 * STEP);  // (a step's V is in the page of its K)
  if (start < end) {
    fetch(kc, start, pg0, 0);
    fetch(vc, start, pg0, 2);
    if (start + STEP < end) fetch(kc, start + STEP, pg1, 1);
    landed(start, 2);
  }
  __syncthreads();
  if (start < wave_ctx) {
#pragma unroll
    for (int sub = 0; sub < 2; ++sub) {
      f32x16 sa[2];
      sa[0] = sa[1] = (f32x16)(0.f);
#pragma unroll
      for (int s = 0; s < 8; ++s) sa[s >> 2] = mfma32x16(key(smem, sub, s), qf[s], sa[s >> 2]);
      st[sub] = sa[0] + sa[1];
    }
    lm = -INFINITY;
    largest(0), largest(1);
  }
  __syncthreads();
  int it = 0;
  for (int b0 = start; b0 < end; b0 += STEP, ++it) {
    const int cur = it & 1;
    const bool more = b0 + STEP < end;
    if (b0 + 2 * STEP < end) fetch(kc, b0 + 2 * STEP, pg2, cur);
    if (more) fetch(vc, b0 + STEP, pg1, 2 + (cur ^ 1));
    pg1 = pg2, pg2 = page(b0 + 3 * STEP);
    const unsigned char *kt = smem + (cur ^ 1) * TILE, *vt = smem + (2 + cur) * TILE;
    if (b0 < wave_ctx) step(b0, kt, vt);
    if (more) landed(b0 + STEP, 2 + (cur ^ 1));
    __syncthreads();
  }
  // ---- epilogue: lane owns row r; O^T accumulator register j of d-tile dt holds
  //      d = 32 dt + 8 (j >> 2) + 4 hh + (j & 3) ----
  l += __shfl_xor(l, 32, 64);
  if (!row_ok) continue;  // (every step above ended in a barrier: the LDS tiles are free)
  const int tok = tok0 + my_t;
  if (NP == 1) {
    const float inv = l > 0.f ? 1.f / l : 0.f;
    bf16_t* orow = out + (int64_t)tok * out_stride + (int64_t)my_h * D;
#pragma unroll
    for (int dt = 0; dt < D / 32; ++dt)
#pragma unroll
      for (int gq = 0; gq < 4; ++gq) {
        u16x4 v;
#pragma unroll
        for (int e = 0; e < 4; ++e) v[e] = f2bf(o[dt][4 * gq + e] * inv);
        *reinterpret_cast<u16x4*>(orow + 32 * dt + 8 * gq + 4 * hh) = v;
      }
  } else {
    const int64_t hp = ((int64_t)tok * nh + my_h) * NP + p;
    float* po = part_o + hp * D;
#pragma unroll
    for (int dt = 0; dt < D / 32; ++dt)
#pragma unroll
      for (int gq = 0; gq < 4; ++gq) {
        f32x4 v;
#pragma unroll
        for (int e = 0; e < 4; ++e) v[e] = o[dt][4 * gq + e];
        *reinterpret_cast<f32x4*>(po + 32 * dt + 8 * gq + 4 * hh) = v;
      }
    if (hh == 0) {
      part_ml[hp * 2] = m;
      part_ml[hp * 2 + 1] = l;
    }
  }
  }  // pass
}

void launch_attn_reduce(const float* part_o, const float* part_ml, void* out, int rows, int NP, int D, int nh, int packed_mt,
                        hipStream_t stream);  // attention.hip

}  // namespace mp

// Prefill blocks: fb_tok0[i] / fb_ntok[i] = first flat token / token count of block i (<= 32 x NW
// / heads_per_block consecutive tokens of ONE sequence, ops.fa_blocks).  D = 128, page_size a
// multiple of 64, heads_per_block = nh / nkv in {1, 2, 4, 8}; row-major output [T, nh * D].
extern "C" int mp_attention_fa(const void* q, int64_t q_stride, const void* kc, const void* vc, const int32_t* bt,
                               int bt_stride, const int32_t* q_seq, const int32_t* q_ctx, const int32_t* fb_tok0,
                               const int32_t* fb_ntok, int NBF, void* out, float* workspace, int T, int nh, int nkv,
                               int D, int page_size, int PS, int NP, float scale, int nw, int pair,
                               hipStream_t stream) {
  (void)hipGetLastError();  // an earlier non-mpamd HIP call's stale error is not this launch's
  using namespace mp;
  if (NBF == 0 || T == 0) return 0;
  if (D != 128 || nh % nkv != 0 || PS % 64 != 0 || NP < 1 || page_size % 64 != 0) return -1;
  int page_log2 = 0;
  while ((1 << page_log2) < page_size) ++page_log2;
  if ((1 << page_log2) != page_size) return -2;
  const int hb = nh / nkv;
  pair = pair ? 1 : 0;
  const int nbp = pair ? (NBF + 1) / 2 : NBF;
  const float scale_log2 = scale * 1.4426950408889634f;
  float* ws_o = workspace;
  float* ws_ml = workspace + (int64_t)T * nh * NP * D;
#define MP_FA(HB_, NW_)                                                                                         \
  hipLaunchKernelGGL((attn_fa_kernel<HB_, NW_>), dim3(nbp * (nh / HB_), NP), dim3(NW_ * 64), 0, stream,           \
                     (const bf16_t*)q, q_stride, (const bf16_t*)kc, (const bf16_t*)vc, bt, bt_stride, q_seq, q_ctx, \
                     fb_tok0, fb_ntok, NBF, (bf16_t*)out, (int64_t)nh * D, ws_o, ws_ml, nkv, nh, page_log2, PS, NP,  \
                     scale_log2, pair)
#define MP_FA_NW(HB_) \
  if (nw == 8) MP_FA(HB_, 8); else MP_FA(HB_, 4);
  switch (hb) {
    case 1: MP_FA_NW(1); break;
    case 2: MP_FA_NW(2); break;
    case 4: MP_FA_NW(4); break;
    case 8: MP_FA_NW(8); break;
    default: return -3;
  }
#undef MP_FA_NW
#undef MP_FA
  if (NP > 1)
    launch_attn_reduce(ws_o, ws_ml, out, T * nh, NP, D, nh, 0, stream);
  return (int)hipGetLastError();
}
