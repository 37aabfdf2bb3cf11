// MFMA flash attention over the paged KV cache for gfx950 (survey K7: "attn_prefill ...
// MFMA QK^T and PV, LDS tiles"; also GQA decode).
//
// A workgroup (4 waves) owns a block of 16 query ROWS of one kv head: row r is query token
// tok0 + r / HB of one sequence and query head hbase + r % HB (HB = heads of the GQA group
// in the block, TB = 16 / HB tokens).  So MHA prefill processes 16 consecutive tokens per
// block (K/V read once per 16 queries instead of once per query), and GQA decode puts the
// whole group (4 or 8 heads of one token) into the MFMA M dimension.
//
// Per wave and per 32-token step of the context (waves interleave steps):
//   S^T[tok][row] = K[tok, :] . Q[row, :]          2 x (D/32) v_mfma_f32_16x16x32_bf16
//       A = K rows straight from the cache page (lane (q, c): 16 B of token c at d = 8q),
//       B = Q^T fragments held in registers for the whole kernel;
//   online softmax per row in the exp2 domain (row = lane & 15; the 4 lanes of a row
//       combine with two xor shuffles), causal + context masking per row;
//   O[row][d] += P[row][tok] . V[tok][d]            D/16 MFMAs
//       A = P straight from the S^T accumulators: lane (q, c) holds row c at tokens
//       {4q..4q+3, 16+4q..16+4q+3}, used as the MFMA k order,
//       B = V^T: the wave copies its 32 rows of V, whole rows a load, into an LDS tile of its own
//       (the tile never straddles a 64-token page; tokens past the context are zeroed so stale
//       cache bytes never meet a p = 0) and reads 4 tokens x 16 columns transposed at a time
//       (ds_read_b64_tr_b16), two per fragment, in the same permuted k order.
// The 4 waves' (m, l, O) are merged through LDS; with num_parts > 1 the merged partials go
// to the split-K workspace reduced by launch_attn_reduce (attention.hip).
//
// ROPE = true (GQA decode: every block is ONE token of one sequence, the last of its context):
// `q` is the unrotated fused qkv row and the kernel also does rope_kv.hip's work.  The block's
// heads and the new token's k are turned once, by a thread each pair of 8-column chunks, and go
// to the waves through LDS; the score q.k_new is summed over the 4 lanes of the row with two xor
// shuffles and replaces the (stale) cache score of token ctx - 1, and the new v row replaces that
// token's in the wave's LDS V tile.  The cache loads stay exactly as without ROPE.  Wave 0 of the
// first block of the kv head whose slice holds the token writes k / v to the page slot (slots[t] < 0:
// nothing written).
// Decode reads K and V once and is bound by them, long contexts by how many workgroups share a CU:
// with 160 registers and 35 KB (V in rows, transposed by the read; the queries turned once) 3 fit, so
// the 640 slices of 12 sessions of 1.7k to 5.8k tokens (32 / 8 heads) run at once - 45 us for 184 MB
// where 2 to a CU took 58 in a full round and a quarter one; 64 sessions up to 512: 25.0 -> 20.6 us,
// one of 900: 12.3 -> 10.1.  A grid column was a session on one XCD, some XCDs with two of the 12: slices turned over
// all XCDs take 43 us instead of 47 in a whole step (and 37.6 with FAR); 1, 2, 20 and 64 sessions as long as before.
// FAR: values are loaded past the caches, so that they leave L2 to the keys, whose rows a wave reads as halves of lines, two
// instructions a line.  Keys stay cached: with both past the caches 12 sessions take 43 us, as with neither, and 64 short ones
// 22.7 instead of 18.4.
#include "common.h"
#include "mx_common.h"

namespace mp {

struct RopeFuseM {
  const int64_t* pos;
  const float* cos_t;
  const float* sin_t;
  const int64_t* slots;
  bf16_t* kw;
  bf16_t* vw;
  QkvPart qp;  // qp.part != nullptr: q / k / v from the qkv GEMM's split-K partials (ROPE path)
  uint8_t* mx_ax = nullptr;  // non-null (single-part launches): the output as the W8A8-MX GEMM's
  uint8_t* mx_as = nullptr;  //   activation (mx_common.h) instead of bf16 - the o projection's input
};

typedef __attribute__((ext_vector_type(8))) __bf16 bf16x8_mf;

__device__ __forceinline__ f32x4 mfma_bf16(const u16x8& a, const u16x8& b, const f32x4& c) {
  return __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(bf16x8_mf, a), __builtin_bit_cast(bf16x8_mf, b), c,
                                                 0, 0, 0);
}

typedef short s16x4_mf __attribute__((ext_vector_type(4)));
// each group of 16 lanes reads 4 rows x 16 columns and gets them transposed: lane i column i, 4 rows
__device__ __forceinline__ u16x4 tr_read16(const unsigned char* p) {
  const s16x4_mf v = __builtin_amdgcn_ds_read_tr16_b64_v4i16(
      (__attribute__((address_space(3))) s16x4_mf*)(const_cast<unsigned char*>(p)));
  return __builtin_bit_cast(u16x4, v);
}

constexpr int VT_PITCH = 36;  // bf16 per LDS row of the transposed V tile (32 tokens + pad; 8-B aligned rows)

// FOLD (ROPE only): q / k / v come from the qkv GEMM's split-K slabs through LDS (s_fold).  A
// compile-time choice: as a run-time one the LDS-or-global q / k / v loads compiled to flat
// loads, which count against vmcnt, so the RoPE prologue waited for the K / V stream issued
// before them.
template <int D, int HB, bool ROPE, bool FOLD = false, bool FAR = false>
__global__ __launch_bounds__(256, 3) void attn_mfma_kernel(
    const bf16_t* __restrict__ q, int64_t q_stride, const bf16_t* __restrict__ kc, const bf16_t* __restrict__ vc,
    const int32_t* __restrict__ block_tables, int bt_stride, const int32_t* __restrict__ q_seq,
    const int32_t* __restrict__ q_ctx, const int32_t* __restrict__ qb_tok0, const int32_t* __restrict__ qb_ntok,
    bf16_t* __restrict__ out, float* __restrict__ part_o, float* __restrict__ part_ml, int nkv, int nh,
    int page_log2, int PS, int NP, int NB, float scale_log2, int packed_mt, RopeFuseM rf) {
  constexpr int TB = 16 / HB;
  constexpr int KD = D / 32;  // k-chunks of the QK^T product
  constexpr int DT = D / 16;  // 16-column tiles of O
  // a wave's V tile [32][D] bf16 in its steps, its O rows [16][D + 1] fp32 for the merge after them
  constexpr int OP = D + 1, WB = (16 * OP * 4 + 255) / 256 * 256;
  __shared__ __attribute__((aligned(256))) unsigned char s_wave[4][WB];
  __shared__ float s_m[4][16], s_l[4][16];

  const int p = blockIdx.z;
  const int hbase = blockIdx.y * HB;
  const int g = hbase / (nh / nkv);
  // (decode: a session's slices go over all XCDs; with its kv heads spread as well, whose rows share pages, 12 took 47 us;
  // NB = gridDim.x, as an argument: read as gridDim.x it comes 0.3 us late)
  const int b = ROPE ? xcd_turn(blockIdx.x, NB, p) : blockIdx.x;
  const int tid = threadIdx.x, lane = tid & 63, w = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int c = lane & 15, qd = lane >> 4;
  // ROPE (decode): block b is token b (``decode_qblocks``: one token per block, in order), so the
  // block-table walk starts from q_seq / q_ctx directly - one dependent global load fewer in the
  // chain (q_seq -> page id -> K / V) that sets the decode kernel's time
  const int tok0 = ROPE ? b : qb_tok0[b], ntok = ROPE ? 1 : qb_ntok[b];
  const int seq = q_seq[tok0];
  const int32_t* bt = block_tables + (int64_t)seq * bt_stride;
  const int page_size = 1 << page_log2;
  const int64_t page_stride = (int64_t)nkv * page_size * D;
  const int64_t head_off = (int64_t)g * page_size * D;

  // this lane's row (for Q^T fragments, masking and softmax state): row c
  const int my_t = c / HB, my_h = hbase + c % HB;
  const bool row_ok = my_t < ntok;
  const int my_ctx = row_ok ? q_ctx[tok0 + my_t] : 0;
  int blk_ctx = 0;  // context the block needs = the largest ctx of its tokens (causal: the last)
  for (int i = 0; i < ntok; ++i) blk_ctx = max(blk_ctx, q_ctx[tok0 + i]);
  const int start = p * PS, end = min(start + PS, blk_ctx);

  constexpr int NV = (32 * D * 2) / 1024;  // 16-B V chunks per lane per step
  // (a page's base is the same in the whole wave: scalar bases, 32-bit lane offsets)
  const unsigned klane = c * D + qd * 8;
  auto load_k = [&](int bs, int64_t pg, u16x8 (&kr)[2][KD]) {
    const bf16_t* kpage = kc + pg * page_stride + head_off + (int64_t)(bs & (page_size - 1)) * D;
#pragma unroll
    for (int sub = 0; sub < 2; ++sub)
#pragma unroll
      for (int kd = 0; kd < KD; ++kd)
        kr[sub][kd] = *reinterpret_cast<const u16x8*>(kpage + kd * 32 + (klane + sub * 16 * D));
  };
  auto load_v = [&](int bs, int64_t pg, u16x8 (&vr)[NV]) {
    const bf16_t* vpage = vc + pg * page_stride + head_off + (int64_t)(bs & (page_size - 1)) * D;
    unsigned vlane = lane;
    asm volatile("" : "+v"(vlane));  // (two offsets formed at each use instead of held)
    vlane *= 8;
#pragma unroll
    for (int i = 0; i < NV; ++i) {
      const u16x8* from = reinterpret_cast<const u16x8*>(vpage + (i & 3) * 512 + (vlane + (i >> 2) * 2048));
      vr[i] = FAR ? __builtin_nontemporal_load(from) : *from;
    }
  };
  f32x4 o[DT];
#pragma unroll
  for (int dt = 0; dt < DT; ++dt) o[dt] = (f32x4)(0.f);
  float m = -INFINITY, l = 0.f;
  if (start < end) {  // (a slice past the context: an empty partial)
    // One register set each for a step's K and V: the next step's K is requested as soon as this
    // step's scores are formed, the next V as soon as this V is in LDS, so both are in flight through
    // the rest of the step, and 3 workgroups fit a CU
    u16x8 ka[2][KD], vr[NV];
    const int b_first = start + w * 32;
    const int b_load = min(b_first, (end - 1) & ~31);  // (a wave with no step of its own reads the last one, unused)
    // Issue order = need order (vmcnt retires in order): what the RoPE needs, then the first step's K
    // and V - the page-table round trip and the K / V stream overlap the rotary prologue instead of
    // following it (decode blocks have one or two steps per wave: these dependent round trips, not
    // the bytes, set the kernel time).
    const int64_t pg_first = bt[b_load >> page_log2];
    int64_t pg_next = b_first + 128 < end ? bt[(b_first + 128) >> page_log2] : 0;

    constexpr int CK = D / 8;    // 8-column chunks per head
    constexpr int HK = CK / 2;   // chunk e of a head turns with chunk e + HK (rotate_half)
    constexpr bool from_part = ROPE && FOLD;
    u16x8 qf[KD];
    u16x8 vn = (u16x8)(0);
    int tnew = -1;
    float qk_new = 0.f;
    if constexpr (!ROPE) {
#pragma unroll
      for (int kd = 0; kd < KD; ++kd)
        qf[kd] = row_ok ? *reinterpret_cast<const u16x8*>(q + (int64_t)(tok0 + my_t) * q_stride + (int64_t)my_h * D +
                                                          kd * 32 + qd * 8)
                        : (u16x8)(0);
      load_k(b_load, pg_first, ka);
      load_v(b_load, pg_first, vr);
    } else {
      // The block's HB query heads and its new key are turned ONCE, a pair of chunks a thread, and
      // reach every wave through LDS (each wave turning them for itself held 96 more registers at the
      // time the first K and V are in flight: 244, two workgroups a CU).
      constexpr int NROT = (HB + 1) * HK;
      static_assert(NROT <= 256, "one pair of chunks a thread");
      __shared__ u16x8 s_rot[(HB + 1) * CK];
      const int ri = min(tid, NROT - 1), rh = ri / HK, re = ri % HK;  // (threads past the pairs: the last one again)
      const int rcol = (rh < HB ? hbase + rh : nh + g) * D + re * 8;
      const int64_t kv_slot = rf.slots[tok0];
      const int64_t ci = rf.pos[tok0] * (D / 2) + re * 8;
      u16x8 xa, xb;
      f32x4 cs[2], sn[2];
      // FOLD: the heads, the key and the value summed from the split-K slabs, row-scaled and rounded
      // (common.h qkv_part_finish8: the reduce launch's bits) once per block into LDS - every slab
      // element read once, not once per lane group of every wave
      constexpr int NFOLD = (HB + 2) * CK;
      constexpr int NI = (NFOLD + 255) / 256;  // fold items per thread (256 threads)
      __shared__ u16x8 s_fold[FOLD ? NFOLD : 1];
      int fcol[NI];
      unsigned long long ssv = 0;
      QkvPart8 ff[NI];
      if constexpr (from_part) {
#pragma unroll
        for (int j = 0; j < NI; ++j) {
          const int fi = min(tid + 256 * j, NFOLD - 1);
          fcol[j] = (fi / CK < HB ? (hbase + fi / CK) * D : fi / CK == HB ? (nh + g) * D : (nh + nkv + g) * D) +
                    (fi % CK) * 8;
        }
        ssv = qkv_part_ss_load(rf.qp, tok0);
#pragma unroll
        for (int j = 0; j < NI; ++j) qkv_part_fetch8(rf.qp, tok0, fcol[j], ff[j]);
      } else {
        const bf16_t* qrow = q + (int64_t)tok0 * q_stride;
        xa = *reinterpret_cast<const u16x8*>(qrow + rcol);
        xb = *reinterpret_cast<const u16x8*>(qrow + rcol + D / 2);
        vn = *reinterpret_cast<const u16x8*>(qrow + (nh + nkv + g) * D + (lane % CK) * 8);
      }
#pragma unroll
      for (int i = 0; i < 2; ++i) {
        cs[i] = *reinterpret_cast<const f32x4*>(rf.cos_t + ci + 4 * i);
        sn[i] = *reinterpret_cast<const f32x4*>(rf.sin_t + ci + 4 * i);
      }
      __builtin_amdgcn_sched_barrier(0);  // (as written: the RoPE waits for its own loads only)
      load_k(b_load, pg_first, ka);
      load_v(b_load, pg_first, vr);
      if constexpr (from_part) {
        const float qrs = qkv_part_ss_scale(rf.qp, ssv);
#pragma unroll
        for (int j = 0; j < NI; ++j)
          if (tid + 256 * j < NFOLD) s_fold[tid + 256 * j] = qkv_part_finish8(rf.qp, tok0, fcol[j], ff[j], qrs);
        lds_wait_barrier();  // (lgkmcnt only: the K / V loads stay in flight)
        xa = s_fold[rh * CK + re];
        xb = s_fold[rh * CK + re + HK];
        vn = s_fold[(HB + 1) * CK + lane % CK];
      }
      u16x8 ra, rb;
#pragma unroll
      for (int j = 0; j < 8; ++j) {
        const float c_ = cs[j >> 2][j & 3], s_ = sn[j >> 2][j & 3];
        const float x = bf2f(xa[j]), y = bf2f(xb[j]);
        ra[j] = f2bf(fmaf(x, c_, -(y * s_)));  // (which product is rounded first is fixed)
        rb[j] = f2bf(fmaf(x, s_, y * c_));
      }
      s_rot[rh * CK + re] = ra;
      s_rot[rh * CK + re + HK] = rb;
      lds_wait_barrier();
      float part = 0.f;
#pragma unroll
      for (int kd = 0; kd < KD; ++kd) {
        qf[kd] = row_ok ? s_rot[(my_h - hbase) * CK + kd * 4 + qd] : (u16x8)(0);
        const u16x8 kn = s_rot[HB * CK + kd * 4 + qd];
#pragma unroll
        for (int j = 0; j < 8; ++j) part += bf2f(qf[kd][j]) * bf2f(kn[j]);
      }
      part += __shfl_xor(part, 16, 64);
      part += __shfl_xor(part, 32, 64);
      qk_new = part;
      tnew = blk_ctx - 1;
      if (w == 0 && tnew >= start && tnew < end && kv_slot >= 0 && hbase % (nh / nkv) == 0 && lane < CK) {
        const int64_t dst =
            (kv_slot >> page_log2) * page_stride + head_off + (kv_slot & (page_size - 1)) * D + lane * 8;
        *reinterpret_cast<u16x8*>(rf.kw + dst) = s_rot[HB * CK + lane];
        *reinterpret_cast<u16x8*>(rf.vw + dst) = vn;
      }
    }

    // 16-byte chunk ch of V row tk lies at tk 2 D + 16 (ch ^ 2 (tk & 7)) (mod the row): the 4 rows that a
    // transposed read touches fall on different banks.  This lane's write and read offsets, up to a xor
    // with constants:
    unsigned char* vt = s_wave[w];
    const int tr = qd * 4 + (c >> 2);
    int vw_off = (lane / CK) * (2 * D) + ((lane % CK) ^ (((lane / CK) << 1) & (CK - 1))) * 16;
    int vr_off = tr * (2 * D) + (((c >> 1) & 1) ^ (((tr & 7) << 1) & (CK - 1))) * 16 + (c & 1) * 8;

    const int my_end = min(my_ctx, end);
    // One 32-token step; MORE: the wave has another one 128 tokens on, so all of this one lies inside the
    // slice.  (A compile-time choice: with loads in a branch the waits before V would cover them too.)
    auto step = [&](int b0, auto more) {
      constexpr bool MORE = decltype(more)::value;
      asm volatile("" : "+v"(vw_off), "+v"(vr_off));  // (their xors formed in each step: 12 registers fewer)
      // ---- S^T = K . Q^T for tokens b0 .. b0+31 (two 16-token subtiles) ----
      f32x4 st[2];
#pragma unroll
      for (int sub = 0; sub < 2; ++sub) {
        st[sub] = (f32x4)(0.f);
#pragma unroll
        for (int kd = 0; kd < KD; ++kd) st[sub] = mfma_bf16(ka[sub][kd], qf[kd], st[sub]);
      }
      if constexpr (MORE) load_k(b0 + 128, pg_next, ka);
      // ---- V tile -> LDS (this wave only; in-order LDS needs no barrier); the new token's row from registers ----
      if constexpr (!MORE) {
#pragma unroll
        for (int i = 0; i < NV; ++i) {
          const int tk = b0 + (i * 64 + lane) / CK;
          if (tk >= end) vr[i] = (u16x8)(0);
          if (ROPE && tk == tnew) vr[i] = vn;
        }
      }
#pragma unroll
      for (int i = 0; i < NV; ++i) *reinterpret_cast<u16x8*>(vt + i * 1024 + (vw_off ^ (D == 128 ? (i & 1) * 128 : 0))) = vr[i];
      if constexpr (MORE) {
        load_v(b0 + 128, pg_next, vr);
        if (b0 + 256 < end) pg_next = bt[(b0 + 256) >> page_log2];
      }
      if constexpr (ROPE && !MORE) {  // the new token's score comes from registers
#pragma unroll
        for (int sub = 0; sub < 2; ++sub)
#pragma unroll
          for (int r = 0; r < 4; ++r) st[sub][r] = b0 + sub * 16 + qd * 4 + r == tnew ? qk_new : st[sub][r];
      }
      // ---- online softmax for row c over this lane's 8 tokens {4qd + r, 16 + 4qd + r} ----
      float s8[8];
      float lm = -INFINITY;
#pragma unroll
      for (int sub = 0; sub < 2; ++sub)
#pragma unroll
        for (int r = 0; r < 4; ++r) {
#pragma clang fp contract(off)  // (scores are scaled and rounded before the maximum is taken off)
          const int tk = b0 + sub * 16 + qd * 4 + r;
          const float v = (ROPE && MORE) || tk < my_end ? st[sub][r] * scale_log2 : -INFINITY;
          s8[sub * 4 + r] = v;
          lm = fmaxf(lm, v);
        }
      lm = fmaxf(lm, __shfl_xor(lm, 16, 64));
      lm = fmaxf(lm, __shfl_xor(lm, 32, 64));
      const float m_new = fmaxf(m, lm);
      const float alpha = (m_new == -INFINITY) ? 1.f : exp2f(m - m_new);
      u16x8 pa;
      float ps = 0.f;
#pragma unroll
      for (int j = 0; j < 8; ++j) {
        const float pv = (m_new == -INFINITY) ? 0.f : exp2f(s8[j] - m_new);
        const bf16_t pb = f2bf(pv);
        pa[j] = pb;
        ps += bf2f(pb);  // l accumulates the rounded p that the MFMA uses
      }
      l = l * alpha + ps;
      m = m_new;
      // O rows are 4qd + r: fetch those rows' alpha from lanes 4qd + r (row == lane & 15)
      float ar[4];
#pragma unroll
      for (int r = 0; r < 4; ++r) ar[r] = __shfl(alpha, qd * 4 + r, 64);
      // ---- O += P . V ----
#pragma unroll
      for (int dt = 0; dt < DT; ++dt) {
        const u16x4 lo = tr_read16(vt + (vr_off ^ (dt * 32)));
        const u16x4 hi = tr_read16(vt + 16 * 2 * D + (vr_off ^ (dt * 32)));
        const u16x8 vfrag = {lo[0], lo[1], lo[2], lo[3], hi[0], hi[1], hi[2], hi[3]};
#pragma unroll
        for (int r = 0; r < 4; ++r) o[dt][r] *= ar[r];
        o[dt] = mfma_bf16(pa, vfrag, o[dt]);
      }
    };
    // the walk over this wave's steps b0 = start + 32 w + 128 i
    if (b_first < end) {
      int b0 = b_first;
      for (; b0 + 128 < end; b0 += 128) step(b0, std::true_type{});
      step(b0, std::false_type{});
    }
  }
  // row sums of l over the 4 lanes of each row
  l += __shfl_xor(l, 16, 64);
  l += __shfl_xor(l, 32, 64);
  if (lane < 16) {
    s_m[w][lane] = m;
    s_l[w][lane] = l;
  }
#pragma unroll
  for (int dt = 0; dt < DT; ++dt)
#pragma unroll
    for (int r = 0; r < 4; ++r) reinterpret_cast<float*>(s_wave[w])[(qd * 4 + r) * OP + dt * 16 + c] = o[dt][r];
  __syncthreads();
  // ---- merge the 4 waves; thread -> (row, d) ----
  for (int i = tid; i < 16 * D; i += 256) {
    const int row = i / D, d = i - row * D;
    const int t = row / HB, h = hbase + row % HB;
    if (t >= ntok) continue;
    float M = -INFINITY;
#pragma unroll
    for (int ww = 0; ww < 4; ++ww) M = fmaxf(M, s_m[ww][row]);
    float num = 0.f, den = 0.f;
    if (M != -INFINITY) {
#pragma unroll
      for (int ww = 0; ww < 4; ++ww) {
        const float f = exp2f(s_m[ww][row] - M);
        num += f * reinterpret_cast<const float*>(s_wave[ww])[row * OP + d];
        den += f * s_l[ww][row];
      }
    }
    const int tok = tok0 + t;
    if (NP == 1) {
      const float v = den > 0.f ? num / den : 0.f;
      const int64_t col = (int64_t)h * D + d;
      if (rf.mx_ax != nullptr) {
        // MX block of (row, col): the 32 dims of this row with the same bit 4 and bits 6+ of col -
        // lanes l ^ {1, 2, 4, 8, 32} of this wave (a wave holds 64 consecutive dims of one row, so
        // the ``continue`` above is wave-uniform)
        const float vb = bf2f(f2bf(v));
        float a = fabsf(vb);
        a = fmaxf(a, __shfl_xor(a, 1, 64));
        a = fmaxf(a, __shfl_xor(a, 2, 64));
        a = fmaxf(a, __shfl_xor(a, 4, 64));
        a = fmaxf(a, __shfl_xor(a, 8, 64));
        a = fmaxf(a, __shfl_xor(a, 32, 64));
        const int e = mx_e8m0(a);
        const float qv = fminf(fmaxf(vb * mx_inv_scale(e), -448.f), 448.f);
        rf.mx_ax[mx_ax_off(tok, (int)col, packed_mt)] = (uint8_t)(__builtin_amdgcn_cvt_pk_fp8_f32(qv, 0.f, 0, false) & 255);
        if ((col & 0x2f) == 0) rf.mx_as[mx_as_off(tok, (int)col)] = (uint8_t)e;
        continue;
      }
      out[packed_mt > 0 ? apk_off(tok, (int)col, packed_mt) : (int64_t)tok * nh * D + col] = f2bf(v);
    } else {
      const int64_t hp = ((int64_t)tok * nh + h) * NP + p;
      part_o[hp * D + d] = num;
      if (d == 0) {
        part_ml[hp * 2] = M;
        part_ml[hp * 2 + 1] = den;
      }
    }
  }
}


// Grouped prefill form: a workgroup owns up to NWG (8) query blocks of ONE sequence (one per wave;
// superblock table sb_first / sb_n) and streams each 32-token context step ONCE into LDS for
// all of them - K as a [32][D] tile read back as MFMA A fragments, V transposed as above - so a
// long prompt reads its K/V 4x less often than with one block per workgroup (the one-block
// kernel re-streams the whole causal context for every 16 query rows: 2K-token MHA prefill was
// K/V-bandwidth-bound at ~94 TFLOP/s).  Every wave runs every step (barriers); a wave's rows
// only see tokens < their own ctx, and each wave finishes its own rows (no cross-wave merge).
template <int D, int HB, int NWG>
__global__ __launch_bounds__(NWG * 64) void attn_mfma_grp_kernel(
    const bf16_t* __restrict__ q, int64_t q_stride, const bf16_t* __restrict__ kc, const bf16_t* __restrict__ vc,
    const int32_t* __restrict__ block_tables, int bt_stride, const int32_t* __restrict__ q_seq,
    const int32_t* __restrict__ q_ctx, const int32_t* __restrict__ qb_tok0, const int32_t* __restrict__ qb_ntok,
    const int32_t* __restrict__ sb_first, const int32_t* __restrict__ sb_n, bf16_t* __restrict__ out,
    float* __restrict__ part_o, float* __restrict__ part_ml, int nkv, int nh, int page_log2, int PS, int NP,
    float scale_log2, int packed_mt) {
  constexpr int KD = D / 32;
  constexpr int DT = D / 16;
  constexpr int KP = D + 8;  // K tile row pitch (bf16): rows 272 B apart stagger the banks
  __shared__ __attribute__((aligned(16))) bf16_t s_k[32 * KP];
  __shared__ __attribute__((aligned(16))) bf16_t s_vt[D * VT_PITCH];

  const int p = blockIdx.z;
  const int hbase = blockIdx.y * HB;
  const int g = hbase / (nh / nkv);
  const int tid = threadIdx.x, lane = tid & 63, w = tid >> 6;
  const int c = lane & 15, qd = lane >> 4;
  const int b_first = sb_first[blockIdx.x], nblk = sb_n[blockIdx.x];
  const bool wave_ok = w < nblk;
  const int b = b_first + (wave_ok ? w : 0);
  const int tok0 = qb_tok0[b], ntok = qb_ntok[b];
  const int32_t* bt = block_tables + (int64_t)q_seq[tok0] * bt_stride;
  const int page_size = 1 << page_log2;
  const int64_t page_stride = (int64_t)nkv * page_size * D;
  const int64_t head_off = (int64_t)g * page_size * D;

  const int my_t = c / HB, my_h = hbase + c % HB;
  const bool row_ok = wave_ok && my_t < ntok;
  const int my_ctx = row_ok ? q_ctx[tok0 + my_t] : 0;
  int grp_ctx = 0;  // the context the workgroup streams: the largest ctx of any of its tokens
  for (int bb = b_first; bb < b_first + nblk; ++bb)
    for (int i = 0; i < qb_ntok[bb]; ++i) grp_ctx = max(grp_ctx, q_ctx[qb_tok0[bb] + i]);
  const int start = p * PS, end = min(start + PS, grp_ctx);

  u16x8 qf[KD];
#pragma unroll
  for (int kd = 0; kd < KD; ++kd) {
    if (row_ok) qf[kd] = *reinterpret_cast<const u16x8*>(q + (int64_t)(tok0 + my_t) * q_stride + (int64_t)my_h * D +
                                                         kd * 32 + qd * 8);
    else qf[kd] = (u16x8)(0);
  }
  f32x4 o[DT];
#pragma unroll
  for (int dt = 0; dt < DT; ++dt) o[dt] = (f32x4)(0.f);
  float m = -INFINITY, l = 0.f;

  // the step's K and V (32 tokens, one page: b0 % 32 == 0 and pages hold 32k tokens) are
  // fetched into registers one step ahead, so the global loads of step i+1 are in flight while
  // step i computes out of LDS
  constexpr int NCH = 32 * D / 8;                           // 16-B chunks per tile
  constexpr int CPT = (NCH + NWG * 64 - 1) / (NWG * 64);  // per thread
  u16x8 kreg[CPT], vreg[CPT];
  auto fetch = [&](int s0) {
    const int64_t pg = bt[s0 >> page_log2];
    const bf16_t* kpage = kc + pg * page_stride + head_off + (int64_t)(s0 & (page_size - 1)) * D;
    const bf16_t* vpage = vc + pg * page_stride + head_off + (int64_t)(s0 & (page_size - 1)) * D;
#pragma unroll
    for (int j = 0; j < CPT; ++j) {
      const int i = tid + NWG * 64 * j;
      if (NCH % (NWG * 64) != 0 && i >= NCH) break;
      const int tk = i / (D / 8), d0 = (i % (D / 8)) * 8;
      kreg[j] = *reinterpret_cast<const u16x8*>(kpage + (int64_t)tk * D + d0);
      // V: tokens vary fastest across lanes, so the transposed LDS writes below are 32
      // consecutive bf16 of one d row per half-wave (no bank conflicts; token-major lanes put
      // 16 lanes on 4 banks)
      const int tv = i % 32, dv = (i / 32) * 8;
      vreg[j] = *reinterpret_cast<const u16x8*>(vpage + (int64_t)tv * D + dv);
    }
  };
  if (start < end) fetch(start);
  for (int b0 = start; b0 < end; b0 += 32) {
#pragma unroll
    for (int j = 0; j < CPT; ++j) {
      const int i = tid + NWG * 64 * j;
      if (NCH % (NWG * 64) != 0 && i >= NCH) break;
      const int tk = i / (D / 8), d0 = (i % (D / 8)) * 8;
      const bool past = b0 + tk >= end;  // past the context: stale cache bytes never meet a p = 0
      *reinterpret_cast<u16x8*>(s_k + tk * KP + d0) = past ? (u16x8)(0) : kreg[j];
      const int tv = i % 32, dv = (i / 32) * 8;
      const bool vpast = b0 + tv >= end;
#pragma unroll
      for (int e = 0; e < 8; ++e) s_vt[(dv + e) * VT_PITCH + tv] = vpast ? (bf16_t)0 : vreg[j][e];
    }
    __syncthreads();
    if (b0 + 32 < end) fetch(b0 + 32);
    if (wave_ok) {
      f32x4 st[2];
#pragma unroll
      for (int sub = 0; sub < 2; ++sub) {
        st[sub] = (f32x4)(0.f);
#pragma unroll
        for (int kd = 0; kd < KD; ++kd) {
          const u16x8 kf = *reinterpret_cast<const u16x8*>(s_k + (sub * 16 + c) * KP + kd * 32 + qd * 8);
          st[sub] = mfma_bf16(kf, qf[kd], st[sub]);
        }
      }
      float s8[8];
      float lm = -INFINITY;
#pragma unroll
      for (int sub = 0; sub < 2; ++sub)
#pragma unroll
        for (int r = 0; r < 4; ++r) {
          const int tk = b0 + sub * 16 + qd * 4 + r;
          const float v = (tk < my_ctx && tk < end) ? st[sub][r] * scale_log2 : -INFINITY;
          s8[sub * 4 + r] = v;
          lm = fmaxf(lm, v);
        }
      lm = fmaxf(lm, __shfl_xor(lm, 16, 64));
      lm = fmaxf(lm, __shfl_xor(lm, 32, 64));
      const float m_new = fmaxf(m, lm);
      const float alpha = (m_new == -INFINITY) ? 1.f : exp2f(m - m_new);
      u16x8 pa;
      float ps = 0.f;
#pragma unroll
      for (int j = 0; j < 8; ++j) {
        const float pv = (m_new == -INFINITY) ? 0.f : exp2f(s8[j] - m_new);
        const bf16_t pb = f2bf(pv);
        pa[j] = pb;
        ps += bf2f(pb);
      }
      l = l * alpha + ps;
      m = m_new;
      float ar[4];
#pragma unroll
      for (int r = 0; r < 4; ++r) ar[r] = __shfl(alpha, qd * 4 + r, 64);
#pragma unroll
      for (int dt = 0; dt < DT; ++dt) {
        const bf16_t* vrow = s_vt + (dt * 16 + c) * VT_PITCH;
        const u16x4 lo = *reinterpret_cast<const u16x4*>(vrow + qd * 4);
        const u16x4 hi = *reinterpret_cast<const u16x4*>(vrow + 16 + qd * 4);
        const u16x8 vb = {lo[0], lo[1], lo[2], lo[3], hi[0], hi[1], hi[2], hi[3]};
#pragma unroll
        for (int r = 0; r < 4; ++r) o[dt][r] *= ar[r];
        o[dt] = mfma_bf16(pa, vb, o[dt]);
      }
    }
    __syncthreads();  // the next step overwrites the tiles
  }
  if (!wave_ok) return;
  l += __shfl_xor(l, 16, 64);
  l += __shfl_xor(l, 32, 64);
  // this lane holds O rows 4 qd + r (columns dt * 16 + c); row rr's m / l live in lane rr
#pragma unroll
  for (int r = 0; r < 4; ++r) {
    const int rr = qd * 4 + r;
    const float lr = __shfl(l, rr, 64), mr = __shfl(m, rr, 64);
    const int t = rr / HB, h = hbase + rr % HB;
    if (t >= ntok) continue;
    const int tok = tok0 + t;
#pragma unroll
    for (int dt = 0; dt < DT; ++dt) {
      const int d = dt * 16 + c;
      if (NP == 1) {
        const float v = lr > 0.f ? o[dt][r] / lr : 0.f;
        const int64_t col = (int64_t)h * D + d;
        out[packed_mt > 0 ? apk_off(tok, (int)col, packed_mt) : (int64_t)tok * nh * D + col] = f2bf(v);
      } else {
        const int64_t hp = ((int64_t)tok * nh + h) * NP + p;
        part_o[hp * D + d] = o[dt][r];
        if (d == 0) {
          part_ml[hp * 2] = mr;
          part_ml[hp * 2 + 1] = lr;
        }
      }
    }
  }
}

template <int D, int HB>
static void launch_attn_mfma(const void* q, int64_t q_stride, const void* kc, const void* vc, const int32_t* bt,
                             int bt_stride, const int32_t* q_seq, const int32_t* q_ctx, const int32_t* qb_tok0,
                             const int32_t* qb_ntok, int NB, void* out, float* ws_o, float* ws_ml, int nkv, int nh,
                             int page_log2, int PS, int NP, float scale_log2, int packed_mt, const RopeFuseM& rf,
                             const int32_t* sb_first, const int32_t* sb_n, int NSB, hipStream_t stream) {
  if (sb_first != nullptr && NSB > 0 && rf.pos == nullptr) {
    hipLaunchKernelGGL((attn_mfma_grp_kernel<D, HB, 8>), dim3(NSB, nh / HB, NP), dim3(512), 0, stream, (const bf16_t*)q,
                       q_stride, (const bf16_t*)kc, (const bf16_t*)vc, bt, bt_stride, q_seq, q_ctx, qb_tok0, qb_ntok,
                       sb_first, sb_n, (bf16_t*)out, ws_o, ws_ml, nkv, nh, page_log2, PS, NP, scale_log2, packed_mt);
    return;
  }
  auto go = [&](auto kern) {
    hipLaunchKernelGGL(kern, dim3(NB, nh / HB, NP), dim3(256), 0, stream, (const bf16_t*)q, q_stride,
                       (const bf16_t*)kc, (const bf16_t*)vc, bt, bt_stride, q_seq, q_ctx, qb_tok0, qb_ntok,
                       (bf16_t*)out, ws_o, ws_ml, nkv, nh, page_log2, PS, NP, NB, scale_log2, packed_mt, rf);
  };
  // Slices of 512 tokens on (4 steps a wave): values past the caches, see above.  Both forms, us: 12 sessions of 1500 to 6000
  // tokens (slices of 1024) 43.5 -> 37.6, 32 of 700 to 2200 (1024) 41.3 -> 35.8, 64 of 500 to 1000 (512) 42.8 -> 35.7, 8 of
  // 1500 to 6000 (512) 26.6 -> 26.2; shorter slices, few steps that wait for each load: 48 of 300 to 700 (384) 21.0 -> 21.9,
  // 4 of 2000 to 6000 (256) 16.0 -> 16.8, 64 of 100 to 512 (256) 18.4 -> 19.4.
  // Other heads, 12 to 64 sessions of 500 to 7000 tokens: 64 / 8, 16 / 2, 8 / 2 and 8 / 1 of 128 take 5 to 17 % less, 64 / 8,
  // 32 / 8 and 16 / 4 of 64 take 4 to 13 % less.
  const bool far = PS >= 512;
  if (rf.pos && rf.qp.part) far ? go(attn_mfma_kernel<D, HB, true, true, true>) : go(attn_mfma_kernel<D, HB, true, true>);
  else if (rf.pos) far ? go(attn_mfma_kernel<D, HB, true, false, true>) : go(attn_mfma_kernel<D, HB, true, false>);
  else go(attn_mfma_kernel<D, HB, false, false>);
}

void launch_attn_reduce(const float* part_o, const float* part_ml, void* out, int rows, int NP, int D, int nh, int packed_mt,
                        hipStream_t stream);  // attention.hip

}  // namespace mp

// Query blocks: qb_tok0[i] = first flat token of block i, qb_ntok[i] = its token count
// (<= 16 / heads_per_block, all from one sequence).  heads_per_block = min(nh / nkv, 16).
// Superblocks (optional, prefill): sb_first[j] / sb_n[j] = runs of <= 8 consecutive query blocks
// of one sequence, one workgroup each (attn_mfma_grp_kernel).
extern "C" int mp_attention_mfma(const void* q, int64_t q_stride, const void* kc, const void* vc, const int32_t* bt,
                                 int bt_stride, const int32_t* q_seq, const int32_t* q_ctx, const int32_t* qb_tok0,
                                 const int32_t* qb_ntok, int NB, void* out, float* workspace, int T, int nh, int nkv,
                                 int D, int page_size, int PS, int NP, float scale, int packed_mt,
                                 const int64_t* rope_pos, const float* cos_t, const float* sin_t,
                                 const int64_t* slots, const int32_t* sb_first, const int32_t* sb_n, int NSB,
                                 const void* qkv_part_v, void* mx_ax, void* mx_as, hipStream_t stream) {
  (void)hipGetLastError();  // an earlier non-mpamd HIP call's stale error is not this launch's
  using namespace mp;
  RopeFuseM rf{rope_pos, cos_t, sin_t, slots, (bf16_t*)const_cast<void*>(kc), (bf16_t*)const_cast<void*>(vc),
               QkvPart{nullptr, 0, 0, 0, nullptr, 0.f, 0.f}};
  const QkvPart* qkv_part = static_cast<const QkvPart*>(qkv_part_v);  // layout mirrored by bindings.cpp
  if (qkv_part != nullptr && qkv_part->part != nullptr) {
    if (rope_pos == nullptr || qkv_part->S < 1) return -4;  // partials only on the fused RoPE decode path
    rf.qp = *qkv_part;
  }
  if (mx_ax != nullptr) {  // MX output: the fused RoPE decode path, one part, packed rows, 128-dim heads
    if (rope_pos == nullptr || NP != 1 || packed_mt <= 0 || D != 128 || mx_as == nullptr) return -7;
    rf.mx_ax = (uint8_t*)mx_ax;
    rf.mx_as = (uint8_t*)mx_as;
  }
  if (NB == 0 || T == 0) return 0;
  if (nh % nkv != 0 || PS % 128 != 0 || NP < 1 || page_size % 32 != 0) return -1;
  int page_log2 = 0;
  while ((1 << page_log2) < page_size) ++page_log2;
  if ((1 << page_log2) != page_size) return -2;
  const int nrep = nh / nkv;
  // the whole GQA group of a kv head in one workgroup's MFMA rows (spreading a group's heads over
  // several workgroups that re-read the same K / V measured 1.6-2.7x slower, profiles/r4k)
  const int hb = nrep >= 16 ? 16 : nrep;
  if (nrep % hb) return -3;
  const float scale_log2 = scale * 1.4426950408889634f;
  float* ws_o = workspace;
  float* ws_ml = workspace + (int64_t)T * nh * NP * D;
#define MP_AM_CASE(DD, HH)                                                                                      \
  if (D == DD && hb == HH) {                                                                                    \
    launch_attn_mfma<DD, HH>(q, q_stride, kc, vc, bt, bt_stride, q_seq, q_ctx, qb_tok0, qb_ntok, NB, out, ws_o,  \
                             ws_ml, nkv, nh, page_log2, PS, NP, scale_log2, packed_mt, rf, sb_first, sb_n, NSB, \
                             stream);                                                                           \
    goto launched;                                                                                              \
  }
  MP_AM_CASE(128, 1)
  MP_AM_CASE(128, 2)
  MP_AM_CASE(128, 4)
  MP_AM_CASE(128, 8)
  MP_AM_CASE(128, 16)
  MP_AM_CASE(64, 1)
  MP_AM_CASE(64, 2)
  MP_AM_CASE(64, 4)
  MP_AM_CASE(64, 8)
  MP_AM_CASE(64, 16)
#undef MP_AM_CASE
  return -4;
launched:
  if (NP > 1)
    launch_attn_reduce(ws_o, ws_ml, out, T * nh, NP, D, nh, packed_mt, stream);
  return (int)hipGetLastError();
}
