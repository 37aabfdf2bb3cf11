// Main loop of the 256 x 256 product tiles (moe.hip: experts, gemm_prompt.hip: prompts): eight waves of 64 rows x 128 weight
// rows, 64 columns a stage.  A workgroup stays on its CU for all its tiles, and its loads run ahead across them.
//   * Rows arrive 128 bytes at a time (8 rows an instruction), whole cache lines: 32-column stages fetch every line twice,
//     and 256 rows of lines are the whole L1, so the second half came from L2 again.  The 16-byte chunks of a row are
//     permuted by its low bits on the way in, which leaves the operand reads free of bank conflicts (none counted).
//     Weights come the same way, packed in fragment order ([N / 16, K / 32, 64, 8]) as they lie, or as columns of a [K, N]
//     matrix: 64 rows of 512 bytes a stage.  Their 32-byte chunks are permuted by the row, and the transposing LDS read
//     turns them into operands (8 rows' 32 bytes in 8 different groups of banks).  The compiler lets that read wait for all
//     loads into LDS that it knows of, so this form issues its own; they have no registers to write.
//   * All 160 KiB of LDS are a ring of five slots of one operand's stage.  Behind the one barrier of a stage its two slots are
//     free: the rows of the stage after the next go to one, the weights of the stage after that to the other, so that
//     weights, which come from HBM, have more than a stage and a half to arrive.  With two slots an operand and workgroups
//     that end with their tile, weights that no cache held cost 4096 x 16384 x 4096 446 us (now 384, the library 353),
//     4096 x 4096 x 14336 362 (322, 314), 6421 x 12288 x 4096 527 (474, 502); the early slot on the rows' side took 404,
//     342 and 497 us.
//   * The operands of a half stage are read from LDS while the MFMAs of the half before it run, across the barrier, one read
//     to two MFMAs; the stage's loads are spread over the half stage behind the barrier: eight at once hold up the MFMAs that
//     stand behind them.
//   * A wave whose 64 rows are past the last only loads; the two waves of a SIMD have different rows, so a tile of up to 128
//     rows takes half the MFMA time (0.8 of a whole tile's where its weights come from HBM: the ring covers less of the wait).
// Bound by MFMA issue (three quarters of the time; the clock falls to 1.8 GHz under it) and by the issue of the loads, an eighth.
// Measured and left: four waves of 128 x 128 (2 to 5 % more), a second barrier that frees the slot sooner (6 % more), 32 x 32
// x 16 MFMAs (12 % more), loads over both halves of a stage (up to 8 % more).
#pragma once
#include "common.h"

namespace mp {

struct WideTile {
  static constexpr int BM = 256, BN = 256, MW = 4, NW = 8, WM = 4, WN = 2, SLOTS = 5, SLOT = 256 * 128, LDS = SLOTS * SLOT;
  static constexpr int CUS = 256;  // workgroups of a launch at most: one to a CU
  enum Weights { ROWS, PACKED, COLUMNS };
  typedef __attribute__((ext_vector_type(8))) __bf16 bf16x8;
  typedef __attribute__((ext_vector_type(4))) short s16x4;
  typedef __attribute__((ext_vector_type(2))) uint32_t u32x2;
  typedef __attribute__((ext_vector_type(4))) uint32_t u32x4;
  typedef __attribute__((address_space(3))) void* lptr_t;

  static __device__ __forceinline__ int wave() { return __builtin_amdgcn_readfirstlane(threadIdx.x >> 6); }
  static __device__ __forceinline__ int wm() { return wave() / WN; }  // (the waves of a SIMD, 4 apart, have different rows)
  static __device__ __forceinline__ int wn() { return wave() % WN; }
  // row of the tile that piece j of this wave reads on this lane, and the byte of it in a stage
  static __device__ __forceinline__ int piece_row(int j) { return 8 * (4 * wave() + j) + ((threadIdx.x & 63) >> 3); }
  static __device__ __forceinline__ int piece_byte() { return 16 * ((threadIdx.x & 7) ^ ((threadIdx.x & 63) >> 3)); }
  // the same of packed weights: 16-row tile and byte
  static __device__ __forceinline__ int packed_tile(int j) { return 2 * wave() + (j >> 1); }
  static __device__ __forceinline__ int packed_byte(int j) { return 1024 * (j & 1) + (threadIdx.x & 63) * 16; }

  // the same of columns: row of a stage, and first of 8 columns
  static __device__ __forceinline__ int column_row(int j) { return 2 * (4 * wave() + j) + ((threadIdx.x & 63) >> 5); }
  static __device__ __forceinline__ int column_first(int j) {
    const int row = column_row(j), chunk = (threadIdx.x & 31) >> 1;
    return 16 * (chunk ^ ((row & 3) | (row >> 3 & 1) << 2)) + 8 * (threadIdx.x & 1);
  }

  // Where an operand of a tile comes from: this lane's byte offsets of the wave's pieces from ``at`` bytes behind the base on,
  // ``step`` bytes a stage.
  struct Source {
    __amdgpu_buffer_rsrc_t base;
    u32x4 words;  // of ``base``
    uint32_t off[4], at, step;
    __device__ __forceinline__ void from(const void* p, uint32_t bytes, uint32_t stage) {
      base = __builtin_amdgcn_make_buffer_rsrc(const_cast<void*>(p), (short)0, (int)bytes, 0x00020000);
      words = (u32x4){(uint32_t)(uintptr_t)p, (uint32_t)((uintptr_t)p >> 32) & 0xffff, bytes, 0x00020000};
      at = 0, step = stage;
    }
  };

  // The workgroup's tiles 0 .. count - 1 (at least one).  ``work``:
  //   int stages(k)                  stages of tile k, at least one
  //   void rows(k, Source&)          its rows
  //   void weights(k, Source&)       its weight rows
  //   bool live(k)                   has this wave rows in it?
  //   bool store(k, acc)             acc[i][j]: weight rows 16 (8 wn + i) .. x rows 16 (4 wm + j) ..; lane: row lane % 16, weight
  //                                  rows 4 (lane / 16) .. + 3.  True: at least work.STORES stores were issued for sure.
  // Ends with no load in flight.
  template <Weights FORM, class Work>
  static __device__ __forceinline__ void run(char* smem, int count, const Work& work) {
    const int lane = threadIdx.x & 63, c16 = lane & 15, g4 = lane >> 4;
    char* mine = smem + wave() * 4096;
    Source x, w;
    int xk = 0, wk = 0, xleft = work.stages(0), wleft = xleft;  // the tile that is being loaded, its stages left
    work.rows(0, x);
    work.weights(0, w);
    auto load = [&](const Source& s, int j, int slot) {
      const lptr_t to = (lptr_t)(mine + slot * SLOT + j * 1024);
      if constexpr (FORM == COLUMNS)  // (m0: nothing else of this form uses it; 5 cycles from a scalar that a vector instruction wrote to its use)
        asm volatile("s_mov_b32 m0, %0\n\ts_nop 4\n\tbuffer_load_dwordx4 %1, %2, %3 offen lds" ::"s"((uint32_t)(uintptr_t)to),
                     "v"(s.off[j]), "s"(s.words), "s"(s.at)
                     : "memory");
      else
        __builtin_amdgcn_raw_ptr_buffer_load_lds(s.base, to, 16, s.off[j], s.at, 0, 0);
    };
    auto load_x = [&](int j, int slot) { load(x, j, slot); };
    auto load_w = [&](int j, int slot) { load(w, j, slot); };
    // (past the last tile its last stage is loaded again: nothing reads it, and the counts stay what they are)
    auto next_x = [&] {
      if (--xleft > 0) x.at += x.step;
      else if (xk + 1 < count) xleft = work.stages(++xk), work.rows(xk, x);
      else xleft = 1;
    };
    auto next_w = [&] {
      if (--wleft > 0) w.at += w.step;
      else if (wk + 1 < count) wleft = work.stages(++wk), work.weights(wk, w);
      else wleft = 1;
    };
    // a row's chunk c lies at 16 (c ^ row % 8)
    const int s0 = 16 * (g4 ^ (c16 & 7)), s1 = 16 * ((4 + g4) ^ (c16 & 7));
    const int xr = (16 * MW * wm() + c16) * 128;
    const int wr = FORM == PACKED    ? 2048 * NW * wn() + lane * 16
                   : FORM == COLUMNS ? (8 * g4 + (c16 >> 2)) * 512 + 256 * wn() + 32 * (c16 >> 2 | (g4 & 1) << 2) + 8 * (c16 & 3)
                                     : (16 * NW * wn() + c16) * 128;
    u16x8 xa[MW], wa[NW], xb[MW], wb[NW];
    f32x4 acc[NW][MW];
    auto multiply1 = [&](int i, const u16x8(&xf)[MW], const u16x8(&wf)[NW]) {
#pragma unroll
      for (int j = 0; j < MW; ++j)
        acc[i][j] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(bf16x8, wf[i]), __builtin_bit_cast(bf16x8, xf[j]),
                                                            acc[i][j], 0, 0, 0);
    };
    auto multiply = [&](const u16x8(&xf)[MW], const u16x8(&wf)[NW]) {
#pragma unroll
      for (int i = 0; i < NW; ++i) multiply1(i, xf, wf);
    };
    int px = 1, pw = 0;  // slots of the stage's rows and weights
    auto take1 = [&](int h, int r, u16x8(&xf)[MW], u16x8(&wf)[NW]) {  // one operand of a half stage
      if (r < MW) {
        xf[r] = *reinterpret_cast<const u16x8*>(smem + px * SLOT + xr + (h ? s1 : s0) + r * 2048);
      } else if constexpr (FORM == COLUMNS) {
        const char* p = smem + ((pw * SLOT + wr) ^ (32 * (r - MW))) + h * 16384;
        const s16x4 lo = __builtin_amdgcn_ds_read_tr16_b64_v4i16((__attribute__((address_space(3))) s16x4*)(p));
        const s16x4 hi = __builtin_amdgcn_ds_read_tr16_b64_v4i16((__attribute__((address_space(3))) s16x4*)(p + 2048));
        wf[r - MW] = __builtin_bit_cast(u16x8, __builtin_shufflevector(lo, hi, 0, 1, 2, 3, 4, 5, 6, 7));
      } else {
        wf[r - MW] = *reinterpret_cast<const u16x8*>(smem + pw * SLOT + wr + (FORM == PACKED ? h * 1024 : h ? s1 : s0) + (r - MW) * 2048);
      }
    };
    auto take = [&](int h, u16x8(&xf)[MW], u16x8(&wf)[NW]) {
#pragma unroll
      for (int r = 0; r < MW + NW; ++r) take1(h, r, xf, wf);
    };
    auto fill = [&](int m, int freed_x, int freed_w) {  // load m of the eight behind a barrier: rows of the next stage but one
      if (m < 4) load_x(m, freed_w);                    // where the stage's weights were, then weights of the one behind it
      else load_w(m - 4, freed_x);
    };
    // the order inside a half stage: 32 MFMAs, a read behind each second, a load behind each fourth.  Without the fences the
    // compiler moves the MFMAs behind the barrier and the reads stand alone.
    auto order = [&](bool loads) {
#pragma unroll
      for (int m = 0; m < NW * MW; ++m) {
        __builtin_amdgcn_sched_group_barrier(0x008, 1, 0);
        if (m < 24 && m % 2) __builtin_amdgcn_sched_group_barrier(0x100, 1, 0);
        if (FORM == COLUMNS && m < 24 && m % 2 && m / 2 >= MW) __builtin_amdgcn_sched_group_barrier(0x100, 1, 0);
        if (loads && m % 4 == 3) __builtin_amdgcn_sched_group_barrier(0x010, 1, 0);
      }
      __builtin_amdgcn_sched_barrier(0);
    };
    auto turn = [&] {  // to the next stage's slots
      px = px >= SLOTS - 2 ? px + 2 - SLOTS : px + 2;
      pw = pw >= SLOTS - 2 ? pw + 2 - SLOTS : pw + 2;
    };
    // the next stage has landed for all waves, and all have read this one.  In flight: the weights of the stage after it and
    // the stores of the tile before
    auto meet = [&](int stored) {
      if (stored) asm volatile("s_waitcnt vmcnt(%0)" ::"n"(4 + Work::STORES) : "memory");
      else asm volatile("s_waitcnt vmcnt(4)" ::: "memory");
      lds_wait_barrier();
      __builtin_amdgcn_sched_barrier(0);
    };
#pragma unroll 1
    for (int s = 0; s < SLOTS; s += 2) {  // w 0, x 0, w 1, x 1, w 2
#pragma unroll
      for (int j = 0; j < 4; ++j) load_w(j, s);
      next_w();
      if (s + 1 == SLOTS) break;
#pragma unroll
      for (int j = 0; j < 4; ++j) load_x(j, s + 1);
      next_x();
    }
    asm volatile("s_waitcnt vmcnt(12)" ::: "memory");
    lds_wait_barrier();
    take(0, xa, wa);
    int stored = 0;
    for (int k = 0; k < count; ++k) {
      const int n = work.stages(k);
      if (!work.live(k)) {
        for (int st = 0; st < n; ++st) {
          meet(stored);
          stored = 0;
          const int fx = px, fw = pw;
          turn();
#pragma unroll
          for (int m = 0; m < 8; ++m) fill(m, fx, fw);
          next_x();
          next_w();
        }
        take(0, xa, wa);
        continue;
      }
#pragma unroll
      for (int i = 0; i < NW; ++i)
#pragma unroll
        for (int j = 0; j < MW; ++j) acc[i][j] = (f32x4)(0.f);
      for (int st = 0; st < n; ++st) {
        __builtin_amdgcn_sched_barrier(0);
        take(1, xb, wb);
        multiply(xa, wa);
        order(false);
        meet(stored);
        stored = 0;
        const int fx = px, fw = pw;
        turn();
        if constexpr (FORM == COLUMNS) {  // (its loads are of no kind that ``order`` knows)
#pragma unroll
          for (int i = 0; i < NW; ++i) {
            if (i < 6) take1(0, 2 * i, xa, wa), take1(0, 2 * i + 1, xa, wa);
            multiply1(i, xb, wb);
            fill(i, fx, fw);
            __builtin_amdgcn_sched_barrier(0);
          }
          next_x();
          next_w();
          continue;
        }
#pragma unroll
        for (int m = 0; m < NW * MW; ++m) {  // (loads write LDS: the compiler keeps the order of loads and reads)
          if (m < 24 && m % 2) take1(0, m / 2, xa, wa);
          if (m % 4 == 3) fill(m / 4, fx, fw);
        }
        multiply(xb, wb);
        order(true);
        next_x();
        next_w();
      }
      stored = work.store(k, acc);
    }
    asm volatile("s_waitcnt vmcnt(0) lgkmcnt(0)" ::: "memory");
  }

  // Rows of ``acc`` from m on (those below ``end``) to out[row][cols], columns from ``col`` on.  GLU: ``act`` makes one of each
  // two fragments (gate, up), else of each one.  A lane holds 4 columns of a row in a fragment; neighbouring fragments trade
  // halves between the lane's rows of 16, so that a lane stores 16 bytes and an instruction 64 bytes of each of 16 rows (8
  // bytes a lane: 6421 x 12288 x 4096 506 -> 480 us).  ``wide``: out is 16-byte aligned.  True: all of them were stored.
  static constexpr int put_stores(bool glu) { return MW * NW / (glu ? 4 : 2); }
  template <bool GLU, class Act>
  static __device__ __forceinline__ bool put(bf16_t* out, int cols, bool wide, int m, int end, int col, const f32x4 (&acc)[NW][MW],
                                             Act act) {
    constexpr int S = GLU ? 2 : 1;
    const int c16 = threadIdx.x & 15, g4 = (threadIdx.x & 63) >> 4, lc = col + 16 * (g4 & 1) + 8 * (g4 >> 1);
    const bool whole = wide && m + 16 * MW <= end && col + 16 * NW / S <= cols;
    bf16_t* at = out + (int64_t)(m + c16) * cols + lc;
    auto each = [&](auto store) {
#pragma unroll
      for (int j = 0; j < MW; ++j) {
#pragma unroll
        for (int i = 0; i < NW; i += 2 * S) {
          uint32_t d[2][2];
#pragma unroll
          for (int h = 0; h < 2; ++h) {
            float y[4];
            act(acc[i + h * S][j], acc[i + h * S + S - 1][j], y);
#pragma unroll
            for (int r = 0; r < 2; ++r) d[h][r] = (uint32_t)f2bf(y[2 * r]) | (uint32_t)f2bf(y[2 * r + 1]) << 16;
          }
          const u32x2 a = __builtin_bit_cast(u32x2, __builtin_amdgcn_permlane16_swap(d[0][0], d[1][0], false, false));
          const u32x2 b = __builtin_bit_cast(u32x2, __builtin_amdgcn_permlane16_swap(d[0][1], d[1][1], false, false));
          store(j, 16 * i / S, at + (int64_t)16 * j * cols + 16 * i / S, (u32x4){a[0], b[0], a[1], b[1]});
        }
      }
    };
    if (whole) {
      each([](int, int, bf16_t* p, const u32x4& v) { *reinterpret_cast<u32x4*>(p) = v; });
    } else {
      each([&](int j, int c, bf16_t* p, const u32x4& v) {
        if (m + 16 * j + c16 >= end || lc + c >= cols) return;  // (columns come in sixteens)
        *reinterpret_cast<u32x2*>(p) = (u32x2){v[0], v[1]};
        *reinterpret_cast<u32x2*>(p + 4) = (u32x2){v[2], v[3]};
      });
    }
    return whole;
  }
};

}  // namespace mp
