// Main loop of the 256 x 256 product tiles (moe.hip: experts, gemm_prompt.hip: prompts): four waves of 128 rows x 128 weight
// rows, 64 columns a stage.  A workgroup stays on its CU for all its tiles, and its loads run ahead across them.
//   * Rows arrive 128 bytes at a time (8 rows an instruction), whole cache lines: 32-column stages fetch every line twice,
//     and 256 rows of lines are the whole L1, so the second half came from L2 again.  The 16-byte chunks of a row are
//     permuted by its low bits on the way in, which leaves the operand reads free of bank conflicts (none counted).
//     Weights come the same way, packed in fragment order ([N / 16, K / 32, 64, 8]) as they lie, or as columns of a [K, N]
//     matrix: 64 rows of 512 bytes a stage.  Their 32-byte chunks are permuted by the row, and the transposing LDS read
//     turns them into operands (8 rows' 32 bytes in 8 different groups of banks).  The compiler lets that read wait for all
//     loads into LDS that it knows of, so this form issues its own; they have no registers to write.
//   * All 160 KiB of LDS are a ring of five slots of one operand's stage.  Behind the one barrier of a stage its two slots are
//     free: the rows of the stage after the next go to one, and before the next barrier the weights of the stage after
//     that to the other.  Rows and weights are thus always at the same stage, and a stage's loads, one to eight MFMAs, never
//     wait for each other.
//   * A wave has its SIMD for itself: 256 sums in accumulation registers, the operands of two half stages in the others.  It
//     reads 128 KB of operands a stage and CU where eight waves of 64 x 128 read 192.  Operands of a half stage are read
//     while the MFMAs of the half before it run, across the barrier, one read to three MFMAs.
//   * The MFMAs stand in inline asm and in this order: left to the compiler, sums move from register to register.  From one
//     to the next only one operand changes (blocks of 2 x 2, there and back), which costs less power and so lets the clock
//     rise: 3 % of a loop of MFMAs alone, 1 to 2 % here.
//   * Nothing in the loop but the loads' 8 instructions depends on the tile: a tile moves the base of what is loaded, not
//     the lanes' offsets, and what is behind its rows and weights is behind the end of the buffer, which loads as zero.
//   * A tile of up to 128 rows has 64 rows a wave and half the MFMAs.
// Counters of 4096 x 8192 x 8192, two tiles of 128 stages a workgroup, their ends counted in: 2480 cycles a stage, 2048 of them MFMAs
// (82 % busy), no bank conflicts; columns 2720 (75 %).  Bound by MFMA issue and, at 1.7 to 2.0 of 2.4 GHz, by power.  Eight waves,
// whose loop decided anew at each stage what to load next, and now, in turn: 4096 x 4096 x 16384 384, 355 us; 6421 x
// 12288 x 4096 469, 440; 2700 x 28672 x 4096 gated 480, 454; columns of 4096 x 4096 x 16384 400, 381, 1554 x 4096 x 28672
// 349, 332, but of 60 x 4096 x 28672 (a tile of half the rows, K in parts) 55, 60.
// Measured and left: loads in the first half stage behind the barrier alone (2 to 6 % more), one load to 4 to 6 MFMAs, one read
// to 2 or 4, 32 x 32 x 16 MFMAs (12 % more on eight waves).
#pragma once
#include "common.h"

namespace mp {

// F: fragments of 16 rows that a wave has of either operand: 8, the form above, or 4, see gemm_mid.hip.
template <int F, int SLOTS_>
struct TileLoop {
  static constexpr int BM = 32 * F, BN = 32 * F, MW = F, NW = F, WM = 2, WN = 2, THREADS = 64 * WM * WN;
  static constexpr int PIECES = F;  // loads of a wave and operand in a stage
  static constexpr int SLOTS = SLOTS_, SLOT = BM * 128, LDS = SLOTS * SLOT;
  static constexpr int AHEAD = (SLOTS - 1) / 2;  // stages that loads are ahead
  static_assert(SLOTS % 2 == 1 && SLOTS >= 5 && LDS <= 160 * 1024);
  static constexpr int ON_CU = 160 * 1024 / LDS;  // workgroups on a CU
  static constexpr int CUS = 256 * ON_CU;      // workgroups of a launch at most
  static constexpr int LINE = 2 * BN;          // bytes of a row of columns
  enum Weights { ROWS, PACKED, COLUMNS };
  template <int V>
  struct Int {
    static constexpr int value = V;
  };
  typedef __attribute__((ext_vector_type(8))) __bf16 bf16x8;
  typedef __attribute__((ext_vector_type(2))) __bf16 bf16x2;
  typedef __attribute__((ext_vector_type(2))) float f32x2;
  typedef __attribute__((ext_vector_type(4))) short s16x4;
  typedef __attribute__((ext_vector_type(2))) uint32_t u32x2;
  typedef __attribute__((ext_vector_type(4))) uint32_t u32x4;
  typedef __attribute__((address_space(3))) void* lptr_t;

  static __device__ __forceinline__ int wave() { return __builtin_amdgcn_readfirstlane(threadIdx.x >> 6); }
  static __device__ __forceinline__ int wm() { return wave() / WN; }
  static __device__ __forceinline__ int wn() { return wave() % WN; }
  // row of the tile that piece j of this wave reads on this lane (of ``pieces`` a wave), and the byte of it in a stage
  static __device__ __forceinline__ int piece_row(int j, int pieces = PIECES) { return 8 * (pieces * wave() + j) + ((threadIdx.x & 63) >> 3); }
  static __device__ __forceinline__ int piece_byte() { return 16 * ((threadIdx.x & 7) ^ ((threadIdx.x & 63) >> 3)); }
  // the same of packed weights: 16-row tile and byte
  static __device__ __forceinline__ int packed_tile(int j) { return PIECES / 2 * wave() + (j >> 1); }
  static __device__ __forceinline__ int packed_byte(int j) { return 1024 * (j & 1) + (threadIdx.x & 63) * 16; }
  // the same of columns: row of a stage, and first of 8 columns
  static __device__ __forceinline__ int column_row(int j) {
    return 1024 / LINE * (PIECES * wave() + j) + (threadIdx.x & 63) / (LINE / 16);
  }
  static __device__ __forceinline__ int column_first(int j) {
    const int row = column_row(j), chunk = threadIdx.x % (LINE / 16) >> 1;
    return 16 * (chunk ^ ((row & 3) | (row >> 3 & 1) << 2)) + 8 * (threadIdx.x & 1);
  }

  // Where an operand of a tile comes from: this lane's byte offsets of the wave's pieces from ``at`` bytes behind the base on,
  // ``step`` bytes a stage.  An offset from ``bytes`` on loads as zero.
  struct Source {
    __amdgpu_buffer_rsrc_t base;
    u32x4 words;  // of ``base``
    uint32_t off[PIECES], at, step;
    __device__ __forceinline__ void from(const void* p, uint32_t bytes, uint32_t first, uint32_t stage) {
      base = __builtin_amdgcn_make_buffer_rsrc(const_cast<void*>(p), (short)0, (int)bytes, 0x00020000);
      words = (u32x4){(uint32_t)(uintptr_t)p, (uint32_t)((uintptr_t)p >> 32) & 0xffff, bytes, 0x00020000};
      at = first, step = stage;
    }
  };

  template <bool LANES>  // (of a value that is the same in all lanes, which the compiler may not see)
  static __device__ __forceinline__ uint32_t scalar(uint32_t v) { return LANES ? __builtin_amdgcn_readfirstlane(v) : v; }

  // The workgroup's tiles 0 .. count - 1 (at least one).  ``work``:
  //   int stages(k)                  stages of tile k, at least one
  //   void row_offsets(Source&), weight_offsets(Source&)   the lane's offsets, once
  //   void rows(k, Source&)          tile k's rows (may change the offsets)
  //   void weights(k, Source&)       its weight rows
  //   FRAGS                          the fragments of a wave's rows that all tiles have (of 8: 4 to 8)
  //   bool half(k)                   where these are all: has tile k at most half of its rows?
  //   TURNS, int turn(k)             does a tile begin with another stage than its first: rows and weights are there, turn(k) stages
  //                                  stand ahead of it and come last
  //   int store<M>(k, acc)           acc[i][j]: weight rows 16 (8 wn + i) .. x rows 16 (M wm + j) .., j < M; lane: row lane % 16,
  //                                  weight rows 4 (lane / 16) .. + 3.  At least how many stores were issued: 0,
  //                                  work.STORES of M = FRAGS, half of them of a half tile.
  // Ends with no load in flight.
  template <Weights FORM, class Work>
  static __device__ __forceinline__ void run(char* smem, int count, const Work& work) {
    const int lane = threadIdx.x & 63, c16 = lane & 15, g4 = lane >> 4;
    constexpr int FRAGS = Work::FRAGS;  // loads of a wave and stage of rows, as many as fragments
    static_assert(FRAGS == MW || (SLOTS == 5 && FRAGS >= 4 && FRAGS < MW));
    Source x, w;
    int lk = 0, left = work.stages(0);  // the tile that is being loaded, its stages left
    int turn = 0;  // how many of them stand ahead of the one it begins with
    if constexpr (Work::TURNS) turn = work.turn(0);
    work.row_offsets(x);
    work.weight_offsets(w);
    work.rows(0, x);
    work.weights(0, w);
    // A load in asm has its place in m0, an operand of it that the compiler sets, and waits five states for scalars that a vector
    // instruction wrote (the compiler may keep some in lanes).  In the loop two MFMAs stand in the place of waits (five waits in
    // front of each load cost 5 % at 1554 x 4096 x 28672).
    auto place = [&](int pieces, int j, int slot) { return (lptr_t)(smem + slot * SLOT + (wave() * pieces + j) * 1024); };
    auto load = [&](const Source& s, int pieces, int j, int slot) {
      if constexpr (FORM == COLUMNS)
        asm volatile("s_nop 4\n\tbuffer_load_dwordx4 %0, %1, %2 offen lds"
                     :: "v"(s.off[j]), "s"(s.words), "s"(scalar<Work::TURNS>(s.at)), "{m0}"((uint32_t)(uintptr_t)place(pieces, j, slot)) : "memory");
      else
        __builtin_amdgcn_raw_ptr_buffer_load_lds(s.base, place(pieces, j, slot), 16, s.off[j], s.at, 0, 0);
    };
    // to the next stage (past the last tile its last stage is loaded again: nothing reads it, and the counts stay what they are)
    auto step = [&] {
      x.at += x.step, w.at += w.step;
      if (__builtin_expect(--left == 0, 0)) {
        x.at -= x.step, w.at -= w.step;
        left = 1;
        if (lk + 1 < count) {
          left = work.stages(++lk), work.rows(lk, x), work.weights(lk, w);
          if constexpr (Work::TURNS) turn = work.turn(lk);
        }
      } else if (Work::TURNS && left == turn) {
        const uint32_t n = work.stages(lk);
        x.at -= n * x.step, w.at -= n * w.step;
      }
    };
    // a row's chunk c lies at 16 (c ^ row % 8)
    const int s0 = 16 * (g4 ^ (c16 & 7)), s1 = 16 * ((4 + g4) ^ (c16 & 7));
    const int wr = FORM == PACKED    ? 2048 * NW * wn() + lane * 16
                   : FORM == COLUMNS
                       ? (8 * g4 + (c16 >> 2)) * LINE + ((32 * NW * wn()) ^ (32 * (c16 >> 2 | (g4 & 1) << 2))) + 8 * (c16 & 3)
                                     : (16 * NW * wn() + c16) * 128;
    u16x8 xa[MW], wa[NW], xb[MW], wb[NW];
    f32x4 acc[NW][MW];
    int px = 1, pw = 0;          // slots of the stage's rows and weights
    int fx, fw = 0;              // slots that the last barrier freed
    int stored = 0;              // stores in flight of the tile before: none, of 64 rows a wave, of 128
    int mode = 0;                // the rows' fragments that xa holds
    auto take1 = [&](int h, int r, int xr, u16x8(&xf)[MW], u16x8(&wf)[NW], int m) {  // one operand of a half stage
      if (r < m) {
        xf[r] = *reinterpret_cast<const u16x8*>(smem + px * SLOT + xr + (h ? s1 : s0) + r * 2048);
      } else if constexpr (FORM == COLUMNS) {
        const char* p = smem + ((pw * SLOT + wr) ^ (32 * (r - m))) + h * 32 * LINE;
        const s16x4 lo = __builtin_amdgcn_ds_read_tr16_b64_v4i16((__attribute__((address_space(3))) s16x4*)(p));
        const s16x4 hi = __builtin_amdgcn_ds_read_tr16_b64_v4i16((__attribute__((address_space(3))) s16x4*)(p + 4 * LINE));
        wf[r - m] = __builtin_bit_cast(u16x8, __builtin_shufflevector(lo, hi, 0, 1, 2, 3, 4, 5, 6, 7));
      } else {
        wf[r - m] = *reinterpret_cast<const u16x8*>(smem + pw * SLOT + wr + (FORM == PACKED ? h * 1024 : h ? s1 : s0) + (r - m) * 2048);
      }
    };
    auto tile = [&](auto fragments, int k) __attribute__((always_inline)) {
      constexpr int M = decltype(fragments)::value;  // fragments of a wave's rows
      constexpr int R = F == 4 ? 1 : M >= 6 ? 3 : 2;  // MFMAs to a read
      constexpr int TURN = 2 * NW;                     // MFMAs of two fragments of rows
      const int xr = (16 * M * wm() + c16) * 128;
      // MFMA q of a half stage: two fragments of rows at a time.  An operand that a vector instruction wrote (a cleared sum, a
      // copy at the loop's head) has to be two wait states old, which nobody counts for asm: a stage's first MFMA has them with it.
      auto weight_of = [](int q) {
        if (q >= TURN * (M / 2)) return M / 2 % 2 ? NW - 1 - q % TURN : q % TURN;  // (the last fragment of an odd number)
        const int b = q % TURN / 4, s = q % 4, down = q / TURN & 1;
        return 2 * (down ? NW / 2 - 1 - b : b) + ((s == 1 || s == 2) != down);
      };
      auto row_of = [](int q) { return q >= TURN * (M / 2) ? M - 1 : 2 * (q / TURN) + ((q % 4 >= 2) != (q % TURN / 4 & 1)); };
      auto multiply1 = [&](int q, const u16x8(&xf)[MW], const u16x8(&wf)[NW], bool first) {
        const int i = weight_of(q), j = row_of(q);
        if (first)
          asm volatile("s_nop 1\n\tv_mfma_f32_16x16x32_bf16 %0, %1, %2, %0" : "+a"(acc[i][j]) : "v"(wf[i]), "v"(xf[j]));
        else
          asm volatile("v_mfma_f32_16x16x32_bf16 %0, %1, %2, %0" : "+a"(acc[i][j]) : "v"(wf[i]), "v"(xf[j]));
      };
      // MFMAs q - 1 and q and a load in asm behind them (more wait states than a first MFMA needs)
      auto multiply2 = [&](int q, const u16x8(&xf)[MW], const u16x8(&wf)[NW], const Source& s, int pieces, int l, int slot) {
        const int i = weight_of(q - 1), j = row_of(q - 1), i1 = weight_of(q), j1 = row_of(q);
        const uint32_t to = (uint32_t)(uintptr_t)place(pieces, l, slot);
        asm volatile("s_nop 2\n\tv_mfma_f32_16x16x32_bf16 %0, %2, %3, %0\n\tv_mfma_f32_16x16x32_bf16 %1, %4, %5, %1\n\t"
                     "buffer_load_dwordx4 %6, %7, %8 offen lds"
                     : "+a"(acc[i][j]), "+a"(acc[i1][j1])
                     : "v"(wf[i]), "v"(xf[j]), "v"(wf[i1]), "v"(xf[j1]), "v"(s.off[l]), "s"(s.words), "s"(scalar<Work::TURNS>(s.at)), "{m0}"(to)
                     : "memory");
      };
      // a half stage: the products of the operands read before, reads of the next half's, the loads of a stage of one operand
      auto half_stage = [&](auto second) __attribute__((always_inline)) {
        constexpr bool B = decltype(second)::value;
#pragma unroll
        for (int q = 0; q < NW * M; ++q) {
          constexpr int AT = B || M < 4 ? 1 : M - 3;
          constexpr int LOADS = B ? FRAGS : PIECES;  // (group q / M of M MFMAs has one)
          const bool loads = q / M < LOADS;
          if (FORM == COLUMNS && loads && q % M == AT) multiply2(q, B ? xb : xa, B ? wb : wa, B ? x : w, LOADS, q / M, B ? fw : fx);
          else if (FORM != COLUMNS || !loads || q % M != AT - 1) multiply1(q, B ? xb : xa, B ? wb : wa, !B && q == 0);
          if (q % R == R - 1 && q / R < M + NW) take1(!B, q / R, xr, B ? xa : xb, B ? wa : wb, M);
          if (FORM != COLUMNS && loads && q % M == AT) load(B ? x : w, LOADS, q / M, B ? fw : fx);
          __builtin_amdgcn_sched_barrier(0);
        }
      };
      if (mode != M) {  // (read for the tile before, which had other rows)
#pragma unroll
        for (int r = 0; r < M; ++r) take1(0, r, xr, xa, wa, M);
        mode = M;
      }
#pragma unroll
      for (int i = 0; i < NW; ++i)
#pragma unroll
        for (int j = 0; j < M; ++j) acc[i][j] = (f32x4)(0.f);
      const int n = work.stages(k);
#pragma unroll 1
      for (int st = 0; st < n; ++st) {
        __builtin_amdgcn_sched_barrier(0);
        half_stage(Int<0>());
        // the next stage has landed for all waves, and all have read this one.  In flight: what is loaded of later stages (of five
        // slots the weights of the stage after the next) and the stores of the tile before
        constexpr int FLY = (SLOTS - 4) * PIECES;
        if (stored == 0) asm volatile("s_waitcnt vmcnt(%0)" ::"n"(FLY) : "memory");
        else if (stored < Work::STORES) asm volatile("s_waitcnt vmcnt(%0)" ::"n"(FLY + Work::STORES / 2) : "memory");
        else asm volatile("s_waitcnt vmcnt(%0)" ::"n"(FLY + Work::STORES) : "memory");
        stored = 0;
        asm volatile("" : "+s"(stored));  // (one loop: the compiler would make the first stage a second one)
        lds_wait_barrier();
        __builtin_amdgcn_sched_barrier(0);
        fx = px, fw = pw;
        px = px >= SLOTS - 2 ? px + 2 - SLOTS : px + 2;
        pw = pw >= SLOTS - 2 ? pw + 2 - SLOTS : pw + 2;
        half_stage(Int<1>());
        step();
      }
      asm volatile("s_nop 15\n\ts_nop 15" ::: "memory");  // (the last sums, which asm reads)
      stored = work.template store<M>(k, acc);
    };
#pragma unroll 1
    for (int s = 0; s < AHEAD; ++s) {  // w 0, x 0, w 1, x 1 ..
#pragma unroll
      for (int j = 0; j < PIECES; ++j) load(w, PIECES, j, 2 * s);
#pragma unroll
      for (int j = 0; j < FRAGS; ++j) load(x, FRAGS, j, 2 * s + 1);
      step();
    }
    fx = SLOTS - 1;  // (the next weights)
    asm volatile("s_waitcnt vmcnt(%0)" ::"n"((AHEAD - 1) * (PIECES + FRAGS)) : "memory");
    lds_wait_barrier();
#pragma unroll
    for (int r = 0; r < NW; ++r) take1(0, r, 0, xa, wa, 0);
    for (int k = 0; k < count; ++k) {
      if constexpr (FRAGS < MW) tile(Int<FRAGS>(), k);
      else if (work.half(k)) tile(Int<MW / 2>(), k);
      else tile(Int<MW>(), k);
    }
    asm volatile("s_waitcnt vmcnt(0) lgkmcnt(0)" ::: "memory");
  }

  // A sum out of the accumulation registers, where and when it is asked for: left to the compiler all 256 are moved at once,
  // more than there is room for.
  static __device__ __forceinline__ f32x4 taken(const f32x4& a) {
    f32x4 y;
#pragma unroll
    for (int r = 0; r < 4; ++r) {
      float t;
      asm volatile("v_accvgpr_read_b32 %0, %1" : "=v"(t) : "a"(a[r]));
      y[r] = t;
    }
    return y;
  }

  // Rows of ``acc`` (``run``, fragments M) to out[row][cols], ``out`` the tile's first row of ``rows``, columns from ``col`` on.
  // GLU: ``act`` makes one of each two fragments (gate, up), else of each one.  A lane holds 4 columns of a row in a fragment;
  // neighbouring fragments trade halves between the lane's rows of 16, so that a lane stores 16 bytes and an instruction 64
  // bytes of each of 16 rows (8 bytes a lane: 6421 x 12288 x 4096 506 -> 480 us with eight waves).  Rows and columns that are
  // not there are stored behind the end of the buffer, which drops them: all stores are issued.
  static constexpr int put_stores(bool glu) { return MW * NW / (glu ? 4 : 2); }
  template <bool GLU, int M, class Act>
  static __device__ __forceinline__ int put(bf16_t* out, int cols, int rows, int col, const f32x4 (&acc)[NW][MW], Act act) {
    constexpr int S = GLU ? 2 : 1;
    const int c16 = threadIdx.x & 15, g4 = (threadIdx.x & 63) >> 4, lc = col + 16 * (g4 & 1) + 8 * (g4 >> 1);
    const uint32_t at = (uint32_t)(c16 * cols + lc) * 2;
    // a buffer is 16 rows: their bytes fit 31 bits wherever a matrix of as many columns and 64 rows has fewer than 2^31 elements
    int left = rows - 16 * M * wm();
    bf16_t* p = out + (int64_t)(16 * M * wm()) * cols;
#pragma unroll
    for (int j = 0; j < M; ++j, left -= 16, p += 16 * cols) {
      const int bytes = left >= 16 ? 32 * cols : left > 0 ? 2 * left * cols : 0;  // (min and max would be made in lanes)
      const __amdgpu_buffer_rsrc_t to = __builtin_amdgcn_make_buffer_rsrc(p, (short)0, bytes, 0x00020000);
#pragma unroll
      for (int i = 0; i < NW; i += 2 * S) {
        uint32_t d[2][2];
#pragma unroll
        for (int h = 0; h < 2; ++h) {
          float y[4];
          const f32x4 v = taken(acc[i + h * S][j]);
          act(v, GLU ? taken(acc[i + h * S + S - 1][j]) : v, y);
#pragma unroll
          for (int r = 0; r < 2; ++r)
            d[h][r] = __builtin_bit_cast(uint32_t, __builtin_convertvector((f32x2){y[2 * r], y[2 * r + 1]}, bf16x2));
        }
        const u32x2 a = __builtin_bit_cast(u32x2, __builtin_amdgcn_permlane16_swap(d[0][0], d[1][0], false, false));
        const u32x2 b = __builtin_bit_cast(u32x2, __builtin_amdgcn_permlane16_swap(d[0][1], d[1][1], false, false));
        const bool there = lc + 16 * i / S < cols;  // (columns come in sixteens)
        // (all of the offset in the lane's part: the buffer's end is compared with that, less the scalar part, and may be 0)
        __builtin_amdgcn_raw_buffer_store_b128((u32x4){a[0], b[0], a[1], b[1]}, to, (there ? at : 1u << 31) + 32 * i / S, 0, 0);
        __builtin_amdgcn_sched_barrier(0);
      }
    }
    return put_stores(GLU) * M / MW;
  }
};
typedef TileLoop<8, 5> WideTile;

}  // namespace mp
