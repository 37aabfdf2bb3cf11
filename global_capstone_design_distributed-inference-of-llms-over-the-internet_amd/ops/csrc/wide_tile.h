// Main loop of the 256 x 256 product tiles (moe.hip: experts, gemm_prompt.hip: prompts): eight waves of 64 rows x 128 weight
// rows, 64 columns a stage in two LDS slots of 64 KiB.
//   * Rows arrive 128 bytes at a time (8 rows an instruction), whole cache lines: 32-column stages fetch every line twice,
//     and 256 rows of lines are the whole L1, so the second half came from L2 again.  The 16-byte chunks of a row are
//     permuted by its low bits on the way in, which leaves the operand reads free of bank conflicts (none counted).
//     Weights come the same way, or packed in fragment order ([N / 16, K / 32, 64, 8]) as they lie.
//   * The operands of a half stage are read from LDS while the MFMAs of the half before it run, across the one barrier a
//     stage has: behind it the other slot has landed for all waves and this one is free.  The loads of the next stage but
//     one are spread over the half stage behind the barrier: eight at once hold up the MFMAs that stand behind them.
//   * A wave whose 64 rows are past the last only loads; the two waves of a SIMD have different rows, so a tile of up to 128
//     rows takes half the time.
// Bound by MFMA issue and, in part, by waits for the next stage.  Measured and left: four waves of 128 x 128 (the same time
// where the tiles are full, 5-10 % more elsewhere; LDS is a quarter busy either way), a second barrier that frees the slot
// sooner (6 % more), loads behind the reads (6 % more), lines of later
// stages brought into L2 ahead (no change), 32 x 32 x 16 MFMAs (12 % more).
#pragma once
#include <type_traits>

#include "common.h"

namespace mp {

struct WideTile {
  static constexpr int BM = 256, BN = 256, MW = 4, NW = 8, WM = 4, WN = 2, XB = BM * 128, SLOT = XB + BN * 128, LDS = 2 * SLOT;
  typedef __attribute__((ext_vector_type(8))) __bf16 bf16x8;
  typedef __attribute__((address_space(3))) void* lptr_t;
  typedef __attribute__((address_space(1))) const void* gptr_t;

  static __device__ __forceinline__ int wave() { return __builtin_amdgcn_readfirstlane(threadIdx.x >> 6); }
  static __device__ __forceinline__ int wm() { return wave() / WN; }  // (the waves of a SIMD, 4 apart, have different rows)
  static __device__ __forceinline__ int wn() { return wave() % WN; }
  // row of the tile that piece j of this wave reads on this lane, and the byte of it in a stage
  static __device__ __forceinline__ int piece_row(int j) { return 8 * (4 * wave() + j) + ((threadIdx.x & 63) >> 3); }
  static __device__ __forceinline__ int piece_byte() { return 16 * ((threadIdx.x & 7) ^ ((threadIdx.x & 63) >> 3)); }
  // the same of packed weights: 16-row tile and byte
  static __device__ __forceinline__ int packed_tile(int j) { return 2 * wave() + (j >> 1); }
  static __device__ __forceinline__ int packed_byte(int j) { return 1024 * (j & 1) + (threadIdx.x & 63) * 16; }

  // acc[i][j] += weight rows 16 (8 wn + i) .. x rows 16 (4 wm + j) .., over ``ks`` stages from ``x`` and ``w`` on; lane: row
  // lane % 16, weight rows 4 (lane / 16) .. + 3.  xo, wo: byte offsets of the wave's pieces.  Starts and ends with LDS
  // that other waves may still read.
  template <bool PACKED>
  static __device__ __forceinline__ void run(char* smem, const char* x, const char* w, const uint32_t (&xo)[4],
                                             const uint32_t (&wo)[4], int ks, bool live, f32x4 (&acc)[NW][MW]) {
    constexpr int WSTEP = PACKED ? 2048 : 128;
    const int lane = threadIdx.x & 63, c16 = lane & 15, g4 = lane >> 4, wv = wave();
    auto issue1 = [&](int st, int j) {  // one of this wave's pieces of stage st
      char* b = smem + (st & 1) * SLOT + wv * 4096;
      if (j < 4)
        __builtin_amdgcn_global_load_lds((gptr_t)(x + (int64_t)st * 128 + xo[j]), (lptr_t)(b + j * 1024), 16, 0, 0);
      else
        __builtin_amdgcn_global_load_lds((gptr_t)(w + (int64_t)st * WSTEP + wo[j - 4]), (lptr_t)(b + XB + (j - 4) * 1024), 16, 0,
                                         0);
    };
    auto issue = [&](int st) {
#pragma unroll
      for (int j = 0; j < 8; ++j) issue1(st, j);
    };
    // a row's chunk c lies at 16 (c ^ row % 8)
    const int s0 = 16 * (g4 ^ (c16 & 7)), s1 = 16 * ((4 + g4) ^ (c16 & 7));
    const int xr0 = (16 * MW * wm() + c16) * 128, wr0 = XB + (PACKED ? 2 * NW * wn() * 1024 + lane * 16 : (16 * NW * wn() + c16) * 128);
    u16x8 xa[MW], wa[NW], xb[MW], wb[NW];
    auto take1 = [&](int st, int h, int r, u16x8(&xr)[MW], u16x8(&wr)[NW]) {  // one operand of a half stage
      const char* b = smem + (st & 1) * SLOT;
      if (r < MW) xr[r] = *reinterpret_cast<const u16x8*>(b + xr0 + (h ? s1 : s0) + r * 2048);
      else if (PACKED) wr[r - MW] = *reinterpret_cast<const u16x8*>(b + wr0 + (2 * (r - MW) + h) * 1024);
      else wr[r - MW] = *reinterpret_cast<const u16x8*>(b + wr0 + (h ? s1 : s0) + (r - MW) * 2048);
    };
    auto multiply = [&](const u16x8(&xr)[MW], const u16x8(&wr)[NW]) {
#pragma unroll
      for (int i = 0; i < NW; ++i)
#pragma unroll
        for (int j = 0; j < MW; ++j)
          acc[i][j] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(bf16x8, wr[i]), __builtin_bit_cast(bf16x8, xr[j]),
                                                              acc[i][j], 0, 0, 0);
    };
    // the order inside a half stage, in eighths: 4 MFMAs, 1 or 2 of the 12 reads, 1 load.  Without the fences the compiler
    // moves the MFMAs behind the barrier and the reads stand alone.
    auto half = [&](auto reads, auto loads) {
      constexpr bool R = decltype(reads)::value, L = decltype(loads)::value;
#pragma unroll
      for (int i = 0; i < NW; ++i) {
        if constexpr (L) __builtin_amdgcn_sched_group_barrier(0x010, 1, 0);
        if constexpr (R) {
          __builtin_amdgcn_sched_group_barrier(0x008, 1, 0);
          __builtin_amdgcn_sched_group_barrier(0x100, 1, 0);
          __builtin_amdgcn_sched_group_barrier(0x008, 1, 0);
          if (i & 1) __builtin_amdgcn_sched_group_barrier(0x100, 1, 0);
          __builtin_amdgcn_sched_group_barrier(0x008, 2, 0);
        } else {
          __builtin_amdgcn_sched_group_barrier(0x008, 4, 0);
        }
      }
      __builtin_amdgcn_sched_barrier(0);
    };
    auto stage = [&](int st, auto next, auto load) {
      __builtin_amdgcn_sched_barrier(0);
#pragma unroll
      for (int r = 0; r < MW + NW; ++r) take1(st, 1, r, xb, wb);
      multiply(xa, wa);
      half(std::true_type{}, std::false_type{});
      if constexpr (decltype(next)::value) {
        asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
        lds_wait_barrier();  // stage st + 1 has landed for all waves, and all have read stage st
        __builtin_amdgcn_sched_barrier(0);
#pragma unroll
        for (int i = 0; i < NW; ++i) {  // (loads write LDS: the compiler keeps the order of loads and reads)
          if constexpr (decltype(load)::value) issue1(st + 2, i);
#pragma unroll
          for (int r = i * 12 / NW; r < (i + 1) * 12 / NW; ++r) take1(st + 1, 0, r, xa, wa);
        }
      }
      multiply(xb, wb);
      half(next, load);
    };
    __syncthreads();
    issue(0);
    if (ks > 1) issue(1);
    if (ks > 1) asm volatile("s_waitcnt vmcnt(8)" ::: "memory");
    else asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
    lds_wait_barrier();
    if (!live) {
      for (int st = 0; st + 1 < ks; ++st) {
        asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
        lds_wait_barrier();
        if (st + 2 < ks) issue(st + 2);
      }
      return;
    }
#pragma unroll
    for (int r = 0; r < MW + NW; ++r) take1(0, 0, r, xa, wa);
    int st = 0;
    for (; st + 2 < ks; ++st) stage(st, std::true_type{}, std::true_type{});
    if (st + 1 < ks) stage(st++, std::true_type{}, std::false_type{});
    stage(st, std::false_type{}, std::false_type{});
  }
};

}  // namespace mp
