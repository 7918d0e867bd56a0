// Products of a long prompt's rows with a bf16 weight where the operations bound them: 256 x 256 tiles, one workgroup of
// eight waves per compute unit, with the epilogues of linear_rows.hpp.
//
// The two waves of a SIMD take turns (a published schedule): in every interval between two barriers one of them multiplies
// (32 matrix instructions, 512 cycles) while the other reads its next operands from LDS, so the matrix unit does not wait for
// LDS and the LDS is read by half of the waves at a time.  Chunks of 64 columns go from memory straight into one of two LDS
// slots while the other one is in use.
//
// 2048 rows by 22016 x 4096: 308-325 us (1.2 PFLOP/s) with or without the gated unit; all eight waves in step 339; four
// waves of 128 x 128 that read ahead in registers 455; matrix instructions of 32 x 32 338.  1999 rows by 18560 x 4096: 295 us.
// The matrix units work in 51 % of its cycles, 57 % of those of full rounds (688 tiles on 256 compute units are three rounds of
// which the last is 69 % full): bound by the turns, whose reads, arriving chunks and barriers take longer than the 512 cycles of
// the other wave; not by memory (0.7 GB fetched), and LDS has no conflicts.
#pragma once
#include "linear_stream.hpp"

namespace dv {

constexpr int kWideTile = 256, kWideChunk = 64;
constexpr size_t kWideLds = (size_t)2 * 2 * kWideTile * kWideChunk * sizeof(bf16_t);

// Grid: row_tiles * col_tiles (rows of W, activation rows).
template <int AFTER>
__global__ __launch_bounds__(512, 2) void linear_wide_kernel(TileArgs a, int row_tiles, int col_tiles) {
  extern __shared__ __attribute__((aligned(16))) unsigned char slots[];
  constexpr int KC = kWideChunk, CH = KC / 8, RPL = 64 / CH, LI = 2 * kWideTile / RPL / 8, SLOT = 2 * kWideTile * KC * 2;
  constexpr int RT = 8, NT = 4, KS = KC / 32;
  const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int wm = wave & 1, wn = wave >> 1, l16 = lane & 15, g = lane >> 4;
  // Consecutive workgroups go round the eight compute dies: each die is given a stretch of the tiles, taken in blocks of
  // eight row tiles by all columns, so that its L2 serves an operand's later uses.
  int bm, bn;
  {
    const int tiles = row_tiles * col_tiles, die = blockIdx.x & 7, k = blockIdx.x >> 3;
    const int id = die * (tiles >> 3) + min(die, tiles & 7) + k;
    const int block = id / (8 * col_tiles), at = id - block * 8 * col_tiles, tall = min(8, row_tiles - block * 8);
    bm = block * 8 + at % tall;
    bn = at / tall;
  }
  const int m0 = bm * kWideTile, n0 = bn * kWideTile;
  const bf16_t* W = reinterpret_cast<const bf16_t*>(a.W);
  const bf16_t* X = reinterpret_cast<const bf16_t*>(a.x);
  const int nch = (a.K + KC - 1) / KC, pieces = a.K / 8;

  // loads and places in LDS as in gemm_ring_kernel
  const bf16_t* src[LI];
  int piece[LI];
#pragma unroll
  for (int i = 0; i < LI; ++i) {
    const int row = (wave * LI + i) * RPL + lane / CH;
    piece[i] = (lane % CH) ^ (row & (CH - 1));
    src[i] = row < kWideTile ? W + (int64_t)min(m0 + row, a.M - 1) * a.ldw : X + (int64_t)min(n0 + row - kWideTile, a.n - 1) * a.ldx;
  }
  auto load = [&](int c, int slot) {
#pragma unroll
    for (int i = 0; i < LI; ++i)
      __builtin_amdgcn_global_load_lds((global_ptr_t)(src[i] + min(c * CH + piece[i], pieces - 1) * 8),
                                       (lds_ptr_t)(slots + slot * SLOT + (wave * LI + i) * 1024), 16, 0, 0);
  };
  uint4_t w[RT], x[NT];
  float4_t acc[RT][NT];
#pragma unroll
  for (int i = 0; i < RT; ++i)
#pragma unroll
    for (int j = 0; j < NT; ++j) acc[i][j] = float4_t{0.f, 0.f, 0.f, 0.f};
  auto fetch = [&](int c, int slot, int ks) {
    const unsigned char* wb = slots + slot * SLOT + (wm * RT * 16 + l16) * KC * 2;
    const unsigned char* xb = slots + slot * SLOT + (kWideTile + wn * NT * 16 + l16) * KC * 2;
    const int at = ((ks * 4 + g) ^ (l16 & (CH - 1))) * 16;
#pragma unroll
    for (int i = 0; i < RT; ++i) w[i] = *reinterpret_cast<const uint4_t*>(wb + i * 16 * KC * 2 + at);
#pragma unroll
    for (int j = 0; j < NT; ++j) x[j] = *reinterpret_cast<const uint4_t*>(xb + j * 16 * KC * 2 + at);
    if ((c + 1) * CH > pieces && c * CH + ks * 4 + g >= pieces) {  // past the end of the rows
#pragma unroll
      for (int i = 0; i < RT; ++i) w[i] = uint4_t{0, 0, 0, 0};
#pragma unroll
      for (int j = 0; j < NT; ++j) x[j] = uint4_t{0, 0, 0, 0};
    }
  };
  auto multiply = [&]() {
    __builtin_amdgcn_s_setprio(1);
#pragma unroll
    for (int i = 0; i < RT; ++i)
#pragma unroll
      for (int j = 0; j < NT; ++j)
        acc[i][j] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(bf16x8_t, w[i]), __builtin_bit_cast(bf16x8_t, x[j]),
                                                            acc[i][j], 0, 0, 0);
    __builtin_amdgcn_s_setprio(0);
  };
  auto turn = [&]() {
    __builtin_amdgcn_sched_barrier(0);
    asm volatile("" ::: "memory");
    __builtin_amdgcn_s_barrier();
    asm volatile("" ::: "memory");
    __builtin_amdgcn_sched_barrier(0);
  };
  const bool second = wave >= 4;  // of the two waves of its SIMD; it runs one interval behind
  load(0, 0);
  wait_loads<0>();
  turn();
  if (second) turn();
  for (int c = 0; c < nch; ++c) {
    const int slot = c & 1;
#pragma unroll
    for (int ks = 0; ks < KS; ++ks) {
      fetch(c, slot, ks);
      // the other slot: its last readers are done since the turn before (past the last chunk: that one, never read)
      if (ks == 0) load(min(c + 1, nch - 1), slot ^ 1);
      asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
      __builtin_amdgcn_sched_barrier(0);
      // everybody's part of the next chunk has to be there by the turn at which the first waves begin to read it
      if (ks == KS - 1 && second) wait_loads<0>();
      turn();
      multiply();
      if (ks == KS - 1 && !second) wait_loads<0>();
      turn();
    }
  }
  if (!second) turn();
#pragma unroll
  for (int i = 0; i < RT; ++i)
#pragma unroll
    for (int j = 0; j < NT; ++j) {
      const int m = m0 + (wm * RT + i) * 16 + g * 4, n = n0 + (wn * NT + j) * 16 + l16;
      if (m < a.M && n < a.n) tile_out<AFTER>(a, m, n, acc[i][j]);
    }
}

}  // namespace dv
