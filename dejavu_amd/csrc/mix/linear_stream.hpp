// Products of a portion's rows (16..256 per tile) with a bf16 weight on the matrix cores, with the epilogues of
// linear_rows.hpp.  The weight's bytes bound the product, not its operations.
//
// A tile is MB rows of W by NB activation rows.  Both operands go from memory straight into a ring of ST LDS slots (no
// registers on the way) ST - 1 chunks of KC columns ahead of their use: a wave's load covers 256 or 128 contiguous bytes of
// a row, where loads in the matrix instruction's own layout cover 64 (a plain read of 22016 x 4096 in these pieces: 6.0,
// 5.2 and 4.3 TB/s).  Where the tiles are fewer than the chip's workgroups, K is split over the grid and a second launch
// adds the sums up; adding them up in the first one, by the workgroup that ends last, costs more (each hand-over between
// compute dies 5 us, fences 40 us).
//
// Before, a workgroup of 32 rows read both operands in operand layout, 24 loads at a time: with 47 rows 4096 x 4096 took
// 24 us, 4096 x 11008 47 us, 22016 x 4096 74 us; now 12.5, 24.5 and 41 us (with 16 rows 13, 43, 51 -> 11, 22, 39).  Bound
// by the stream: 41 us are 4.4 TB/s beside a plain read's 6.
#pragma once
#include <type_traits>

#include "elem.hpp"
#include "stream.hpp"

namespace dv {

using TileArgs = dvTileArgs;

typedef const __attribute__((address_space(1))) void* global_ptr_t;
typedef __attribute__((address_space(3))) void* lds_ptr_t;

// Waits until at most N of this wave's loads are still on their way.
template <int N>
__device__ __forceinline__ void wait_loads() {
  asm volatile("s_waitcnt vmcnt(%0)" ::"i"(N) : "memory");
}

__device__ __forceinline__ bool aligned_to(const void* p, unsigned bytes) { return (reinterpret_cast<uintptr_t>(p) & (bytes - 1)) == 0; }

// The results of a lane: rows m .. m + 3 of W (m % 4 == 0), activation row n.
template <int AFTER>
__device__ __forceinline__ void tile_out(const TileArgs& a, int m, int n, float4_t v) {
  if (n >= a.n || m >= a.M) return;
  const bool whole = m + 3 < a.M;
  if (AFTER != DV_OUT_GLU && a.bias) {
#pragma unroll
    for (int e = 0; e < 4; ++e) v[e] += to_f(reinterpret_cast<const bf16_t*>(a.bias)[min(m + e, a.M - 1)]);
  }
  if constexpr (AFTER == DV_OUT_GLU) {
    bf16_t* o = reinterpret_cast<bf16_t*>(a.out) + (int64_t)n * a.ldo + (m >> 1);
    const bf16_t o0 = (bf16_t)glu_f(v[0], v[1], a.act, a.limit), o1 = (bf16_t)glu_f(v[2], v[3], a.act, a.limit);
    if (whole && a.ldo % 2 == 0 && aligned_to(a.out, 4)) {
      typedef bf16_t pair_t __attribute__((ext_vector_type(2)));
      *reinterpret_cast<pair_t*>(o) = pair_t{o0, o1};
    } else {
      if (m + 1 < a.M) o[0] = o0;
      if (whole) o[1] = o1;
    }
  } else if constexpr (AFTER == DV_OUT_RESIDUAL) {
    const int64_t at = (int64_t)n * a.M + m;
#pragma unroll
    for (int e = 0; e < 4; ++e)
      if (m + e < a.M) residual_apply<bf16_t>(a.res, at + e, m + e, v[e]);
  } else {
    typedef typename std::conditional<AFTER == DV_OUT_F32, float, bf16_t>::type out_t;
    out_t* o = reinterpret_cast<out_t*>(a.out) + (int64_t)n * a.ldo + m;
    if (whole && a.ldo % 4 == 0 && aligned_to(a.out, 4 * sizeof(out_t))) {
      store_quad<out_t>(o, v);
    } else {
#pragma unroll
      for (int e = 0; e < 4; ++e)
        if (m + e < a.M) o[e] = from_f<out_t>(v[e]);
    }
  }
}

// NT_W: the weight bypasses the caches (worth 10 % where the activations are few).
// Grid: (tiles of W, tiles of activation rows, splits of K).  part: with several splits, the sums [split][tile][value][thread].
template <int AFTER, int MB, int NB, int KC, int ST, int WM, int WN, bool NT_W>
__global__ __launch_bounds__(WM * WN * 64) void linear_stream_kernel(TileArgs a, float4_t* __restrict__ part) {
  extern __shared__ __attribute__((aligned(16))) unsigned char slots[];
  constexpr int WAVES = WM * WN, THREADS = WAVES * 64;
  constexpr int CH = KC / 8;               // 16-byte pieces of a row's chunk
  constexpr int RPL = 64 / CH;             // rows per load of a wave
  constexpr int SWAP = (CH < 16 ? CH : 16) - 1;
  constexpr int LI = (MB + NB) / RPL / WAVES;
  constexpr int SLOT = (MB + NB) * KC * 2;
  constexpr int RT = MB / WM / 16, NT = NB / WN / 16, KS = KC / 32;
  static_assert((MB + NB) % (RPL * WAVES) == 0 && MB % RPL == 0, "loads do not tile");
  const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int wm = wave % WM, wn = wave / WM, l16 = lane & 15, g = lane >> 4;
  const int m0 = blockIdx.x * MB, n0 = blockIdx.y * NB;
  const bf16_t* W = reinterpret_cast<const bf16_t*>(a.W);
  const bf16_t* X = reinterpret_cast<const bf16_t*>(a.x);
  const int nch = (a.K + KC - 1) / KC;
  const int c0 = nch * blockIdx.z / gridDim.z, c1 = nch * (blockIdx.z + 1) / gridDim.z;

  // A row's pieces lie in LDS at places exchanged by the row (place = piece ^ row), so that 16 rows' pieces are read
  // from different banks; the lanes fetch them in that order.
  const bf16_t* src[LI];
  int piece[LI];
#pragma unroll
  for (int i = 0; i < LI; ++i) {
    const int row = (wave * LI + i) * RPL + lane / CH;
    piece[i] = (lane % CH) ^ (row & SWAP);
    src[i] = row < MB ? W + (int64_t)min(m0 + row, a.M - 1) * a.ldw : X + (int64_t)min(n0 + row - MB, a.n - 1) * a.ldx;
  }
  const int pieces = a.K / 8;
  auto load = [&](int c, int slot) {
    // past the last piece: that one again (set to zero when it is used); past the last chunk: into a slot that is not read
#pragma unroll
    for (int i = 0; i < LI; ++i) {
      const global_ptr_t from = (global_ptr_t)(src[i] + min(c * CH + piece[i], pieces - 1) * 8);
      const lds_ptr_t to = (lds_ptr_t)(slots + slot * SLOT + (wave * LI + i) * 1024);
      if (NT_W && (wave * LI + i) * RPL < MB) __builtin_amdgcn_global_load_lds(from, to, 16, 0, 2 /* read once */);
      else __builtin_amdgcn_global_load_lds(from, to, 16, 0, 0);
    }
  };
#pragma unroll
  for (int d = 0; d < ST - 1; ++d) load(c0 + d, d);

  float4_t acc[RT][NT];
#pragma unroll
  for (int i = 0; i < RT; ++i)
#pragma unroll
    for (int j = 0; j < NT; ++j) acc[i][j] = float4_t{0.f, 0.f, 0.f, 0.f};
  int slot = 0;
  for (int c = c0; c < c1; ++c) {
    wait_loads<LI*(ST - 2)>();
    __builtin_amdgcn_s_barrier();  // everybody's part of the slot is there, and the slot before it is free
    asm volatile("" ::: "memory");
    load(c + ST - 1, slot == 0 ? ST - 1 : slot - 1);
    const unsigned char* wb = slots + slot * SLOT + (wm * RT * 16 + l16) * KC * 2;
    const unsigned char* xb = slots + slot * SLOT + (MB + wn * NT * 16 + l16) * KC * 2;
#pragma unroll
    for (int ks = 0; ks < KS; ++ks) {
      const int at = ((ks * 4 + g) ^ (l16 & SWAP)) * 16;
      uint4_t w[RT], x[NT];
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
#pragma unroll
      for (int i = 0; i < RT; ++i)
#pragma unroll
        for (int j = 0; j < NT; ++j)
          acc[i][j] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(bf16x8_t, w[i]),
                                                              __builtin_bit_cast(bf16x8_t, x[j]), acc[i][j], 0, 0, 0);
    }
    slot = slot == ST - 1 ? 0 : slot + 1;
  }
  if (gridDim.z > 1) {
    float4_t* p = part + (((int64_t)blockIdx.z * gridDim.y + blockIdx.y) * gridDim.x + blockIdx.x) * (MB * NB / 4) + threadIdx.x;
#pragma unroll
    for (int i = 0; i < RT; ++i)
#pragma unroll
      for (int j = 0; j < NT; ++j) p[(i * NT + j) * THREADS] = acc[i][j];
  } else {
#pragma unroll
    for (int i = 0; i < RT; ++i)
#pragma unroll
      for (int j = 0; j < NT; ++j)
        tile_out<AFTER>(a, m0 + (wm * RT + i) * 16 + g * 4, n0 + (wn * NT + j) * 16 + l16, acc[i][j]);
  }
  wait_loads<0>();  // no load into LDS outlives the workgroup
}

// Adds the splits' sums up, in their order.  Grid: (tiles of W, tiles of activation rows, values of a thread).
template <int AFTER, int MB, int NB, int WM, int WN>
__global__ __launch_bounds__(WM * WN * 64) void linear_stream_sum_kernel(TileArgs a, const float4_t* __restrict__ part, int splits) {
  constexpr int THREADS = WM * WN * 64, RT = MB / WM / 16, NT = NB / WN / 16;
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6, wm = wave % WM, wn = wave / WM;
  const int i = blockIdx.z / NT, j = blockIdx.z % NT;
  const int m = blockIdx.x * MB + (wm * RT + i) * 16 + (lane >> 4) * 4, n = blockIdx.y * NB + (wn * NT + j) * 16 + (lane & 15);
  if (n >= a.n || m >= a.M) return;
  const int64_t step = (int64_t)gridDim.y * gridDim.x * (MB * NB / 4);
  const float4_t* p = part + ((int64_t)blockIdx.y * gridDim.x + blockIdx.x) * (MB * NB / 4) + blockIdx.z * THREADS + threadIdx.x;
  float4_t v = p[0];
  for (int s = 1; s < splits; ++s) v += p[s * step];
  tile_out<AFTER>(a, m, n, v);
}

}  // namespace dv
