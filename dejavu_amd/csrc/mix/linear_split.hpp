// fp32 products of many rows on the bf16 matrix instructions: out(m, n) = sum_k W[m, k] x[n, k].
//
// A value is the sum of three bf16 parts, rounded one after the other (the published bf16x3 splitting: Henry, Tang and Heinecke,
// 2019), which hold all of its 24 bits (2^-8 and 2^-17 of it at most, the others).  Products of parts are exact in the instruction's
// fp32 sums; the six largest are taken, what is left out is 2^-24 of a product at most and 2^-27.5 in the root mean square.  Products of
// one size have sums of their own, in which the second and third parts stand 2^8 and 2^16 times as large: so the smallest values'
// parts are no zeros, and no sum overflows where that of the values' magnitudes would not.  What is lost is relative to each value and
// not to its row, so rows of any range are as exact as others (two fp16 parts with an exponent for a row, three quarters of this time, lose
// what lies far below the row's largest value: with one column 2^24 times as large as the others and the weight's as much smaller a row was
// 2e-5 from 64 bits, with 2^40 0.9).  Infinities and NaN are in the first parts, whose sums are the result where they are not finite;
// other results do not see them.  At the very end of the range: a weight below 2^-126 loses its last bit, and values below 2^-133
// are zeros to an infinity.
//
// The parts of x are made beforehand (split_rows_kernel); those of W in registers, by the one wave that uses them.
// Six bf16 products at 2.5 PFLOP/s are 2.6 times the fp32 instructions' 157 TFLOP/s.  500 rows by 11264 x 2048: 155 us, the library's fp32
// GEMM 197 (two fp16 parts 123); 2048 by 22016 x 4096 2112 us, 2630.  From 64 bits 2.7e-7 and 4e-7, the library 8.1e-7 and 1.15e-6.
// Bound by the matrix instructions and what stands between them: their units work in 57 % of the cycles (at 2.1 GHz) of the 176 compute
// units that have a tile of the first; wave priorities, reads further ahead, a third slot, 128 x 256 tiles and chunks of 16 columns took as
// long or longer.
#pragma once
#include "../gemm_ring.hpp"
#include "elem.hpp"

namespace dv {

// A workgroup's tile (rows of W, rows of x), columns of a chunk, LDS slots for chunks.  A wave has 32 rows of W and all of x.
constexpr int kSplitRows = 256, kSplitCols = 128, kSplitChunk = 32, kSplitThreads = 512, kSplitSlots = 2;

__device__ __forceinline__ unsigned bf16_pair(float a, float b) {
  typedef bf16_t pair_t __attribute__((ext_vector_type(2)));
  return __builtin_bit_cast(unsigned, pair_t{(bf16_t)a, (bf16_t)b});
}
// The parts of two values of x, or of the halves of two of W, a word of two bf16 each.  The first part of a finite value is finite: what
// would round to an infinity is the largest bf16 (W's halves need no such care, and all sums are half as large).
template <bool OF_W>
__device__ __forceinline__ void split_pair(float a, float b, unsigned (&part)[3]) {
  auto first = [](float v) { return OF_W || !(fabsf(v) < INFINITY) ? v : __builtin_amdgcn_fmed3f(v, -0x1.fep127f, 0x1.fep127f); };
  if (OF_W) a *= 0.5f, b *= 0.5f;
  part[0] = bf16_pair(first(a), first(b));
  a = (a - __uint_as_float(part[0] << 16)) * 256.f, b = (b - __uint_as_float(part[0] & 0xffff0000u)) * 256.f;
  part[1] = bf16_pair(a, b);
  part[2] = bf16_pair((a - __uint_as_float(part[1] << 16)) * 256.f, (b - __uint_as_float(part[1] & 0xffff0000u)) * 256.f);
}
template <bool OF_W>
__device__ __forceinline__ void split8(const float4_t& a, const float4_t& b, uint4_t (&part)[3]) {
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    unsigned p[3];
    split_pair<OF_W>(i < 2 ? a[2 * i] : b[2 * i - 4], i < 2 ? a[2 * i + 1] : b[2 * i - 3], p);
#pragma unroll
    for (int s = 0; s < 3; ++s) part[s][i] = p[s];
  }
}

struct SplitOperands {
  const float* x;
  int64_t ldx;
  const float* W;
  int64_t ldw;
  bf16_t* parts;  // of x: [chunk][part][n][columns of a chunk], zeros from K on
  int n, M, K;
  __host__ __device__ int chunks() const { return (K + kSplitChunk - 1) / kSplitChunk; }
};

constexpr int kSplitPieces = kSplitChunk / 8, kSplitPartRows = 256 / kSplitPieces;  // 16 bytes of a part's row; rows of a workgroup

// The parts of x, 1 KiB in a row of each for a wave.  Grid: chunks * (n / kSplitPartRows, rounded up), chunks first.  K % 4 == 0.
__global__ __launch_bounds__(256) void split_rows_kernel(SplitOperands a) {
  const int chunks = a.chunks(), c = blockIdx.x % chunks;
  const int64_t row = (int64_t)(blockIdx.x / chunks) * kSplitPartRows + threadIdx.x / kSplitPieces;
  if (row >= a.n) return;
  const int at = threadIdx.x % kSplitPieces * 8, k = c * kSplitChunk + at;
  const float* r = a.x + row * a.ldx + k;
  const float4_t zero = {0.f, 0.f, 0.f, 0.f};
  uint4_t part[3];
  split8<false>(k < a.K ? *reinterpret_cast<const float4_t*>(r) : zero, k + 4 < a.K ? *reinterpret_cast<const float4_t*>(r + 4) : zero, part);
#pragma unroll
  for (int s = 0; s < 3; ++s) *reinterpret_cast<uint4_t*>(a.parts + (((int64_t)c * 3 + s) * a.n + row) * kSplitChunk + at) = part[s];
}

struct SplitPlan {
  int rows, cols, splits, chunks;
  int64_t tiles() const { return (int64_t)rows * cols; }
  size_t parts_bytes(int n) const { return ((size_t)3 * n * chunks * kSplitChunk * sizeof(bf16_t) + 255) / 256 * 256; }
  size_t workspace_bytes(int n) const {
    return parts_bytes(n) + (splits > 1 ? (size_t)splits * tiles() * kSplitRows * kSplitCols * sizeof(float) : 0);
  }
};
// K is split where that takes less: a round of workgroups 2.2 us a chunk, a second launch 4, a tile's sums 0.05 (in units of these).  A split
// has at least 256 columns.
inline SplitPlan plan_split(int n, int M, int K, int units) {
  SplitPlan p;
  p.chunks = (K + kSplitChunk - 1) / kSplitChunk;
  p.rows = (M + kSplitRows - 1) / kSplitRows;
  p.cols = (n + kSplitCols - 1) / kSplitCols;
  p.splits = 1;
  int64_t least = INT64_MAX;
  for (int s = 1; s <= 8 && (s == 1 || s <= K / 256); ++s) {
    const int64_t rounds = (s * p.tiles() + units - 1) / units, cost = rounds * ((p.chunks + s - 1) / s) * 44 + (s > 1 ? 80 + s * p.tiles() : 0);
    if (cost < least) least = cost, p.splits = s;
  }
  return p;
}
constexpr size_t kSplitLds = (size_t)kSplitSlots * (kSplitRows * kSplitChunk * sizeof(float) + 3 * kSplitCols * kSplitChunk * sizeof(bf16_t));

// Grid: (tiles, those of W first; splits of K).  part: with several splits, the sums [split][tile][value][thread].
template <typename Out>
__global__ __launch_bounds__(kSplitThreads, 2) void linear_split_kernel(SplitOperands a, int row_tiles, Out out, float4_t* __restrict__ part) {
  extern __shared__ __attribute__((aligned(16))) unsigned char slots[];
  constexpr int KC = kSplitChunk, MB = kSplitRows, NB = kSplitCols, NT = NB / 32, WAVES = kSplitThreads / 64;
  constexpr int WBYTES = MB * KC * 4, PLANE = NB * KC * 2, SLOT = WBYTES + 3 * PLANE, PX = kSplitPieces, PW = KC / 4;
  constexpr int LW = WBYTES / 1024 / WAVES, LX = 3 * PLANE / 1024 / WAVES;  // a wave's loads of a chunk, 1 KiB each
  static_assert(MB == WAVES * 32 && (LW * WAVES + LX * WAVES) * 1024 == SLOT && KC == 32, "tile");
  const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int l32 = lane & 31, half = lane >> 5;
  const int m0 = blockIdx.x % row_tiles * MB, n0 = blockIdx.x / row_tiles * NB;
  const int nch = a.chunks(), c0 = nch * blockIdx.y / gridDim.y, c1 = nch * (blockIdx.y + 1) / gridDim.y;

  // A load is eight rows of W (eight pieces of 16 bytes each) or sixteen of a part of x (four pieces).  Pieces are exchanged by the row,
  // so that sixteen rows' are read from different banks.
  const float* wsrc[LW];
  const bf16_t* xsrc[LX];
  int step[LW];
#pragma unroll
  for (int i = 0; i < LW; ++i) {
    const int row = (wave * LW + i) * (64 / PW) + lane / PW;
    step[i] = (lane % PW ^ (row & 7)) * 4;
    wsrc[i] = a.W + (int64_t)min(m0 + row, a.M - 1) * a.ldw;
  }
#pragma unroll
  for (int i = 0; i < LX; ++i) {
    const int row = (wave * LX + i) * (64 / PX) + lane / PX, s = row / NB, r = row % NB;
    xsrc[i] = a.parts + ((int64_t)s * a.n + min(n0 + r, a.n - 1)) * KC + (lane % PX ^ (r >> 2 & 3)) * 8;
  }
  const int64_t xstep = (int64_t)3 * a.n * KC;
  auto load = [&](int c, int slot) {
    unsigned char* to = slots + slot * SLOT;
#pragma unroll
    for (int i = 0; i < LW; ++i)  // (past the end of a row its last piece: set to zero when it is used)
      __builtin_amdgcn_global_load_lds((global_ptr_t)(wsrc[i] + min(c * KC + step[i], a.K - 4)), (lds_ptr_t)(to + (wave * LW + i) * 1024), 16, 0, 0);
#pragma unroll
    for (int i = 0; i < LX; ++i)
      __builtin_amdgcn_global_load_lds((global_ptr_t)(xsrc[i] + c * xstep), (lds_ptr_t)(to + WBYTES + (wave * LX + i) * 1024), 16, 0, 0);
  };
  float16_t sum[3][NT];  // of products of 1, 2^-8 and 2^-16 of the values' size
#pragma unroll
  for (int s = 0; s < 3; ++s)
#pragma unroll
    for (int j = 0; j < NT; ++j)
#pragma unroll
      for (int r = 0; r < 16; ++r) sum[s][j][r] = 0.f;
  auto add = [](float16_t& acc, const uint4_t& w, const uint4_t& x) {
    acc = __builtin_amdgcn_mfma_f32_32x32x16_bf16(__builtin_bit_cast(bf16x8_t, w), __builtin_bit_cast(bf16x8_t, x), acc, 0, 0, 0);
  };
#pragma unroll
  for (int d = 0; d < kSplitSlots - 1; ++d) load(min(c0 + d, nch - 1), d);
  int slot = 0;
  for (int c = c0; c < c1; ++c, slot = slot == kSplitSlots - 1 ? 0 : slot + 1) {
    // everybody's part of the slot is there, and nobody reads the one before it any more, which is loaded next
    asm volatile("s_waitcnt vmcnt(%0) lgkmcnt(0)" ::"i"((LW + LX) * (kSplitSlots - 2)) : "memory");
    __builtin_amdgcn_s_barrier();
    asm volatile("" ::: "memory");
    load(min(c + kSplitSlots - 1, nch - 1), slot == 0 ? kSplitSlots - 1 : slot - 1);  // (past the end: into a slot that is not read)
    const unsigned char* wb = slots + slot * SLOT + (wave * 32 + l32) * KC * 4;
    const unsigned char* xb = slots + slot * SLOT + WBYTES + l32 * KC * 2;
#pragma unroll
    for (int ks = 0; ks < KC / 16; ++ks) {
      const int p = ks * 4 + half * 2;
      // (read as words: with reads as floats the compiler waits for all loads into LDS in front of them)
      uint4_t w0 = *reinterpret_cast<const uint4_t*>(wb + ((p ^ (l32 & 7)) * 16));
      uint4_t w1 = *reinterpret_cast<const uint4_t*>(wb + (((p + 1) ^ (l32 & 7)) * 16));
      if ((c + 1) * KC > a.K) {  // past the end of the rows
        if (c * KC + p * 4 >= a.K) w0 = uint4_t{0, 0, 0, 0};
        if (c * KC + p * 4 + 4 >= a.K) w1 = uint4_t{0, 0, 0, 0};
      }
      uint4_t w[3], x[3];
      split8<true>(__builtin_bit_cast(float4_t, w0), __builtin_bit_cast(float4_t, w1), w);
#pragma unroll
      for (int j = 0; j < NT; ++j) {
#pragma unroll
        for (int s = 0; s < 3; ++s)
          x[s] = *reinterpret_cast<const uint4_t*>(xb + s * PLANE + j * 32 * KC * 2 + (((ks * 2 + half) ^ (l32 >> 2 & 3)) * 16));
        add(sum[0][j], w[0], x[0]);
        add(sum[1][j], w[1], x[0]);
        add(sum[2][j], w[2], x[0]);
        add(sum[1][j], w[0], x[1]);
        add(sum[2][j], w[1], x[1]);
        add(sum[2][j], w[0], x[2]);
      }
    }
  }
  wait_loads<0>();  // no load into LDS outlives the workgroup
  float4_t* to = part + ((int64_t)blockIdx.y * gridDim.x + blockIdx.x) * (MB * NB / 4) + threadIdx.x;
#pragma unroll
  for (int j = 0; j < NT; ++j)
#pragma unroll
    for (int q = 0; q < 4; ++q) {
      float4_t v;
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        const float top = sum[0][j][4 * q + e], mid = sum[1][j][4 * q + e], low = sum[2][j][4 * q + e];
        v[e] = 2.f * (fabsf(top) < INFINITY ? __builtin_fmaf(__builtin_fmaf(low, 0x1p-8f, mid), 0x1p-8f, top) : top);
      }
      if (gridDim.y > 1) {
        to[(j * 4 + q) * kSplitThreads] = v;
      } else {
        const int m = m0 + wave * 32 + q * 8 + half * 4, n = n0 + j * 32 + l32;
        if (m < a.M && n < a.n) out(m, n, v);
      }
    }
}

// Adds the splits' sums up, in their order.  Grid: (tiles, values of a thread).
template <typename Out>
__global__ __launch_bounds__(kSplitThreads) void linear_split_sum_kernel(int rows, int M, int row_tiles, Out out, const float4_t* __restrict__ part,
                                                                         int splits) {
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6, j = blockIdx.y / 4, q = blockIdx.y % 4;
  const int m = blockIdx.x % row_tiles * kSplitRows + wave * 32 + q * 8 + (lane >> 5) * 4;
  const int n = blockIdx.x / row_tiles * kSplitCols + j * 32 + (lane & 31);
  if (n >= rows || m >= M) return;
  const int64_t step = (int64_t)gridDim.x * (kSplitRows * kSplitCols / 4);
  const float4_t* p = part + (int64_t)blockIdx.x * (kSplitRows * kSplitCols / 4) + blockIdx.y * kSplitThreads + threadIdx.x;
  float4_t v = p[0];
  for (int s = 1; s < splits; ++s) v += p[s * step];
  out(m, n, v);
}

// fp32 results with a bias, row n of x at y + n * ldy; M % 4 == 0.
struct SplitOut {
  float* y;
  int64_t ldy;
  const float* bias;
  __device__ __forceinline__ void operator()(int m, int n, float4_t v) const {
    if (bias) v += *reinterpret_cast<const float4_t*>(bias + m);
    *reinterpret_cast<float4_t*>(y + (int64_t)n * ldy + m) = v;
  }
};

}  // namespace dv
