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
// Six bf16 products at 2.5 PFLOP/s are 2.6 times the fp32 instructions' 157 TFLOP/s.  From 64 bits 2.7e-7 (K = 2048) and 4e-7 (4096), the library
// 8.1e-7 and 1.15e-6.  While W's parts of half a chunk are multiplied, the next half's are made, four instructions of that behind each
// multiplication, and x is read a step ahead, also over the barrier, so that the matrix units wait neither for the splitting nor for LDS:
// 500 rows by 11264 x 2048 180 -> 153 us (inside a prompt 170 -> 127, where the library's fp32 GEMM takes 195 with its weight cold), 2048 by 22016 x 4096 2124 -> 1773 (2580),
// 500 by 2048 x 5632 75 -> 67, 300 by 11264 x 2048 135 -> 116.  (Split beside the multiplication, but with x read where it is used: 165 and 1960.)
// Bound by power: the second was 5930 cycles a chunk at 1.89 GHz, 3072 of them the matrix units', and is 4080 at 1.64.  So the same work dealt
// out evenly to all compute units, where the first's 176 tiles leave 80 of them idle, takes as long (155 us).
#pragma once
#include "../gemm_ring.hpp"
#include "elem.hpp"

namespace dv {

// A workgroup's tile (rows of W, rows of x), columns of a chunk.  A wave has 32 rows of W and all of x.
constexpr int kSplitRows = 256, kSplitCols = 128, kSplitChunk = 32, kSplitThreads = 512;

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
constexpr int kSplitWSlots = 3, kSplitXSlots = 2;
constexpr size_t kSplitLds = (size_t)kSplitWSlots * kSplitRows * kSplitChunk * sizeof(float) + (size_t)kSplitXSlots * 3 * kSplitCols * kSplitChunk * sizeof(bf16_t);
constexpr int64_t kSplitMaxStride = 1 << 25;  // 32 rows' bytes are counted in 32 bits
constexpr int kSplitMostRows = 1 << 24;       // and those of a chunk's parts

// Grid: (tiles, those of W first; splits of K).  part: with several splits, the sums [split][tile][value][thread].
// FAR: every lane has addresses of its own, for strides and sizes beyond these two.
template <bool FAR, typename Out>
__global__ __launch_bounds__(kSplitThreads, 2) void linear_split_kernel(SplitOperands a, int row_tiles, Out out, float4_t* __restrict__ part) {
#if defined(__HIP_DEVICE_COMPILE__)  // (the loads' resources have no type on the host)
  extern __shared__ __attribute__((aligned(16))) unsigned char slots[];
  constexpr int KC = kSplitChunk, MB = kSplitRows, NB = kSplitCols, NT = NB / 32, WAVES = kSplitThreads / 64;
  constexpr int WBYTES = MB * KC * 4, PLANE = NB * KC * 2, XBYTES = 3 * PLANE, PX = kSplitPieces, PW = KC / 4;
  constexpr int LW = WBYTES / 1024 / WAVES, LX = XBYTES / 1024 / WAVES;  // a wave's loads of a chunk, 1 KiB each
  static_assert(MB == WAVES * 32 && LW * 64 / PW == 32 && LX * WAVES * 1024 == XBYTES && KC == 32 && kSplitXSlots == 2 && NT == 4 && LW <= 4, "tile");
  const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int l32 = lane & 31, half = lane >> 5;
  const int m0 = blockIdx.x % row_tiles * MB, n0 = blockIdx.x / row_tiles * NB;
  const int nch = a.chunks(), c0 = nch * blockIdx.y / gridDim.y, c1 = nch * (blockIdx.y + 1) / gridDim.y;

  // A load is eight rows of W (eight pieces of 16 bytes each) or sixteen of a part of x (four pieces).  Pieces are exchanged by the row,
  // so that sixteen rows' are read from different banks.  A wave loads the 32 rows of W that it multiplies.  What is loaded for rows past the
  // end (nothing, or other rows' values) is in results that are not stored.
  const int w_row = min(m0 + wave * 32, a.M - 1);
  const auto wr = __builtin_amdgcn_make_buffer_rsrc(const_cast<float*>(a.W) + w_row * a.ldw, 0,
                                                    (int)((unsigned)(min(32, a.M - w_row) - 1) * (unsigned)a.ldw * 4u + a.K * 4u), 0x00020000);
  const unsigned w_at = (unsigned)(lane / PW) * (unsigned)a.ldw * 4u, w_step = (unsigned)(64 / PW) * (unsigned)a.ldw * 4u;
  const int w_col = (lane % PW ^ lane / PW) * 4;
  const unsigned x_at = lane / PX * (KC * 2) + (lane % PX ^ (lane / PX >> 2 & 3)) * 16;
  auto load_w = [&](int c, int slot, int i) {  // (past the end of a row its last piece: set to zero when it is used)
    const lds_ptr_t to = (lds_ptr_t)(slots + slot * WBYTES + (wave * LW + i) * 1024);
    const int col = min(c * KC + w_col, a.K - 4);
    if constexpr (FAR) {
      const float* row = a.W + (int64_t)min(m0 + wave * 32 + i * (64 / PW) + lane / PW, a.M - 1) * a.ldw;
      __builtin_amdgcn_global_load_lds((global_ptr_t)(row + col), to, 16, 0, 0);
    } else {
      __builtin_amdgcn_raw_ptr_buffer_load_lds(wr, to, 16, w_at + (unsigned)col * 4u + i * w_step, 0, 0, 0);
    }
  };
  auto load_x = [&](int c, int slot) {
    const auto xr = __builtin_amdgcn_make_buffer_rsrc(a.parts + (int64_t)c * 3 * a.n * KC, 0, (int)((unsigned)a.n * (3u * KC * 2u)), 0x00020000);
#pragma unroll
    for (int i = 0; i < LX; ++i) {
      const int row = (wave * LX + i) * (64 / PX), s = row / NB;
      const lds_ptr_t to = (lds_ptr_t)(slots + kSplitWSlots * WBYTES + slot * XBYTES + (wave * LX + i) * 1024);
      if constexpr (FAR) {
        const int64_t at = ((int64_t)c * 3 + s) * a.n + min(n0 + row % NB + lane / PX, a.n - 1);
        __builtin_amdgcn_global_load_lds((global_ptr_t)(a.parts + at * KC + (lane % PX ^ (lane / PX >> 2 & 3)) * 8), to, 16, 0, 0);
      } else {
        __builtin_amdgcn_raw_ptr_buffer_load_lds(xr, to, 16, x_at + ((unsigned)s * a.n + n0 + row % NB) * (KC * 2u), 0, 0, 0);
      }
    }
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
  const unsigned char* wb = slots + (wave * 32 + l32) * KC * 4;
  const unsigned char* xb = slots + kSplitWSlots * WBYTES + l32 * KC * 2;
  // The eight values of W of a lane of half a chunk.  (Read as words: with reads as floats the compiler waits for all loads into LDS
  // in front of them.)
  auto read_w = [&](uint4_t (&raw)[2], int c, int slot, int ks) {
    const int p = ks * 4 + half * 2;
#pragma unroll
    for (int i = 0; i < 2; ++i) raw[i] = *reinterpret_cast<const uint4_t*>(wb + slot * WBYTES + (((p + i) ^ (l32 & 7)) * 16));
    if ((c + 1) * KC > a.K) {  // past the end of the rows
#pragma unroll
      for (int i = 0; i < 2; ++i)
        if (c * KC + p * 4 + i * 4 >= a.K) raw[i] = uint4_t{0, 0, 0, 0};
    }
  };
  auto split = [](const uint4_t (&raw)[2], uint4_t (&w)[3], int i) {
    unsigned p[3];
    split_pair<true>(__uint_as_float(raw[i / 2][i % 2 * 2]), __uint_as_float(raw[i / 2][i % 2 * 2 + 1]), p);
#pragma unroll
    for (int s = 0; s < 3; ++s) {
      asm volatile("" : "+v"(p[s]));  // made here, not where it is used
      w[s][i] = p[s];
    }
  };
  auto read_x = [&](uint4_t (&x)[3], int slot, int ks, int j) {
#pragma unroll
    for (int s = 0; s < 3; ++s)
      x[s] = *reinterpret_cast<const uint4_t*>(xb + slot * XBYTES + s * PLANE + j * 32 * KC * 2 + (((ks * 2 + half) ^ (l32 >> 2 & 3)) * 16));
  };
  if (c0 < c1) {
    const int last = nch - 1;  // (past it: that chunk again, into slots that are not read)
    uint4_t raw[2], w[2][3], x[2][3];
#pragma unroll
    for (int i = 0; i < LW; ++i) load_w(c0, 0, i);
    load_x(c0, 0);
#pragma unroll
    for (int i = 0; i < LW; ++i) load_w(min(c0 + 1, last), 1, i);
    load_x(min(c0 + 1, last), 1);
    asm volatile("s_waitcnt vmcnt(%0)" ::"i"(LW + LX) : "memory");
    __builtin_amdgcn_s_barrier();
    asm volatile("" ::: "memory");
    read_w(raw, c0, 0, 0);
    read_x(x[0], 0, 0, 0);
#pragma unroll
    for (int i = 0; i < 4; ++i) split(raw, w[0], i);
    int slot = 0, x_slot = 0;
    for (int c = c0; c < c1; ++c) {
      const int after = slot == kSplitWSlots - 1 ? 0 : slot + 1, free_slot = slot == 0 ? kSplitWSlots - 1 : slot - 1;
      // Eight steps: 32 rows of x by half of the columns.  While one is multiplied, x of the next is read and a pair of W's values of the
      // next half is taken apart.
#pragma unroll
      for (int g = 0; g < 8; ++g) {
        const int ks = g / 4, j = g % 4;
        if (g == 0) read_w(raw, c, slot, 1);
        if (g == 4) {
          asm volatile("s_waitcnt vmcnt(%0)" ::"i"(LW + LX) : "memory");  // the next chunk's W
          read_w(raw, min(c + 1, last), after, 0);
        }
        if (g == 7) {  // everybody's part of the next chunk's x is there (what was loaded behind it is W), and nobody reads this one's any more
          asm volatile("s_waitcnt vmcnt(%0) lgkmcnt(0)" ::"i"(LW) : "memory");
          __builtin_amdgcn_s_barrier();
          asm volatile("" ::: "memory");
          load_x(min(c + 2, last), x_slot);
        }
        if (g < LW) load_w(min(c + 2, last), free_slot, g);
        read_x(x[(g + 1) & 1], x_slot ^ (g == 7), (g + 1) / 4 & 1, (g + 1) % 4);
        const uint4_t(&v)[3] = x[g & 1];
        add(sum[2][j], w[ks][2], v[0]);
        add(sum[0][j], w[ks][0], v[0]);
        add(sum[1][j], w[ks][1], v[0]);
        add(sum[2][j], w[ks][1], v[1]);
        add(sum[1][j], w[ks][0], v[1]);
        add(sum[2][j], w[ks][0], v[2]);
        split(raw, w[ks ^ 1], j);
#pragma unroll
        for (int i = 0; i < 6; ++i) {  // four of the splitting's instructions behind each multiplication
          __builtin_amdgcn_sched_group_barrier(8, 1, 0);
          __builtin_amdgcn_sched_group_barrier(2, 4, 0);
        }
        __builtin_amdgcn_sched_barrier(0);
      }
      slot = after, x_slot ^= 1;
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
#endif
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
