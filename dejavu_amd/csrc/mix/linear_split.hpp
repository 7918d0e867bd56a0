// fp32 products of many rows on the fp16 matrix instructions: out(m, n) = sum_k W[m, k] x[n, k].
//
// Every row is scaled by a power of two that brings its largest value to 2^14 .. 2^15; a value then is the sum of two fp16 parts,
// rounded one after the other (an error of up to 2^-24 of it, or 2^-39 of the largest), a product the three products of parts
// above 2^-24 of it.  Products of fp16 are exact in the instruction's fp32 sums; those of the large parts and the small ones are
// kept apart.  The parts of x are made beforehand, with the rows' exponents (split_rows_kernel); those of W in registers, by the waves
// that use them.  What a row's exponent cannot hold (infinities, NaN, rows below 2^-100) makes a tile's results infinite or NaN, and such
// tiles are computed again from the values themselves, in fp32.
//
// Three fp16 products at 2.5 PFLOP/s are five times the fp32 instructions' 157 TFLOP/s.  500 rows by 11264 x 2048: 131 us, of which the
// exponents take 18 (they read the weight a first time) and what a compute unit fetches (48 KB a chunk, 40 bytes a ns) 73; the
// library's fp32 GEMM 228.  2048 rows by 22016 x 4096 1392 us, 2624.  From 64 bits 3.0e-7 and 4.1e-7, the library 8.1e-7 and 1.15e-6 (its sums
// run over more columns).  Six products of three bf16 parts, which need no exponents, took 211 us for the first.
#pragma once
#include "../gemm_ring.hpp"
#include "elem.hpp"

namespace dv {

constexpr int kSplitRows = 128, kSplitChunk = 32, kSplitThreads = 512, kSplitSlots = 3;
typedef float float16_t __attribute__((ext_vector_type(16)));

// The parts of two scaled values, each a word of two fp16.
__device__ __forceinline__ void split_pair(float a, float b, float scale, unsigned& h, unsigned& l) {
  typedef half_t half2_t __attribute__((ext_vector_type(2)));
  const half2_t high = {(half_t)(a * scale), (half_t)(b * scale)};
  const half2_t low = {(half_t)__builtin_fmaf(a, scale, -(float)high[0]), (half_t)__builtin_fmaf(b, scale, -(float)high[1])};
  h = __builtin_bit_cast(unsigned, high);
  l = __builtin_bit_cast(unsigned, low);
}
__device__ __forceinline__ void split8(const float4_t& a, const float4_t& b, float scale, uint4_t& h, uint4_t& l) {
  unsigned t[2][4];
#pragma unroll
  for (int i = 0; i < 2; ++i) {
    split_pair(a[2 * i], a[2 * i + 1], scale, t[0][i], t[1][i]);
    split_pair(b[2 * i], b[2 * i + 1], scale, t[0][2 + i], t[1][2 + i]);
  }
  h = uint4_t{t[0][0], t[0][1], t[0][2], t[0][3]};
  l = uint4_t{t[1][0], t[1][1], t[1][2], t[1][3]};
}

// The exponent of a row's scale from the bits of its largest magnitude; of rows that have none, one that makes everything infinite.
__device__ __forceinline__ int row_exponent(unsigned top) {
  const int e = (int)(top >> 23) - 127;
  return top == 0u ? 0 : e > 127 || e < -100 ? 1000 : 14 - e;
}

inline int split_columns(int K) { return (K + kSplitChunk - 1) / kSplitChunk * kSplitChunk; }

struct SplitOperands {
  const float* x;
  int64_t ldx;
  const float* W;
  int64_t ldw;
  half_t* parts;     // of x: [part][n][KP], zeros from K on
  int *x_exp, *w_exp;
  int n, M, K, KP;
};

// Exponents of the rows, a wave to a row, and the parts of x.  Grid: (n + M + 3) / 4.  K % 4 == 0.
__global__ __launch_bounds__(256) void split_rows_kernel(SplitOperands a) {
  const int lane = threadIdx.x & 63, row = blockIdx.x * 4 + (threadIdx.x >> 6);
  if (row >= a.n + a.M) return;
  const bool of_x = row < a.n;
  const float* r = of_x ? a.x + (int64_t)row * a.ldx : a.W + (int64_t)(row - a.n) * a.ldw;
  constexpr int U = 8;  // loads on their way together
  unsigned top = 0u;
  for (int k = lane * 4; k < a.K; k += U * 256) {
    float4_t v[U];
#pragma unroll
    for (int u = 0; u < U; ++u) v[u] = *reinterpret_cast<const float4_t*>(r + min(k + u * 256, a.K - 4));
#pragma unroll
    for (int u = 0; u < U; ++u)
#pragma unroll
      for (int e = 0; e < 4; ++e) top = max(top, __float_as_uint(v[u][e]) & 0x7fffffffu);
  }
#pragma unroll
  for (int off = 32; off > 0; off >>= 1) top = max(top, (unsigned)__shfl_xor((int)top, off, kWave));
  const int e = row_exponent(top);
  if (lane == 0) (of_x ? a.x_exp + row : a.w_exp + (row - a.n))[0] = e;
  if (!of_x) return;
  const float scale = ldexpf(1.f, e);
  const float4_t zero = {0.f, 0.f, 0.f, 0.f};
  for (int k = lane * 8; k < a.KP; k += 512) {
    uint4_t h, l;
    split8(k < a.K ? *reinterpret_cast<const float4_t*>(r + k) : zero, k + 4 < a.K ? *reinterpret_cast<const float4_t*>(r + k + 4) : zero, scale, h,
           l);
    *reinterpret_cast<uint4_t*>(a.parts + (int64_t)row * a.KP + k) = h;
    *reinterpret_cast<uint4_t*>(a.parts + ((int64_t)a.n + row) * a.KP + k) = l;
  }
}

struct SplitPlan {
  int nb, rows, cols, splits, KP;
  size_t parts_bytes(int n) const { return ((size_t)2 * n * KP * sizeof(half_t) + 255) / 256 * 256; }
  size_t sums_offset(int n, int M) const { return parts_bytes(n) + ((size_t)(n + M) * sizeof(int) + 255) / 256 * 256; }
  size_t workspace_bytes(int n, int M) const {
    return sums_offset(n, M) + (splits > 1 ? (size_t)splits * rows * cols * kSplitRows * nb * sizeof(float) : 0);
  }
};
// K is split while the workgroups are no more than the compute units; a split has at least 256 columns.
inline SplitPlan plan_split(int n, int M, int K, int units) {
  SplitPlan p;
  p.KP = split_columns(K);
  p.nb = n <= 128 ? 128 : 256;
  p.rows = (M + kSplitRows - 1) / kSplitRows;
  p.cols = (n + p.nb - 1) / p.nb;
  int64_t s = units / ((int64_t)p.rows * p.cols);
  if (s > K / 256) s = K / 256;
  p.splits = (int)(s < 1 ? 1 : s > 8 ? 8 : s);
  return p;
}
constexpr size_t split_lds(int nb) { return (size_t)kSplitSlots * (kSplitRows * kSplitChunk * 4 + 2 * nb * kSplitChunk * 2); }

// Grid: (tiles of W, tiles of x, splits of K).  part: with several splits, the sums [split][tile][value][thread].
template <int NB, typename Out>
__global__ __launch_bounds__(kSplitThreads, 2) void linear_split_kernel(SplitOperands a, Out out, float4_t* __restrict__ part) {
  extern __shared__ __attribute__((aligned(16))) unsigned char slots[];
  __shared__ int again;
  constexpr int KC = kSplitChunk, WBYTES = kSplitRows * KC * 4, PLANE = NB * KC * 2, SLOT = WBYTES + 2 * PLANE;
  constexpr int WL = kSplitRows / 8, LOADS = WL + 2 * NB / 16, LI = LOADS / 8, NT = NB / 64;
  static_assert(LOADS % 8 == 0, "loads do not tile");
  const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int wm = wave & 3, wn = wave >> 2, l32 = lane & 31, half = lane >> 5;
  const int m0 = blockIdx.x * kSplitRows, n0 = blockIdx.y * NB;
  const int nch = a.KP / KC, c0 = nch * blockIdx.z / gridDim.z, c1 = nch * (blockIdx.z + 1) / gridDim.z;
  if (threadIdx.x == 0) again = 0;
  const float scale = ldexpf(1.f, a.w_exp[min(m0 + wm * 32 + l32, a.M - 1)]);

  // Loads of 1 KiB: eight rows of W (eight pieces of 16 bytes each) or sixteen of a part of x (four pieces).  Pieces are exchanged
  // by the row, so that sixteen rows' are read from different banks.
  const unsigned char* src[LI];
  int step[LI], last[LI];
#pragma unroll
  for (int i = 0; i < LI; ++i) {
    const int load = wave * LI + i;
    if (load < WL) {
      const int row = load * 8 + lane / 8, piece = lane % 8 ^ (row & 7);
      src[i] = reinterpret_cast<const unsigned char*>(a.W + (int64_t)min(m0 + row, a.M - 1) * a.ldw);
      step[i] = piece, last[i] = a.K / 4 - 1;  // (past the end of a row its last piece: the parts of x are zero there)
    } else {
      const int row = (load - WL) * 16 + lane / 4, s = row / NB, r = row % NB, piece = lane % 4 ^ (r >> 2 & 3);
      src[i] = reinterpret_cast<const unsigned char*>(a.parts + ((int64_t)s * a.n + min(n0 + r, a.n - 1)) * a.KP);
      step[i] = piece, last[i] = a.KP / 8 - 1;
    }
  }
  auto load = [&](int c, int slot) {
#pragma unroll
    for (int i = 0; i < LI; ++i) {
      const int at = min(c * (wave * LI + i < WL ? 8 : 4) + step[i], last[i]);
      __builtin_amdgcn_global_load_lds((global_ptr_t)(src[i] + (int64_t)at * 16), (lds_ptr_t)(slots + slot * SLOT + (wave * LI + i) * 1024), 16,
                                       0, 0);
    }
  };
  float16_t large[NT], small[NT];
#pragma unroll
  for (int j = 0; j < NT; ++j)
#pragma unroll
    for (int r = 0; r < 16; ++r) large[j][r] = small[j][r] = 0.f;
  auto mfma = [](const uint4_t& w, const uint4_t& x, float16_t acc) {
    return __builtin_amdgcn_mfma_f32_32x32x16_f16(__builtin_bit_cast(half8_t, w), __builtin_bit_cast(half8_t, x), acc, 0, 0, 0);
  };
#pragma unroll
  for (int d = 0; d < kSplitSlots - 1; ++d) load(min(c0 + d, nch - 1), d);
  int slot = 0;
  for (int c = c0; c < c1; ++c, slot = slot == kSplitSlots - 1 ? 0 : slot + 1) {
    // everybody's part of the slot is there, and nobody reads the one before it any more, which is loaded next
    asm volatile("s_waitcnt vmcnt(%0) lgkmcnt(0)" ::"i"(LI * (kSplitSlots - 2)) : "memory");
    __builtin_amdgcn_s_barrier();
    asm volatile("" ::: "memory");
    load(min(c + kSplitSlots - 1, nch - 1), slot == 0 ? kSplitSlots - 1 : slot - 1);  // (past the end: into a slot that is not read)
    const unsigned char* wb = slots + slot * SLOT + (wm * 32 + l32) * KC * 4;
    const unsigned char* xb = slots + slot * SLOT + WBYTES + (wn * NT * 32 + l32) * KC * 2;
#pragma unroll
    for (int ks = 0; ks < KC / 16; ++ks) {
      const int p = ks * 4 + half * 2;
      uint4_t wh, wl, x[2][NT];
#pragma unroll
      for (int s = 0; s < 2; ++s)
#pragma unroll
        for (int j = 0; j < NT; ++j)
          x[s][j] = *reinterpret_cast<const uint4_t*>(xb + s * PLANE + j * 32 * KC * 2 + (((ks * 2 + half) ^ (l32 >> 2 & 3)) * 16));
      // (read as words: with reads as floats the compiler waits for all loads into LDS in front of them)
      const uint4_t w0 = *reinterpret_cast<const uint4_t*>(wb + ((p ^ (l32 & 7)) * 16));
      const uint4_t w1 = *reinterpret_cast<const uint4_t*>(wb + (((p + 1) ^ (l32 & 7)) * 16));
      split8(__builtin_bit_cast(float4_t, w0), __builtin_bit_cast(float4_t, w1), scale, wh, wl);
#pragma unroll
      for (int j = 0; j < NT; ++j) large[j] = mfma(wh, x[0][j], large[j]);
#pragma unroll
      for (int j = 0; j < NT; ++j) small[j] = mfma(wl, x[0][j], small[j]);
#pragma unroll
      for (int j = 0; j < NT; ++j) small[j] = mfma(wh, x[1][j], small[j]);
    }
  }
  wait_loads<0>();
  // value q of tile j: rows m .. m + 3, row n of x
  auto place = [&](int j, int q, int& m, int& n) {
    m = m0 + wm * 32 + q * 8 + half * 4;
    n = n0 + (wn * NT + j) * 32 + l32;
  };
  bool odd = false;
#pragma unroll
  for (int j = 0; j < NT; ++j) {
    large[j] += small[j];
    const int xe = a.x_exp[min(n0 + (wn * NT + j) * 32 + l32, a.n - 1)];
#pragma unroll
    for (int r = 0; r < 16; ++r) {
      int m, n;
      place(j, r / 4, m, n);
      odd |= !(fabsf(large[j][r]) < INFINITY);
      large[j][r] = ldexpf(large[j][r], -xe - a.w_exp[min(m + r % 4, a.M - 1)]);
    }
  }
  __syncthreads();  // (the last reads of the slots, and of `again`)
  if (odd) again = 1;
  __syncthreads();
  if (again) {
    float* mine = reinterpret_cast<float*>(slots) + threadIdx.x;
    for (int v = 0; v < 16; ++v) {  // (as a loop: it is not what the kernel is for)
#pragma unroll
      for (int j = 0; j < NT; ++j) {
        int m, n;
        place(j, v / 4, m, n);
        const float* w = a.W + (int64_t)min(m + v % 4, a.M - 1) * a.ldw;
        const float* x = a.x + (int64_t)min(n, a.n - 1) * a.ldx;
        float s = 0.f;
        for (int k = c0 * KC; k < min(c1 * KC, a.K); ++k) s = __builtin_fmaf(w[k], x[k], s);
        mine[j * kSplitThreads] = s;
      }
#pragma unroll
      for (int j = 0; j < NT; ++j)
#pragma unroll
        for (int r = 0; r < 16; ++r)
          if (r == v) large[j][r] = mine[j * kSplitThreads];
    }
  }
  float4_t* to = part + (((int64_t)blockIdx.z * gridDim.y + blockIdx.y) * gridDim.x + blockIdx.x) * (kSplitRows * NB / 4) + threadIdx.x;
#pragma unroll
  for (int j = 0; j < NT; ++j)
#pragma unroll
    for (int q = 0; q < 4; ++q) {
      const float4_t v = {large[j][4 * q], large[j][4 * q + 1], large[j][4 * q + 2], large[j][4 * q + 3]};
      if (gridDim.z > 1) {
        to[(j * 4 + q) * kSplitThreads] = v;
      } else {
        int m, n;
        place(j, q, m, n);
        if (m < a.M && n < a.n) out(m, n, v);
      }
    }
}

// Adds the splits' sums up, in their order.  Grid: (tiles of W, tiles of x, values of a thread).
template <int NB, typename Out>
__global__ __launch_bounds__(kSplitThreads) void linear_split_sum_kernel(int rows, int M, Out out, const float4_t* __restrict__ part, int splits) {
  constexpr int NT = NB / 64;
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6, j = blockIdx.z / 4, q = blockIdx.z % 4;
  const int m = blockIdx.x * kSplitRows + (wave & 3) * 32 + q * 8 + (lane >> 5) * 4;
  const int n = blockIdx.y * NB + ((wave >> 2) * NT + j) * 32 + (lane & 31);
  if (n >= rows || m >= M) return;
  const int64_t step = (int64_t)gridDim.y * gridDim.x * (kSplitRows * NB / 4);
  const float4_t* p = part + ((int64_t)blockIdx.y * gridDim.x + blockIdx.x) * (kSplitRows * NB / 4) + blockIdx.z * kSplitThreads + threadIdx.x;
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
