// QKV of the chosen heads for a back-fill window of several sequences: out of up to 16 window tokens a head takes part in only
// those it has missed since it was last chosen and the newest one, two or three of sixteen when every third head is chosen at a time.
// A workgroup owns the 128 weight rows of a head's queries, keys or values and multiplies the rows of X of the tokens that are live for the head,
// found from the slot list when it starts, 64, 128 or 256 of them at a time, as many as it takes; queries are wanted of the newest
// token only.  The ring of gemm_ring.hpp does the rest.
//
// Bound by the stream of the weights (24 of 72 heads of 9216, sixteen sequences: 30 us of 46 + 7) and by the heads with the most live tokens, whose
// workgroups end last.
#pragma once
#include "gemm_out.hpp"
#include "gemm_ring.hpp"

namespace dv {

constexpr int kWindowRows = 128, kWindowCols = 256;
constexpr size_t kWindowLds = (size_t)3 * (kWindowRows + kWindowCols) * 64 * 2;

struct WindowPlan {
  int rows, chunks, splits;  // tiles of 128 weight rows, of 256 rows of X, splits of K
  size_t workspace_bytes() const {
    return splits > 1 ? (size_t)splits * chunks * rows * kWindowRows * kWindowCols * sizeof(float) : 0;
  }
};

// About a workgroup per compute unit: most tiles' rows of X are one chunk, the workgroups of the others end at once.
inline WindowPlan plan_window(int n, int M, int K, int units) {
  WindowPlan p;
  p.rows = (M + kWindowRows - 1) / kWindowRows;
  p.chunks = (n + kWindowCols - 1) / kWindowCols;
  int s = units / p.rows;
  if (s > K / 256) s = K / 256;
  p.splits = s < 1 ? 1 : s > 8 ? 8 : s;
  return p;
}

// The rows of X of a tile: those of the tokens of `mask`, ascending.
struct LiveCols {
  unsigned mask;
  int nseq;
  __device__ __forceinline__ int rows() const { return __builtin_popcount(mask) * nseq; }
  __device__ __forceinline__ int operator()(int n) const {
    const int k = n / nseq;
    unsigned rest = mask;
    for (int i = 0; i < k; ++i) rest &= rest - 1;
    return (__builtin_ctz(rest) - k) * nseq + n;
  }
};

// Which windows it takes; the others' tokens are all multiplied by the ring.  us, all tokens / the live ones, every third head chosen by chance (and
// all heads, once a window): 72 heads of 9216 with 208 / 256 / 312 / 416 rows 68 / 58, 70 / 58, 96 / 63, 152 / 89 (256 rows 185 / 156, 512 355 / 242), 96 of 12288 with 208 / 256 / 512
// 122 / 101, 124 / 111, 210 / 111 (409 / 343, 646 / 332), 40 of 5120 31 / 28, 32 / 24, 44 / 34 (69 / 55, 105 / 81), every second of 32 of 4096 30 / 27, 31 / 23, 46 / 39 (51 / 37, 82 / 49).  Up
// to 192 rows the weights' stream is the time whatever the rows, and finding the live ones comes on top: 72 heads with 72 / 128 / 192 rows 43 / 45, 45 / 47,
// 55 / 60, 96 with 108 / 180 77 / 83, 107 / 124.  Smaller heads share a tile and each other's tokens (48 of 64, 260 to 360 rows: 0.76 to 1.1 times the
// speed), and fewer than a workgroup per compute unit in eight splits leave it idle (8 of 32 heads of 4096: 0.83 to 1.2).
// Where every chosen head has missed all tokens, as hardly ever, the live ones take up to a fifth longer (13 of 40 heads, 384 rows: 39 / 47).
inline bool window_live(int tokens, int nseq, int hd, int M, int units) {
  return tokens > 1 && tokens * nseq > 192 && hd == kWindowRows && M >= units * 16;
}

// The tokens that the head of rows m0 .. m0 + 127 needs; the same for all threads.
__device__ __forceinline__ LiveCols live_tokens(const QkvScatter& q, int m0) {
  const int lane = threadIdx.x & 63;
  const int k = m0 / kWindowRows, t = k / q.Hk, i = k - t * q.Hk, h = q.head_idx[i];
  if (h < 0 || h >= q.H) return LiveCols{0, q.nseq};
  // a lane for each token: one wait (token after token 8 us)
  const bool live = q.live[(int64_t)i * q.live_stride + (int64_t)min(lane, q.tokens - 1) * q.live_tstride] >= 0;
  return LiveCols{(unsigned)__ballot(lane < q.tokens && live && (t > 0 || lane == q.y_token)), q.nseq};
}

// Grid: (tiles of W, chunks of 256 rows of X, splits of K).  part: [split][chunk][tile][value][thread].
// (Chunks of 64 rows instead, each a workgroup and two of them to a compute unit: 58 us where this takes 45, the flush 299 / 181: those
// with rows land beside each other while compute units are idle.)
__global__ __launch_bounds__(512) void qkv_window_live_kernel(RingOperands<half_t> a, QkvRows rows, QkvOut out, float4_t* __restrict__ part) {
  extern __shared__ __attribute__((aligned(16))) unsigned char slots[];
  const int m0 = blockIdx.x * kWindowRows, n0 = blockIdx.y * kWindowCols;
  const LiveCols cols = live_tokens(rows.q, m0);
  const int n = cols.rows(), here = n - n0;
  if (here <= 0) return;
  float4_t* p = part + (((int64_t)blockIdx.z * gridDim.y + blockIdx.y) * gridDim.x + blockIdx.x) * (kWindowRows * kWindowCols / 4);
  if (here <= 64) ring_tile<half_t, kWindowRows, 64, 64, 6, 2, 4, false, false>(a, rows, cols, out, m0, n0, n, p, slots);
  else if (here <= 128) ring_tile<half_t, kWindowRows, 128, 64, 4, 2, 4, false, false>(a, rows, cols, out, m0, n0, n, p, slots);
  else ring_tile<half_t, kWindowRows, 256, 64, 3, 2, 4, false, false>(a, rows, cols, out, m0, n0, n, p, slots);
}

// Adds the splits' sums up, in their order.  Grid: (tiles of W, chunks, values of a thread of the widest tile).
__global__ __launch_bounds__(512) void qkv_window_sum_kernel(QkvRows rows, QkvOut out, int M, const float4_t* __restrict__ part, int splits) {
  const int m0 = blockIdx.x * kWindowRows, n0 = blockIdx.y * kWindowCols;
  const LiveCols cols = live_tokens(rows.q, m0);
  const int n = cols.rows(), here = n - n0, nt = here <= 64 ? 1 : here <= 128 ? 2 : 4;  // tiles of 16 columns a wave
  if (here <= 0 || (int)blockIdx.z >= 4 * nt) return;
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6, wm = wave & 1, wn = wave >> 1;
  const int i = blockIdx.z / nt, j = blockIdx.z % nt;
  const int m = m0 + (wm * 4 + i) * 16 + (lane >> 4) * 4, col = n0 + (wn * nt + j) * 16 + (lane & 15);
  if (m >= M || col >= n) return;
  const int64_t step = (int64_t)gridDim.y * gridDim.x * (kWindowRows * kWindowCols / 4);
  const float4_t* p = part + ((int64_t)blockIdx.y * gridDim.x + blockIdx.x) * (kWindowRows * kWindowCols / 4) + blockIdx.z * 512 + threadIdx.x;
  float4_t v = p[0];
  for (int s = 1; s < splits; ++s) v += p[s * step];
  out(m, cols(col), v);
}

}  // namespace dv
