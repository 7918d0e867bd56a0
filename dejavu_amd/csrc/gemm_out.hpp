// What the rows and the results of the products in gemm_ring.hpp and gemm_big.hpp are: rows of a weight, gathered rows, or
// the q, k, v rows of selected heads with their scatter into the caches.
#pragma once
#include "common.hpp"
#include "gemm_wide.hpp"

namespace dv {

// QKV mode: the M = 3 * Hk * hd output rows are the q, k, v rows of the selected heads
// (m = (t * Hk + i) * hd + j -> weight row (t * H + head_idx[i]) * hd + j).  The X rows are `tokens`
// window tokens of `nseq` sequences each, row r = s * nseq + b (tokens == 1: one token per sequence).
// live[i * live_stride + s * live_tstride] < 0 skips (head i, token s); a head with no live token, or out
// of range, is skipped altogether.  The result of token y_token goes to column `weight row` of
// Y (nseq, 3, H, hd); the K / V rows of every live (head, token) are appended to the per-sequence caches
// k_cache (nseq, H, hd/8, S, 8), v_cache (nseq, H, S, hd) at position
// positions[per_sample ? b : 0] + pos_add + s.
struct QkvScatter {
  const int* head_idx;
  const int* live;
  int live_stride, Hk, H, hd;
  half_t* k_cache;
  half_t* v_cache;
  const int* positions;
  int per_sample, pos_add, S;
  int nseq, tokens, live_tstride, y_token;
};

__device__ __forceinline__ int qkv_row_of(const QkvScatter& q, int m) {
  const int t = m / (q.Hk * q.hd);
  const int rem = m - t * q.Hk * q.hd;
  const int i = rem / q.hd, j = rem - i * q.hd;
  const int h = q.head_idx[i];
  if (h < 0 || h >= q.H || t > 2) return -1;
  if (q.live != nullptr) {
    bool any = false;
    for (int s = 0; s < q.tokens; ++s)
      any |= q.live[(int64_t)i * q.live_stride + (int64_t)s * q.live_tstride] >= 0;
    if (!any) return -1;
  }
  return (t * q.H + h) * q.hd + j;
}

// stores four finished values: consecutive output rows m .. m + 3 of X row r (m % 4 == 0, so they belong to
// one head and one 8-pack of the key cache; weight rows rid .. rid + 3): one 8-byte store to Y for the token
// that is wanted there and, for K / V rows, one to the cache
__device__ __forceinline__ void qkv_store4(const QkvScatter& q, half_t* __restrict__ Y, int r, int m, int rid,
                                           const float (&val)[4]) {
  const int s = q.tokens > 1 ? r / q.nseq : 0;
  const int b = r - s * q.nseq;
  if (q.live != nullptr && q.tokens > 1) {
    const int i = (m % (q.Hk * q.hd)) / q.hd;
    if (q.live[(int64_t)i * q.live_stride + (int64_t)s * q.live_tstride] < 0) return;
  }
  const half4_t o = {(half_t)val[0], (half_t)val[1], (half_t)val[2], (half_t)val[3]};
  if (s == q.y_token) *reinterpret_cast<half4_t*>(Y + (int64_t)b * 3 * q.H * q.hd + rid) = o;
  if (q.k_cache == nullptr) return;
  const int t = rid / (q.H * q.hd);
  if (t == 0) return;
  const int rem = rid - t * q.H * q.hd;
  const int h = rem / q.hd, j = rem - h * q.hd;
  const int dst = (q.positions ? q.positions[q.per_sample ? b : 0] : 0) + q.pos_add + s;
  if (dst < 0 || dst >= q.S) return;
  half_t* p = t == 1 ? q.k_cache + ((((int64_t)b * q.H + h) * (q.hd / 8) + j / 8) * q.S + dst) * 8 + (j & 7)
                     : q.v_cache + (((int64_t)b * q.H + h) * q.S + dst) * q.hd + j;
  *reinterpret_cast<half4_t*>(p) = o;
}

struct QkvRows {  // (a head out of range reads row 0 and is not stored)
  static constexpr bool kPastCaches = false;
  static constexpr int kMostCols = 256;
  QkvScatter q;
  __device__ __forceinline__ int64_t operator()(int m) const {
    const int t = m / (q.Hk * q.hd), rem = m - t * q.Hk * q.hd, i = rem / q.hd, h = q.head_idx[i];
    return h < 0 || h >= q.H ? 0 : (t * q.H + h) * q.hd + rem - i * q.hd;
  }
};
struct QkvOut {
  const half_t* bias;
  half_t* Y;
  QkvScatter q;
  // the four values are four consecutive rows of one (q|k|v, head): hd % 4 == 0
  __device__ __forceinline__ void operator()(int m, int r, float4_t v) const {
    const int t = m / (q.Hk * q.hd), rem = m - t * q.Hk * q.hd, i = rem / q.hd, h = q.head_idx[i];
    if (h < 0 || h >= q.H) return;
    if (q.live != nullptr && q.tokens == 1 && q.live[(int64_t)i * q.live_stride] < 0) return;
    const int rid = (t * q.H + h) * q.hd + rem - i * q.hd;
    float val[4];
#pragma unroll
    for (int e = 0; e < 4; ++e) val[e] = v[e] + (bias != nullptr ? (float)bias[rid + e] : 0.f);
    qkv_store4(q, Y, r, m, rid, val);
  }
};

// act(v) to rows m .. m + 3 of column n of Y (n_rows, ldy)
__device__ __forceinline__ void store_rows4(half_t* Y, int64_t ldy, int M, int m, int n, const float (&val)[4], int act) {
  half4_t o;
#pragma unroll
  for (int e = 0; e < 4; ++e) o[e] = (half_t)(act ? act_f(val[e], act) : val[e]);
  half_t* dst = Y + (int64_t)n * ldy + m;
  if (m + 3 < M && (ldy & 3) == 0 && (reinterpret_cast<uintptr_t>(Y) & 7) == 0) {
    *reinterpret_cast<half4_t*>(dst) = o;
  } else {
#pragma unroll
    for (int e = 0; e < 4; ++e)
      if (m + e < M) dst[e] = o[e];
  }
}

struct PlainOut {
  const half_t* bias;
  int act;
  half_t* Y;
  int64_t ldy;
  int M;
  __device__ __forceinline__ void operator()(int m, int n, float4_t v) const {
    float val[4];
#pragma unroll
    for (int e = 0; e < 4; ++e) val[e] = v[e] + (bias != nullptr ? (float)bias[m + e < M ? m + e : M - 1] : 0.f);
    store_rows4(Y, ldy, M, m, n, val, act);
  }
};

// The same as gemm_wide.hpp stores it, for the activations that are cheap enough to stand there once for every sum.  It stands in
// for the library's product with the activation behind it, so a sum that is no number stays one (act_f makes it zero).
template <int ACT>
struct WidePlainOut {
  static constexpr int kOuts = 4;
  static_assert(ACT == 0 || ACT == 1 || ACT == 4, "identity, ReLU, squared ReLU");
  const half_t* bias;
  half_t* Y;
  int64_t ldy;
  int M;
  __device__ __forceinline__ half_t* base() const { return Y; }
  __device__ __forceinline__ int64_t ld() const { return ldy; }
  __device__ __forceinline__ int columns() const { return M; }
  struct Row : WideBias<half_t> {};
  __device__ __forceinline__ Row row(int m) const {
    Row r;
    r.load(bias, M, m);
    return r;
  }
  __device__ __forceinline__ half4_t make(const Row& r, const float4_t& v) const {
    half4_t o;
#pragma unroll
    for (int e = 0; e < 4; ++e) {
      float s = v[e] + (float)r.v[e];
      if (ACT != 0) s = s < 0.f ? 0.f : s;
      o[e] = (half_t)(ACT == 4 ? s * s : s);
    }
    return o;
  }
};

// What wide_sum_kernel stores: WidePlainOut's results, rows on 8-byte boundaries.
template <int ACT>
struct WideSumOut {
  WidePlainOut<ACT> out;
  typedef typename WidePlainOut<ACT>::Row Ready;
  __device__ __forceinline__ Ready ready(int64_t, int m) const { return out.row(m); }
  __device__ __forceinline__ void operator()(int64_t row, int m, const float4_t& v, const Ready& r) const {
    *reinterpret_cast<half4_t*>(out.Y + row * out.ldy + m) = out.make(r, v);
  }
};

struct GatheredRows {
  static constexpr bool kPastCaches = true;
  static constexpr int kMostCols = 64;
  const void* idx;
  int idx_bytes, Z;
  __device__ __forceinline__ int64_t operator()(int m) const {  // an index out of range reads row 0; its result is act(0)
    const int64_t id = load_index(idx, idx_bytes, m);
    return id >= 0 && id < Z ? id : 0;
  }
};
struct GatheredOut {
  GatheredRows rows;
  const half_t* bias;
  int act;
  half_t* Y;
  int64_t ldy;
  int M;
  __device__ __forceinline__ void operator()(int m, int n, float4_t v) const {
    float val[4];
#pragma unroll
    for (int e = 0; e < 4; ++e) {
      const int64_t id = load_index(rows.idx, rows.idx_bytes, m + e < M ? m + e : M - 1);
      const bool ok = id >= 0 && id < rows.Z;
      val[e] = ok ? v[e] + (bias != nullptr ? (float)bias[id] : 0.f) : 0.f;
    }
    store_rows4(Y, ldy, M, m, n, val, act);
  }
};

}  // namespace dv
