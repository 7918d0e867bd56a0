// The epilogues of linear_rows.hpp behind the tiles of gemm_ring.hpp and gemm_wide.hpp.
#pragma once
#include <type_traits>

#include "../gemm_wide.hpp"
#include "elem.hpp"
#include "stream.hpp"

namespace dv {

using TileArgs = dvTileArgs;

__device__ __forceinline__ bool aligned_to(const void* p, unsigned bytes) { return (reinterpret_cast<uintptr_t>(p) & (bytes - 1)) == 0; }

// The results of a lane: rows m .. m + 3 of W (m % 4 == 0), activation row n.
template <int AFTER>
__device__ __forceinline__ void tile_out(const TileArgs& a, int m, int n, float4_t v) {
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

template <int AFTER>
struct MixOut {
  TileArgs a;
  __device__ __forceinline__ void operator()(int m, int n, const float4_t& v) const { tile_out<AFTER>(a, m, n, v); }
};

// What gemm_wide.hpp stores: the results of rows m .. m + 3 of W (DV_OUT_T or DV_OUT_GLU).
template <int AFTER>
struct WideOut {
  static constexpr int kOuts = AFTER == DV_OUT_GLU ? 2 : 4;
  typedef bf16_t vec_t __attribute__((ext_vector_type(kOuts)));
  TileArgs a;
  __device__ __forceinline__ bf16_t* base() const { return reinterpret_cast<bf16_t*>(a.out); }
  __device__ __forceinline__ int64_t ld() const { return a.ldo; }
  __device__ __forceinline__ int columns() const { return AFTER == DV_OUT_GLU ? a.M / 2 : a.M; }
  struct Row : WideBias<bf16_t> {};
  __device__ __forceinline__ Row row(int m) const {
    Row r;
    r.load(AFTER == DV_OUT_GLU ? nullptr : reinterpret_cast<const bf16_t*>(a.bias), a.M, m);
    return r;
  }
  __device__ __forceinline__ vec_t make(const Row& r, const float4_t& v) const {
    if constexpr (AFTER == DV_OUT_GLU)
      return vec_t{(bf16_t)glu_f(v[0], v[1], a.act, a.limit), (bf16_t)glu_f(v[2], v[3], a.act, a.limit)};
    else
      return vec_t{(bf16_t)(v[0] + to_f(r.v[0])), (bf16_t)(v[1] + to_f(r.v[1])), (bf16_t)(v[2] + to_f(r.v[2])), (bf16_t)(v[3] + to_f(r.v[3]))};
  }
};

// What follows a sublayer's last product behind the sums of its parts, four channels at a time (residual_norm_kernel's arithmetic on the
// sums as they are).
struct WideResidual {
  dvResidual r;
  int M;
  struct Ready {
    float4_t x, x0;
  };
  __device__ __forceinline__ Ready ready(int64_t row, int m) const {
    Ready o;
    o.x = *reinterpret_cast<const float4_t*>(r.x + row * M + m);
    o.x0 = r.x0 ? *reinterpret_cast<const float4_t*>(r.x0 + row * M + m) : float4_t{0.f, 0.f, 0.f, 0.f};
    return o;
  }
  __device__ __forceinline__ void operator()(int64_t row, int m, const float4_t& y, const Ready& o) const {
    const int64_t at = row * M + m;
    float4_t v = o.x, h;
    const float4_t w = *reinterpret_cast<const float4_t*>(r.post.w + m), b = *reinterpret_cast<const float4_t*>(r.post.b + m);
#pragma unroll
    for (int e = 0; e < 4; ++e) v[e] += __builtin_fmaf(tanh_f(r.post.alpha * y[e]), w[e], b[e]);
    if (r.x0) v += o.x0;
    *reinterpret_cast<float4_t*>(r.x + at) = v;
    if (!r.h) return;
    const float4_t pw = *reinterpret_cast<const float4_t*>(r.pre.w + m), pb = *reinterpret_cast<const float4_t*>(r.pre.b + m);
#pragma unroll
    for (int e = 0; e < 4; ++e) h[e] = __builtin_fmaf(tanh_f(r.pre.alpha * v[e]), pw[e], pb[e]);
    store_quad(reinterpret_cast<bf16_t*>(r.h) + at, h);
  }
};

// The parts' sums as rows of bf16, on 8-byte boundaries.
struct WideSumOut {
  WideOut<DV_OUT_T> out;
  typedef WideOut<DV_OUT_T>::Row Ready;
  __device__ __forceinline__ Ready ready(int64_t, int m) const { return out.row(m); }
  __device__ __forceinline__ void operator()(int64_t row, int m, const float4_t& v, const Ready& r) const {
    typedef WideOut<DV_OUT_T>::vec_t vec_t;
    *reinterpret_cast<vec_t*>(out.base() + row * out.ld() + m) = out.make(r, v);
  }
};

}  // namespace dv
