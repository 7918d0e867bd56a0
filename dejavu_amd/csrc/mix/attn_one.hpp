// Softmax attention of one decode row whose keys are few, in one launch: a workgroup of sixteen waves per query head takes all
// of them, so nothing is left for a launch that merges, and heads that share keys read them again from L2.  bf16 keys and
// values, fp32 arithmetic.
//
// Bound by latency and by what one compute unit fetches (about 70 bytes a ns): a launch that depends on the one before costs 2.7 to
// 4.5 us whatever it does, so the split kernel and its merge lose to this one while the keys are few.  All of a head's vectors
// and the first U keys a lane are requested before anything waits: in a model, where each of these waits is one for memory, that
// took 6.6 us where requests in the order of their use took 13 to 16 (81 keys, 32 heads on 8).
// us, before and now: a ring of 81 keys, 16 heads on 4 key heads of 128 + 128, 10.9 -> 6.4, 366 keys 10.9 -> 10.2; latents of rank 256, 16
// heads (three launches) 81 keys 12.3 -> 6.1, 366 13.1 -> 9.3; rank 512, 32 heads, 81 keys 17.4 -> 10.2.
#pragma once
#include "attn_rows.hpp"

namespace dv {

constexpr int kOneWaves = 16, kOneThreads = 64 * kOneWaves;

__device__ __forceinline__ float dot8(const float (&q)[8], const Pack8<bf16_t>& k) {
  float s = q[0] * k.get(0), t = q[1] * k.get(1);
#pragma unroll
  for (int e = 2; e < 8; e += 2) {
    s = __builtin_fmaf(q[e], k.get(e), s);
    t = __builtin_fmaf(q[e + 1], k.get(e + 1), t);
  }
  return s + t;
}

// Softmax over the keys of a wave: LPK lanes hold a key, eight entries each; a lane's U scores are those of its group's keys.
template <int LPK, int U>
struct OneSums {
  float m = -1e30f, l = 0.f, acc[8] = {0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f};
  __device__ __forceinline__ void add(const float (&s)[U], const bool (&in)[U], const Pack8<bf16_t> (&v)[U]) {
    float top = m;
#pragma unroll
    for (int u = 0; u < U; ++u)
      if (in[u]) top = fmaxf(top, s[u]);
#pragma unroll
    for (int off = LPK; off < 64; off <<= 1) top = fmaxf(top, __shfl_xor(top, off, kWave));
    const float c = exp_f(m - top);
    m = top;
    l *= c;
#pragma unroll
    for (int e = 0; e < 8; ++e) acc[e] *= c;
#pragma unroll
    for (int u = 0; u < U; ++u) {
      const float p = in[u] ? exp_f(s[u] - top) : 0.f;
      l += p;
      if (in[u]) {  // (what lies past the last key may be anything)
#pragma unroll
        for (int e = 0; e < 8; ++e) acc[e] = __builtin_fmaf(p, v[u].get(e), acc[e]);
      }
    }
  }
  // the groups of the wave
  __device__ __forceinline__ void join() {
#pragma unroll
    for (int off = LPK; off < 64; off <<= 1) {
      l += __shfl_xor(l, off, kWave);
#pragma unroll
      for (int e = 0; e < 8; ++e) acc[e] += __shfl_xor(acc[e], off, kWave);
    }
  }
};

// What closes a head, as in attn_factor: its sink and the logit of its gate, requested long before they are used.
struct HeadEnd {
  float sink, gate;
  __device__ __forceinline__ HeadEnd(const AttnArgs& a, int head, const float* other)
      : sink(*(a.sink ? a.sink + head : other)), gate(*(a.gate ? reinterpret_cast<const float*>(a.gate) + head : other)) {}
  __device__ __forceinline__ float factor(const AttnArgs& a, float m, float l) const {
    const float mm = a.sink ? fmaxf(m, sink) : m, c = exp_f(m - mm);
    float f = c / (a.sink ? __builtin_fmaf(l, c, exp_f(sink - mm)) : l * c);
    if (a.gate) f *= sigmoid_f(gate);
    return f;
  }
};

// Sum of entry d over the waves, and the maximum and denominator of all.
__device__ __forceinline__ float one_total(const float* red, int stride, const float (*ml)[2], int d, float* m, float* l) {
  float top = -1e30f, den = 0.f, t = 0.f;
#pragma unroll
  for (int w = 0; w < kOneWaves; ++w) top = fmaxf(top, ml[w][0]);
#pragma unroll
  for (int w = 0; w < kOneWaves; ++w) {
    const float c = exp_f(ml[w][0] - top);
    den = __builtin_fmaf(ml[w][1], c, den);
    t = __builtin_fmaf(red[w * stride + d], c, t);
  }
  *m = top;
  *l = den;
  return t;
}

// Keys and values of up to 128 entries in a ring or a list; this token's come as fp32 from fresh_k / fresh_v and are stored.
// Grid: (H).  U: 64 keys each a turn.
template <int U>
__global__ __launch_bounds__(kOneThreads) void attn_one_kernel(AttnArgs a) {
  __shared__ float red[kOneWaves * 128], ml[kOneWaves][2];
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6, sub = lane & 15, group = threadIdx.x >> 4;
  const int head = blockIdx.x, rep = a.H / a.G, g = head / rep;
  const int ck = min(sub * 8, a.dim_s - 8), cv = min(sub * 8, a.vdim_s - 8);
  const bool in_k = sub * 8 < a.dim_s;
  // What does not depend on the position is requested first and all together (from the query where there is none), what closes
  // the head included: one wait for all of it.
  const float* qp = reinterpret_cast<const float*>(a.q) + (int64_t)head * a.dim_s + ck;
  Pack8<float> qr, qw, fk, kw, fv, ov;
  qr.load(qp);
  qw.load(a.q_w ? a.q_w + ck : qp);
  fk.load(a.fresh_k ? a.fresh_k + (int64_t)g * a.dim_s + ck : qp);
  kw.load(a.k_w ? a.k_w + ck : qp);
  fv.load(a.fresh_v ? a.fresh_v + (int64_t)g * a.vdim_s + cv : qp);
  ov.load(a.other_v ? a.other_v + (int64_t)g * a.vdim_s + cv : qp);
  const float lam = *(a.other_v ? a.lambda : qp);
  const HeadEnd end(a, head, qp);
  const int pos = seq_position(a.pos_dev, a.pos_host), lo = oldest_key(a, pos);
  const bf16_t* K = reinterpret_cast<const bf16_t*>(a.k) + (int64_t)g * a.k_head + ck;
  const bf16_t* V = reinterpret_cast<const bf16_t*>(a.v) + (int64_t)g * a.v_head + cv;
  const float* rel = a.rel ? a.rel + (int64_t)head * a.rel_len : qp;
  const int s0 = a.ring > 0 ? lo % a.ring : lo - a.base, rel_last = a.rel ? a.rel_len - 1 : 0;
  auto slot = [&](int j) -> int64_t {
    const int s = s0 + (j - lo);
    return a.ring > 0 && s >= a.ring ? s - a.ring : s;
  };
  Pack8<bf16_t> k[U], v[U];
  float bias[U];
  auto load = [&](int jt) {
#pragma unroll
    for (int u = 0; u < U; ++u) k[u].load(K + slot(min(jt + u * 64 + group, pos)) * a.ldk);
#pragma unroll
    for (int u = 0; u < U; ++u) v[u].load(V + slot(min(jt + u * 64 + group, pos)) * a.ldv);
#pragma unroll
    for (int u = 0; u < U; ++u) bias[u] = rel[min(max(pos - (jt + u * 64 + group), 0), rel_last)];
  };
  load(lo);
  // eight entries of a normed row; the mean over norm_dim of them
  auto normed = [&](const Pack8<float>& r, const Pack8<float>& w, bool weighted, float (&y)[8]) {
    float s = 1.f;
    if (a.norm_dim > 0) {
      float ss = 0.f;
#pragma unroll
      for (int e = 0; e < 8; ++e)
        if (sub * 8 + e < a.norm_dim) ss = __builtin_fmaf(r.get(e), r.get(e), ss);
      s = 1.f / sqrtf(row16_sum(ss) / a.norm_dim + a.eps);
    }
#pragma unroll
    for (int e = 0; e < 8; ++e) y[e] = in_k ? r.get(e) * s * (weighted ? w.get(e) : 1.f) : 0.f;
  };
  float q[8];
  normed(qr, qw, a.q_w != nullptr, q);
  Pack8<bf16_t> kf, vf;
  if (a.fresh_k) {
    typedef bf16_t pack_t __attribute__((ext_vector_type(8)));
    float y[8];
    normed(fk, kw, a.k_w != nullptr, y);
    pack_t t;
#pragma unroll
    for (int e = 0; e < 8; ++e) t[e] = (bf16_t)y[e];
    kf.v = __builtin_bit_cast(uint4_t, t);
#pragma unroll
    for (int e = 0; e < 8; ++e) t[e] = (bf16_t)(a.other_v ? __builtin_fmaf(lam, ov.get(e), (1.f - lam) * fv.get(e)) : fv.get(e));
    vf.v = __builtin_bit_cast(uint4_t, t);
    if (head == g * rep && group == 0) {  // one of the workgroups of a key head stores the rows; nobody reads them here
      if (in_k) *reinterpret_cast<uint4_t*>(const_cast<bf16_t*>(K) + slot(pos) * a.ldk) = kf.v;
      if (sub * 8 < a.vdim_s) *reinterpret_cast<uint4_t*>(const_cast<bf16_t*>(V) + slot(pos) * a.ldv) = vf.v;
    }
  }
  OneSums<16, U> sums;
  for (int jt = lo; jt <= pos; jt += 64 * U) {
    float s[U];
    bool in[U];
#pragma unroll
    for (int u = 0; u < U; ++u) {
      const int j = jt + u * 64 + group;
      in[u] = j <= pos;
      if (a.fresh_k && j == pos) k[u] = kf, v[u] = vf;
      s[u] = row16_sum(in_k ? dot8(q, k[u]) : 0.f) * a.scale;
      if (a.rel) s[u] += bias[u];
    }
    sums.add(s, in, v);
    if (jt + 64 * U <= pos) load(jt + 64 * U);
  }
  sums.join();
  if (lane < 16) {
#pragma unroll
    for (int e = 0; e < 8; ++e) red[wave * 128 + lane * 8 + e] = sums.acc[e];
    if (lane == 0) ml[wave][0] = sums.m, ml[wave][1] = sums.l;
  }
  __syncthreads();
  const int d = threadIdx.x;
  if (d < a.vdim_s) {
    float m, l;
    const float t = one_total(red, 128, ml, d, &m, &l);
    reinterpret_cast<bf16_t*>(a.out)[(int64_t)head * a.vdim_s + d] = (bf16_t)(t * end.factor(a, m, l));
  }
}

// Latent attention of one row: W_uk applied to the query, attention over the latents, W_uv applied to what they add up to.
// q (H, dim_s) fp32, Wk (H * dim_s, rank), Wv (H * vrows, rank), the latents a.k with rank a.dim_s <= 8 * LPK entries.
// Grid: (H).  U: 1024 / LPK keys each a turn.
template <int LPK, int U>
__global__ __launch_bounds__(kOneThreads) void latent_one_kernel(AttnArgs a, const bf16_t* __restrict__ Wk, int dim_s,
                                                                 const bf16_t* __restrict__ Wv, int vrows, bf16_t* __restrict__ out) {
  constexpr int G = kOneThreads / LPK, RW = 128 / G;  // rows at a time; loads that 128 rows take
  __shared__ __attribute__((aligned(16))) float red[kOneWaves * LPK * 8], lat[LPK * 8], ml[kOneWaves][2];
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6, sub = lane & (LPK - 1), group = threadIdx.x / LPK;
  const int head = blockIdx.x, rank = a.dim_s, col = min(sub * 8, rank - 8);
  const bool in_row = sub * 8 < rank;
  const bf16_t* C = reinterpret_cast<const bf16_t*>(a.k) + col;
  const float* q = reinterpret_cast<const float*>(a.q) + (int64_t)head * dim_s;
  Wk += (int64_t)head * dim_s * rank + col;
  Wv += (int64_t)head * vrows * rank + col;
  const HeadEnd end(a, head, q);
  Pack8<bf16_t> w[RW], k[U];
  float qv[RW];
#pragma unroll
  for (int i = 0; i < RW; ++i) {
    const int d = min(i * G + group, dim_s - 1);
    w[i].load(Wk + (int64_t)d * rank);
    qv[i] = q[d];
  }
  const int pos = seq_position(a.pos_dev, a.pos_host);
  auto load = [&](int jt) {
#pragma unroll
    for (int u = 0; u < U; ++u) k[u].load(C + (int64_t)min(jt + u * G + group, pos) * a.ldk);
  };
  load(0);
  // a wave's sums over its rows lie in red, those over all waves in lat
  auto all_waves = [&](float (&x)[8]) {
#pragma unroll
    for (int off = LPK; off < 64; off <<= 1)
#pragma unroll
      for (int e = 0; e < 8; ++e) x[e] += __shfl_xor(x[e], off, kWave);
    if (lane < LPK) {
#pragma unroll
      for (int e = 0; e < 8; ++e) red[wave * LPK * 8 + lane * 8 + e] = x[e];
    }
    __syncthreads();
  };
  auto mine = [&](float (&x)[8]) {
    __syncthreads();
    Pack8<float> t;
    t.load(lat + sub * 8);
#pragma unroll
    for (int e = 0; e < 8; ++e) x[e] = in_row ? t.get(e) : 0.f;
  };
  float x[8] = {0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f};
#pragma unroll
  for (int i = 0; i < RW; ++i) {
    if (i * G + group < dim_s) {
#pragma unroll
      for (int e = 0; e < 8; ++e) x[e] = __builtin_fmaf(w[i].get(e), qv[i], x[e]);
    }
  }
  for (int d = RW * G + group; d < dim_s; d += G) {
    Pack8<bf16_t> r;
    r.load(Wk + (int64_t)d * rank);
#pragma unroll
    for (int e = 0; e < 8; ++e) x[e] = __builtin_fmaf(r.get(e), q[d], x[e]);
  }
  all_waves(x);
  const int d = threadIdx.x;
  if (d < LPK * 8) {
    float t = 0.f;
#pragma unroll
    for (int i = 0; i < kOneWaves; ++i) t += red[i * LPK * 8 + d];
    lat[d] = t;
  }
  mine(x);
#pragma unroll
  for (int i = 0; i < RW; ++i) w[i].load(Wv + (int64_t)min(i * G + group, vrows - 1) * rank);
  auto across = [&](float s) {
    s = row16_sum(s);
#pragma unroll
    for (int off = 16; off < LPK; off <<= 1) s += __shfl_xor(s, off, kWave);
    return s;
  };
  OneSums<LPK, U> sums;
  for (int jt = 0; jt <= pos; jt += U * G) {
    float s[U];
    bool in[U];
#pragma unroll
    for (int u = 0; u < U; ++u) {
      in[u] = jt + u * G + group <= pos;
      s[u] = across(in_row ? dot8(x, k[u]) : 0.f) * a.scale;
    }
    sums.add(s, in, k);
    if (jt + U * G <= pos) load(jt + U * G);
  }
#pragma unroll
  for (int off = LPK; off < 64; off <<= 1) sums.l += __shfl_xor(sums.l, off, kWave);
  if (lane == 0) ml[wave][0] = sums.m, ml[wave][1] = sums.l;
  all_waves(sums.acc);
  if (d < LPK * 8) {
    float m, l;
    const float t = one_total(red, LPK * 8, ml, d, &m, &l);
    lat[d] = t * end.factor(a, m, l);
  }
  mine(x);
  for (int i = 0; i * G < vrows; ++i) {
    const int r = i * G + group;
    Pack8<bf16_t> t = w[0];
    if (i >= RW) t.load(Wv + (int64_t)min(r, vrows - 1) * rank);
#pragma unroll
    for (int n = 1; n < RW; ++n)
      if (i == n) t = w[n];
    const float s = across(in_row ? dot8(x, t) : 0.f);
    if (sub == 0 && r < vrows) out[(int64_t)head * vrows + r] = (bf16_t)s;
  }
}

}  // namespace dv
