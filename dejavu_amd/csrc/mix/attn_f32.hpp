// Causal softmax attention of a portion of a prompt in fp32 on the fp32 matrix instructions: what attn_tiles.hpp does, with
// all operands, scores, weights and sums in fp32, for heads of up to 128.
//
// A workgroup takes 32 queries of one head; its four waves take every fourth tile of 32 keys and add up in LDS, so that
// short prompts fill the chip too (500 tokens and 16 heads: 256 workgroups).  Scores are computed transposed, so a lane holds
// one query's, and the order in which the keys enter the second product is the one the accumulator has them in.  Keys and
// values come straight from memory in operand layout: 32 KB a tile and wave beside 8192 cycles of matrix instructions, so
// nothing is staged.  A lane's value columns are neighbours (column = lane * VT + tile): one load serves all tiles.
//
// The instruction adds its products one after the other, so both products are cut into short sums: with one sum for all
// entries and one for all keys, the error against 64 bits was twice the row kernel's; as it is, 1.28e-7 (500 tokens, heads
// of 128) and 1.67e-7 (after another 500) beside 1.32e-7 and 1.88e-7.  The empty asm statements keep the compiler from
// running all short sums side by side, which the registers don't hold (45 us instead of 37).
//
// 500 tokens, 16 heads of 128: 37 us; the row kernel, which reads a key for one query at a time, 180.  Bound by the
// chain of the last queries' tiles: 33 of its 80 thousand cycles are matrix instructions (64 each), the rest loads and the additions
// between them.
#pragma once
#include "attn_rows.hpp"

namespace dv {

constexpr int kF32Q = 32, kF32K = 32, kF32Waves = 4;
__device__ __attribute__((aligned(16))) const float kF32Zero[4] = {0.f, 0.f, 0.f, 0.f};
constexpr int f32_row(int vt) { return 32 * vt + 4; }  // floats of a query's sums in LDS
constexpr size_t f32_lds(int vt) { return (size_t)kF32Waves * kF32Q * f32_row(vt) * sizeof(float); }

// DU: query/key entries over 8, WHOLE: no fewer than that (finding the zeros costs 6 to 10 %), VT: value entries over 32.  Grid: H * ceil(n / 32), head fastest, last queries first.
template <int DU, bool WHOLE, int VT>
__global__ __launch_bounds__(256) void attn_f32_kernel(AttnArgs a, int keys /* rows behind k and v */) {
  extern __shared__ __attribute__((aligned(16))) float sums[];  // [wave][query][f32_row]
  __shared__ float mls[kF32Waves][kF32Q][2], wgt[kF32Waves][kF32Q];
  typedef float vals_t __attribute__((ext_vector_type(VT)));
  constexpr int ROW = f32_row(VT);
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6, l32 = lane & 31, hh = lane >> 5;
  const int head = blockIdx.x % a.H, g = head / (a.H / a.G);
  const int nblk = (a.n + kF32Q - 1) / kF32Q;
  const int q0 = (nblk - 1 - (int)(blockIdx.x / a.H)) * kF32Q;
  const int off = a.pos_host - a.base;  // key slot of query 0
  const float* K = reinterpret_cast<const float*>(a.k) + (int64_t)g * a.k_head;
  const float* V = reinterpret_cast<const float*>(a.v) + (int64_t)g * a.v_head;

  const int qi = q0 + l32;  // this lane's query; it holds entries 8 u + 4 hh .. + 3
  float4_t qf[DU];
  {
    const float* q = reinterpret_cast<const float*>(a.q) + (int64_t)(qi < a.n ? qi : 0) * a.ldq + (int64_t)head * a.dim_s;
#pragma unroll
    for (int u = 0; u < DU; ++u) {
      const int d = u * 8 + hh * 4;
      qf[u] = float4_t{0.f, 0.f, 0.f, 0.f};
      if (qi < a.n && d < a.dim_s) qf[u] = *reinterpret_cast<const float4_t*>(q + d);
    }
  }
  auto oldest_slot = [&](int q) { return max(0, oldest_key(a, a.pos_host + q) - a.base); };
  const int qslot = off + qi, klo = oldest_slot(min(qi, a.n - 1));
  const int first = oldest_slot(q0) / kF32K * kF32K, last = off + min(q0 + kF32Q, a.n) - 1;
  const float* rel = a.rel ? a.rel + (int64_t)head * a.rel_len : nullptr;
  const int vcol = min(l32 * VT, a.vdim_s - VT);  // past the last column: nothing is stored

  // tiles from here on, or before there, hold keys that some of the queries don't see
  const int some = off + q0, none = oldest_slot(min(q0 + kF32Q, a.n) - 1);
  float* mine = sums + ((int64_t)wave * kF32Q + l32) * ROW;

  float16_t o[VT];
#pragma unroll
  for (int t = 0; t < VT; ++t)
#pragma unroll
    for (int i = 0; i < 16; ++i) o[t][i] = 0.f;
  float m = -1e30f, l = 0.f;  // l: this half wave's share
  for (int k0 = first + wave * kF32K; k0 <= last; k0 += kF32Waves * kF32K) {
    auto key_of = [&](int i) { return k0 + 8 * (i >> 2) + 4 * hh + (i & 3); };
    const float* kp = K + (int64_t)min(k0 + l32, keys - 1) * a.ldk;
    // past the entries of a head that is not WHOLE zeros, like the query's: 0 times an infinite entry would be undefined
    auto key4 = [&](int u) { return *reinterpret_cast<const float4_t*>(WHOLE || u * 8 < a.dim_s ? kp + u * 8 + hh * 4 : kF32Zero); };
    float4_t kf[DU];
#pragma unroll
    for (int u = 0; u < 8; ++u) kf[u] = key4(u);
    vals_t vv[16];
#pragma unroll
    for (int i = 0; i < 16; ++i) vv[i] = *reinterpret_cast<const vals_t*>(V + (int64_t)min(key_of(i), keys - 1) * a.ldv + vcol);
    float16_t s, half;  // short sums instead of a long one: four at a time over 32 entries
#pragma unroll
    for (int u0 = 0; u0 < DU; u0 += 4) {
      float16_t part[4];
#pragma unroll
      for (int e = 0; e < 4; ++e)
#pragma unroll
        for (int i = 0; i < 16; ++i) part[e][i] = 0.f;
#pragma unroll
      for (int u = u0; u < u0 + 4; ++u)
#pragma unroll
        for (int e = 0; e < 4; ++e) part[e] = __builtin_amdgcn_mfma_f32_32x32x2f32(kf[u][e], qf[u][e], part[e], 0, 0, 0);
      const float16_t sum = (part[0] + part[1]) + (part[2] + part[3]);
      if (u0 % 8 == 0) {
        half = sum;
      } else {
        s = u0 > 4 ? s + (half + sum) : half + sum;
      }
      if (u0 + 8 < DU) {
        asm volatile("" : "+v"(kp), "+v"(*(u0 % 8 ? &s : &half)));  // keys and sums of more than two groups would not fit the registers
#pragma unroll
        for (int u = u0 + 8; u < u0 + 12; ++u) kf[u] = key4(u);
      }
    }
    float mx = -INFINITY;
#pragma unroll
    for (int i = 0; i < 16; ++i) {
      const int key = key_of(i);
      float x = s[i] * a.scale;
      if (rel) x += rel[min(max(qslot - key, 0), a.rel_len - 1)];
      if (key > qslot || key < klo) x = -INFINITY;
      s[i] = x;
      mx = fmaxf(mx, x);
    }
    mx = fmaxf(mx, __shfl_xor(mx, 32, kWave));
    const float m1 = fmaxf(m, mx), c = exp_f(m - m1);
    m = m1;
    float ps[4] = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int i = 0; i < 16; ++i) {
      const float p = s[i] == -INFINITY ? 0.f : exp_f(s[i] - m1);
      s[i] = p;
      ps[i & 3] += p;
    }
    l = __builtin_fmaf(l, c, (ps[0] + ps[1]) + (ps[2] + ps[3]));
    bool odd = false;  // an infinite or undefined value must not reach queries that don't see it: 0 times it is undefined
    if (k0 + kF32K - 1 > some || k0 < none) {
      float zero = 0.f;
#pragma unroll
      for (int i = 0; i < 16; ++i)
#pragma unroll
        for (int t = 0; t < VT; ++t) zero = __builtin_fmaf(vv[i][t], 0.f, zero);
      odd = __any(!(zero == 0.f));
    }
    if (odd) {
#pragma unroll
      for (int i = 0; i < 16; ++i) {
        mine[key_of(i) - k0] = s[i];
#pragma unroll
        for (int t = 0; t < VT; ++t)
          if (!(fabsf(vv[i][t]) < INFINITY)) vv[i][t] = 0.f;
      }
    }
#pragma unroll
    for (int t = 0; t < VT; ++t) {
      if (t >= 2) asm volatile("" : "+v"(s), "+v"(o[t - 2]));  // two tiles' sums at a time
      float16_t add[4];  // this tile's keys by themselves: the long sum has a term for 32 keys
#pragma unroll
      for (int i = 0; i < 16; ++i) add[0][i] = add[1][i] = add[2][i] = add[3][i] = 0.f;
#pragma unroll
      for (int i = 0; i < 16; ++i) add[i & 3] = __builtin_amdgcn_mfma_f32_32x32x2f32(vv[i][t], s[i], add[i & 3], 0, 0, 0);
#pragma unroll
      for (int i = 0; i < 16; ++i) o[t][i] = __builtin_fmaf(o[t][i], c, (add[0][i] + add[1][i]) + (add[2][i] + add[3][i]));
    }
    if (odd) {
      asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");  // a query's weights were stored by two lanes of this wave
      for (int key = max(k0, klo); key <= min(k0 + kF32K - 1, qslot); ++key) {
        const float p = mine[key - k0];
        const float* row = V + (int64_t)min(key, keys - 1) * a.ldv;
#pragma unroll
        for (int i = 0; i < 16; ++i)
#pragma unroll
          for (int t = 0; t < VT; ++t) {
            const float v = row[min((8 * (i >> 2) + 4 * hh + (i & 3)) * VT, a.vdim_s - VT) + t];
            if (!(fabsf(v) < INFINITY)) o[t][i] = __builtin_fmaf(p, v, o[t][i]);
          }
      }
      asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
    }
  }
  l += __shfl_xor(l, 32, kWave);

#pragma unroll
  for (int i = 0; i < 16; ++i) {
    vals_t v;
#pragma unroll
    for (int t = 0; t < VT; ++t) v[t] = o[t][i];
    *reinterpret_cast<vals_t*>(mine + (8 * (i >> 2) + 4 * hh + (i & 3)) * VT) = v;
  }
  if (hh == 0) {
    mls[wave][l32][0] = m;
    mls[wave][l32][1] = l;
  }
  __syncthreads();
  if (tid < kF32Q) {
    float mm = mls[0][tid][0];
#pragma unroll
    for (int w = 1; w < kF32Waves; ++w) mm = fmaxf(mm, mls[w][tid][0]);
    float den = 0.f, e[kF32Waves];
#pragma unroll
    for (int w = 0; w < kF32Waves; ++w) {
      e[w] = exp_f(mls[w][tid][0] - mm);
      den = __builtin_fmaf(mls[w][tid][1], e[w], den);
    }
    float c = 0.f;
    if (q0 + tid < a.n) {
      const float f = attn_factor<float>(a, q0 + tid, head, mm, den, &c);
      c *= f;
    }
#pragma unroll
    for (int w = 0; w < kF32Waves; ++w) wgt[w][tid] = e[w] * c;
  }
  __syncthreads();
  const int quads = a.vdim_s / 4;
  for (int at = tid; at < kF32Q * quads; at += 256) {
    const int q = at / quads, d = (at - q * quads) * 4;
    if (q0 + q >= a.n) break;
    float4_t v = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int w = 0; w < kF32Waves; ++w) v += *reinterpret_cast<const float4_t*>(sums + ((int64_t)w * kF32Q + q) * ROW + d) * wgt[w][q];
    *reinterpret_cast<float4_t*>(reinterpret_cast<float*>(a.out) + ((int64_t)(q0 + q) * a.H + head) * a.vdim_s + d) = v;
  }
}

}  // namespace dv
