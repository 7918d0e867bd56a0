// Prompt-phase (prefill) causal attention on the matrix cores, writing the prompt's K / V rows
// straight into the decode caches.
//
//   ctx[b, t, h, :] = softmax_{s <= t}( q[b, t, h] . k[b, s, h] * scale ) . v[b, s, h]
//   k_cache[b, h, j / 8, pos0 + t, j % 8] = k[b, t, h, j];  v_cache[b, h, pos0 + t, j] = v[b, t, h, j]
//
// qkv is the output of the Wqkv product, (B, T, 3, H, hd) fp16.  A workgroup takes 32 queries of one
// (b, h); its four wavefronts (WAVES) take every fourth block of 32 keys with an online softmax (fp32 scores,
// maximum and sum) and add up in LDS: 128 tokens of 40 heads are 160 workgroups with one block per
// wavefront, where 64 queries and a wavefront for 16 of them were 80 with eight blocks in a row.
//   S^T (32 keys x 32 queries) = K . Q^T   v_mfma_f32_32x32x16_f16, both operands straight from memory;
//                                          a lane holds the scores of ONE query
//   O^T (hd x 32) += V^T . P^T             P is in operand layout if the keys are taken in the order the
//                                          accumulator has them (0-3, 8-11 | 4-7, 12-15 inside 16); V goes
//                                          through wavefront-private LDS as it is and is read transposed
// K and V of the next block are requested when the registers of this one's are free, so no wavefront
// waits for another before the end.  A row of V is stored with its 16-byte pieces exchanged by the row's
// number, so that the eight rows of a transposed read use all banks.  The workgroup also copies its 32
// tokens' K and V rows into the caches (consecutive lanes take consecutive positions: 512 bytes of the
// packed key layout in a row).
//
// 40 heads of 128 and 128 tokens: 7.5 us (one wavefront for 16 queries and all their keys: 27); 32 heads
// and 777 tokens 30 us (215, and 75 with the library's attention and the copies into the caches).  Short
// prompts are bound by one block's chain of loads and exchanges, long ones by L2: each workgroup reads
// the keys and values before its 32 queries, 160 MB at 777 tokens.  Where short prompts make workgroups enough, two
// wavefronts do: of four, some have no block at all, yet hold their registers and LDS (16 sequences of 16 / 33 / 128
// tokens and 96 heads of 64: 9.4 / 17.4 / 38 us with four, 7.0 / 13.8 / 33 with two; of 128: 16 / 35 / 107 and 15 / 25 / 97).
//
// HD in {64, 128}.  Grid (H * ceil(T / 32), B), head fastest, WAVES * 64 threads: the workgroups of a head run
// on one die where the heads are a multiple of eight, the last queries (the most keys) first.
#pragma once
#include "common.hpp"
#include "gemm_mfma.hpp"

namespace dv {

constexpr int kPfQueries = 32;
constexpr int kPfKeys = 32;  // keys per step of a wavefront
constexpr int pf_row(int hd) { return hd + 4; }  // floats of a query's sums
constexpr size_t pf_lds(int hd, int waves) { return (size_t)waves * kPfQueries * pf_row(hd) * sizeof(float); }

// 16-byte piece p of row r of V in LDS: four rows of 32 columns are then on different banks.
template <int HD>
__device__ __forceinline__ int pf_piece(int r, int p) {
  return p ^ ((HD == 128 ? r & 3 : (r >> 1) & 1) << 2);
}

template <int HD, int WAVES>
__global__ __launch_bounds__(WAVES * 64, 2) void prefill_attn_kernel(
    const half_t* __restrict__ qkv, int T, int H, float scale, half_t* __restrict__ ctx, int ctx16 /* ctx on 16 bytes */,
    half_t* __restrict__ k_cache, half_t* __restrict__ v_cache, int pos0, int S) {
  typedef float acc_t __attribute__((ext_vector_type(16)));
  typedef short tr_t __attribute__((ext_vector_type(4)));
  typedef __attribute__((address_space(3))) tr_t* tr_ptr_t;
  constexpr int DT = HD / 16, VT = HD / 32, P8 = HD / 8, ROW = pf_row(HD);
  extern __shared__ __attribute__((aligned(16))) float sums[];  // [wavefront][query][ROW]; V blocks before
  __shared__ float s_m[WAVES][kPfQueries], s_l[WAVES][kPfQueries];
  static_assert(kPfKeys * HD * sizeof(half_t) <= kPfQueries * ROW * sizeof(float), "a block of V fits into the sums");
  const int tid = threadIdx.x, lane = tid & 63, l32 = lane & 31, hh = lane >> 5;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int h = blockIdx.x % H, b = blockIdx.y;
  const int q0 = ((int)((gridDim.x - 1) / H) - (int)(blockIdx.x / H)) * kPfQueries;
  const int64_t tstride = (int64_t)3 * H * HD;  // elements between consecutive tokens
  const half_t* Qb = qkv + (int64_t)b * T * tstride + (int64_t)h * HD;
  const half_t* Kb = Qb + (int64_t)H * HD;
  const half_t* Vb = Kb + (int64_t)H * HD;
  half_t* vs = reinterpret_cast<half_t*>(sums + (int64_t)wave * kPfQueries * ROW);

  // first blocks of K and V, the queries, and the rows for the caches
  half8_t kf[DT], vr[VT * 2], qf[DT];
  auto fetch_k = [&](int k0) {
    const half_t* kp = Kb + (int64_t)min(k0 + l32, T - 1) * tstride + hh * 8;
#pragma unroll
    for (int t = 0; t < DT; ++t) kf[t] = load8(kp + t * 16);
  };
  auto fetch_v = [&](int k0) {
#pragma unroll
    for (int i = 0; i < VT * 2; ++i) {
      const int at = i * 64 + lane;
      vr[i] = load8(Vb + (int64_t)min(k0 + at / P8, T - 1) * tstride + at % P8 * 8);
    }
  };
  const int q = q0 + l32, last = min(q0 + kPfQueries, T) - 1;
  {
    const half_t* qp = Qb + (int64_t)min(q, T - 1) * tstride + hh * 8;
#pragma unroll
    for (int t = 0; t < DT; ++t) qf[t] = load8(qp + t * 16);
  }
  int k0 = wave * kPfKeys;
  if (k0 <= last) {
    fetch_k(k0);
    fetch_v(k0);
  }
  if (k_cache != nullptr) {
    const int64_t bh = (int64_t)b * H + h;
#pragma unroll
    for (int i = 0; i < kPfQueries * P8 / (WAVES * 64); ++i) {
      const int at = i * (WAVES * 64) + tid, j8 = at / kPfQueries, t = q0 + at % kPfQueries;
      const int vt = q0 + at / P8, vj = at % P8;
      if (t < T && pos0 + t < S)
        store8(k_cache + ((bh * P8 + j8) * S + pos0 + t) * 8, load8(Kb + (int64_t)t * tstride + j8 * 8));
      if (vt < T && pos0 + vt < S)
        store8(v_cache + (bh * S + pos0 + vt) * HD + vj * 8, load8(Vb + (int64_t)vt * tstride + vj * 8));
    }
  }

  acc_t o[VT];
#pragma unroll
  for (int t = 0; t < VT; ++t)
#pragma unroll
    for (int i = 0; i < 16; ++i) o[t][i] = 0.f;
  float m = -1e30f, l = 0.f;  // l: this half wavefront's share
  const float sc = scale * 1.44269504088896340736f;
  const int j = lane & 15, tr_row = 4 * hh + (j >> 2), tr_col = 16 * ((lane >> 4) & 1) + (j & 3) * 4;
  for (; k0 <= last; k0 += WAVES * kPfKeys) {
    acc_t s;
#pragma unroll
    for (int i = 0; i < 16; ++i) s[i] = 0.f;
#pragma unroll
    for (int t = 0; t < DT; ++t) s = __builtin_amdgcn_mfma_f32_32x32x16_f16(kf[t], qf[t], s, 0, 0, 0);
#pragma unroll
    for (int i = 0; i < VT * 2; ++i) {
      const int at = i * 64 + lane, r = at / P8;
      store8(vs + r * HD + pf_piece<HD>(r, at % P8) * 8, vr[i]);
    }
    const int k1 = k0 + WAVES * kPfKeys;
    if (k1 <= last) {
      fetch_k(k1);
      fetch_v(k1);
    }
    __builtin_amdgcn_fence(__ATOMIC_SEQ_CST, "wavefront");
    __builtin_amdgcn_wave_barrier();
    const bool edge = k0 + kPfKeys - 1 > q0;
    float mx = -INFINITY;
#pragma unroll
    for (int i = 0; i < 16; ++i) {
      float x = s[i] * sc;
      if (edge && k0 + 8 * (i >> 2) + 4 * hh + (i & 3) > q) x = -INFINITY;
      s[i] = x;
      mx = fmaxf(mx, x);
    }
    mx = fmaxf(mx, __shfl_xor(mx, 32, kWave));
    const float m1 = fmaxf(m, mx), c = __builtin_amdgcn_exp2f(m - m1);
    m = m1;
    l *= c;
#pragma unroll
    for (int i = 0; i < 16; ++i) {
      const float p = __builtin_amdgcn_exp2f(s[i] - m1);
      s[i] = p;
      l += p;
    }
#pragma unroll
    for (int t = 0; t < VT; ++t)
#pragma unroll
      for (int i = 0; i < 16; ++i) o[t][i] *= c;
#pragma unroll
    for (int ks = 0; ks < 2; ++ks) {
      half8_t pf;
#pragma unroll
      for (int e = 0; e < 8; ++e) pf[e] = (half_t)s[8 * ks + e];
#pragma unroll
      for (int t = 0; t < VT; ++t) {
        union {
          tr_t part[2];
          half8_t all;
        } w;
#pragma unroll
        for (int u = 0; u < 2; ++u) {
          const int r = ks * 16 + u * 8 + tr_row, col = t * 32 + tr_col;
          w.part[u] = __builtin_amdgcn_ds_read_tr16_b64_v4i16(
              (tr_ptr_t)(vs + r * HD + pf_piece<HD>(r, col >> 3) * 8 + (col & 7)));
        }
        o[t] = __builtin_amdgcn_mfma_f32_32x32x16_f16(w.all, pf, o[t], 0, 0, 0);
      }
    }
    __builtin_amdgcn_fence(__ATOMIC_SEQ_CST, "wavefront");  // the next block of V is stored over this one
    __builtin_amdgcn_wave_barrier();
  }
  l += __shfl_xor(l, 32, kWave);

  // this wavefront's sums over its last block of V; the wavefronts meet here for the first time
  float* mine = sums + ((int64_t)wave * kPfQueries + l32) * ROW;
#pragma unroll
  for (int t = 0; t < VT; ++t)
#pragma unroll
    for (int i = 0; i < 16; i += 4)
      *reinterpret_cast<float4_t*>(mine + t * 32 + 2 * i + 4 * hh) = float4_t{o[t][i], o[t][i + 1], o[t][i + 2], o[t][i + 3]};
  if (hh == 0) {
    s_m[wave][l32] = m;
    s_l[wave][l32] = l;
  }
  __syncthreads();
#pragma unroll
  for (int i = 0; i < kPfQueries * P8 / (WAVES * 64); ++i) {
    const int at = i * (WAVES * 64) + tid, qq = at / P8, d = at % P8 * 8;
    float mm = s_m[0][qq], den = 0.f, v[8] = {0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int w = 1; w < WAVES; ++w) mm = fmaxf(mm, s_m[w][qq]);
#pragma unroll
    for (int w = 0; w < WAVES; ++w) {
      const float e = __builtin_amdgcn_exp2f(s_m[w][qq] - mm);
      const float* part = sums + ((int64_t)w * kPfQueries + qq) * ROW + d;
      den = __builtin_fmaf(s_l[w][qq], e, den);
#pragma unroll
      for (int k = 0; k < 8; ++k) v[k] = __builtin_fmaf(part[k], e, v[k]);
    }
    if (q0 + qq >= T) break;
    const float inv = den > 0.f ? 1.f / den : 0.f;
    half_t* dst = ctx + ((int64_t)b * T + q0 + qq) * H * HD + (int64_t)h * HD + d;
    half8_t out;
#pragma unroll
    for (int k = 0; k < 8; ++k) out[k] = (half_t)(v[k] * inv);
    if (ctx16) {
      store8(dst, out);
    } else {
#pragma unroll
      for (int k = 0; k < 8; ++k) dst[k] = out[k];
    }
  }
}

}  // namespace dv
