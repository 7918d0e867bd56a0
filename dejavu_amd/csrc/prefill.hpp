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
// the keys and values before its 32 queries, 160 MB at 777 tokens (prefill_tiles_kernel, below, takes those of 1000 on,
// 800 with 40 heads; the line is prefill_in_tiles').  Where short prompts make workgroups enough, two
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

// The same for long prompts, 128 queries a workgroup: eight wavefronts, two groups of four that take the key tiles of 64 in turn, the even and
// the odd ones, with K and V through LDS for all queries of the group (a quarter of the reads from L2), and whose sums meet at the end.  The
// last queries' chain of tiles is half as long as one group's, and a SIMD has two wavefronts, with 256 registers each.  Bound by a tile's chain:
// LDS reads, two products, the softmax.  us, 32 queries a workgroup / this: 32 heads of 128, 777 / 1000 / 2000 / 4000 / 8192 tokens 29.9 / 27.1, 37.7 / 32.5, 105 / 70,
// 353 / 227, 1337 / 806; 40 heads 777 / 2000 32.6 / 27.6, 124 / 90; 16 sequences of 777 tokens 376 / 288; 96 heads of 64, 2000 tokens 162 / 102.
// Grid (H * ceil(T / 128), B), head fastest, the last queries first.
constexpr int kPtQueries = 128, kPtKeys = 64;
template <int HD>
constexpr size_t pt_group = (size_t)kPtKeys * (HD + 8 + HD) * sizeof(half_t);  // a group's tiles of K and V
template <int HD>
constexpr size_t pt_lds = 2 * pt_group<HD> > (size_t)256 * (HD / 2 + 2) * 4 ? 2 * pt_group<HD> : (size_t)256 * (HD / 2 + 2) * 4;

template <int HD>
__global__ __launch_bounds__(512, HD == 64 ? 4 : 2) void prefill_tiles_kernel(const half_t* __restrict__ qkv, int T, int H, float scale, half_t* __restrict__ ctx,
                                                            half_t* __restrict__ k_cache, half_t* __restrict__ v_cache, int pos0, int S) {
  typedef float acc_t __attribute__((ext_vector_type(16)));
  typedef short tr_t __attribute__((ext_vector_type(4)));
  typedef __attribute__((address_space(3))) tr_t* tr_ptr_t;
  constexpr int DT = HD / 16, VT = HD / 32, P8 = HD / 8, DL = HD + 8;
  extern __shared__ __attribute__((aligned(16))) unsigned char tiles[];
  const int group = __builtin_amdgcn_readfirstlane(threadIdx.x >> 8);
  half_t* const ks = reinterpret_cast<half_t*>(tiles + group * pt_group<HD>);
  half_t* const vs = ks + kPtKeys * DL;
  const int tid = threadIdx.x & 255, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6), l32 = lane & 31, hh = lane >> 5;
  const int h = blockIdx.x % H, b = blockIdx.y;
  const int q0 = ((int)((gridDim.x - 1) / H) - (int)(blockIdx.x / H)) * kPtQueries;
  const int64_t tstride = (int64_t)3 * H * HD;
  const half_t* Qb = qkv + (int64_t)b * T * tstride + (int64_t)h * HD;
  const half_t* Kb = Qb + (int64_t)H * HD;
  const half_t* Vb = Kb + (int64_t)H * HD;
  const int w0 = q0 + wave * 32, q = w0 + l32, last = min(q0 + kPtQueries, T) - 1;

  constexpr int PV = kPtKeys * P8 / 256;  // 16-byte pieces of a tile per thread
  half8_t kr[PV], vr[PV], qf[DT];
  auto fetch = [&](int k0) {  // (past the last token: that one again, whose weights are zero)
#pragma unroll
    for (int i = 0; i < PV; ++i) {
      const int at = i * 256 + tid;
      const int64_t row = (int64_t)min(k0 + at / P8, T - 1) * tstride + at % P8 * 8;
      kr[i] = load8(Kb + row);
      vr[i] = load8(Vb + row);
    }
  };
  {
    const half_t* qp = Qb + (int64_t)min(q, T - 1) * tstride + hh * 8;
#pragma unroll
    for (int t = 0; t < DT; ++t) qf[t] = load8(qp + t * 16);
  }
  fetch(group * kPtKeys);
  if (k_cache != nullptr) {
    const int64_t bh = (int64_t)b * H + h;
#pragma unroll
    for (int i = 0; i < kPtQueries * P8 / 512; ++i) {
      const int at = i * 512 + threadIdx.x, j8 = at / kPtQueries, t = q0 + at % kPtQueries;
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
  for (int b0 = 0; b0 <= last; b0 += 2 * kPtKeys) {
    const int k0 = b0 + group * kPtKeys;  // (a group may be past the last tile)
    __syncthreads();
#pragma unroll
    for (int i = 0; i < PV; ++i) {
      const int at = i * 256 + tid, r = at / P8;
      store8(ks + r * DL + at % P8 * 8, kr[i]);
      store8(vs + r * HD + pf_piece<HD>(r, at % P8) * 8, vr[i]);
    }
    __syncthreads();
    if (k0 + 2 * kPtKeys <= last) fetch(k0 + 2 * kPtKeys);
    if (k0 > w0 + 31) continue;  // nothing that this wavefront's queries see
    // Queries that begin where the tile does see its first 32 keys only.  The weights of the others are zeros, but zero times a value
    // that is not finite is none: they multiply the first 32 values once more.  (Branches around the halves of the products: 3 % more, 2000 to 8192 tokens.)
    const half_t* const vs32 = k0 < w0 ? vs : vs - 32 * HD;  // (pf_piece is the same 32 rows on)
    acc_t s[2];
#pragma unroll
    for (int kt = 0; kt < 2; ++kt) {
#pragma unroll
      for (int i = 0; i < 16; ++i) s[kt][i] = 0.f;
#pragma unroll
      for (int t = 0; t < DT; ++t)
        s[kt] = __builtin_amdgcn_mfma_f32_32x32x16_f16(load8_lds(ks + (kt * 32 + l32) * DL + t * 16 + hh * 8), qf[t], s[kt], 0, 0, 0);
    }
    const bool edge = k0 + kPtKeys - 1 > w0;
    float mx = -INFINITY;
#pragma unroll
    for (int kt = 0; kt < 2; ++kt)
#pragma unroll
      for (int i = 0; i < 16; ++i) {
        float x = s[kt][i] * sc;
        if (edge && k0 + kt * 32 + 8 * (i >> 2) + 4 * hh + (i & 3) > q) x = -INFINITY;
        s[kt][i] = x;
        mx = fmaxf(mx, x);
      }
    mx = fmaxf(mx, __shfl_xor(mx, 32, kWave));
    const float m1 = fmaxf(m, mx), c = __builtin_amdgcn_exp2f(m - m1);
    m = m1;
    l *= c;
#pragma unroll
    for (int kt = 0; kt < 2; ++kt)
#pragma unroll
      for (int i = 0; i < 16; ++i) {
        const float p = __builtin_amdgcn_exp2f(s[kt][i] - m1);
        s[kt][i] = p;
        l += p;
      }
    if (__any(c != 1.f)) {  // a new maximum somewhere: rare after the first tiles
#pragma unroll
      for (int t = 0; t < VT; ++t)
#pragma unroll
        for (int i = 0; i < 16; ++i) o[t][i] *= c;
    }
#pragma unroll
    for (int ks4 = 0; ks4 < 4; ++ks4) {
      half8_t pf;
#pragma unroll
      for (int e = 0; e < 8; ++e) pf[e] = (half_t)s[ks4 >> 1][8 * (ks4 & 1) + e];
#pragma unroll
      for (int t = 0; t < VT; ++t) {
        union {
          tr_t part[2];
          half8_t all;
        } w;
#pragma unroll
        for (int u = 0; u < 2; ++u) {
          const int r = ks4 * 16 + u * 8 + tr_row, col = t * 32 + tr_col;
          w.part[u] = __builtin_amdgcn_ds_read_tr16_b64_v4i16((tr_ptr_t)((ks4 < 2 ? vs : vs32) + r * HD + pf_piece<HD>(r, col >> 3) * 8 + (col & 7)));
        }
        o[t] = __builtin_amdgcn_mfma_f32_32x32x16_f16(w.all, pf, o[t], 0, 0, 0);
      }
    }
  }
  float* mg = reinterpret_cast<float*>(tiles) + tid;  // [value][thread of a group]
  __syncthreads();
  if (group == 1) {
#pragma unroll
    for (int t = 0; t < VT; ++t)
#pragma unroll
      for (int i = 0; i < 16; ++i) mg[(t * 16 + i) * 256] = o[t][i];
    mg[VT * 16 * 256] = m;
    mg[(VT * 16 + 1) * 256] = l;
  }
  __syncthreads();
  if (group == 1) return;
  const float mo = mg[VT * 16 * 256], m1 = fmaxf(m, mo), c0 = __builtin_amdgcn_exp2f(m - m1), c1 = __builtin_amdgcn_exp2f(mo - m1);
  l = __builtin_fmaf(mg[(VT * 16 + 1) * 256], c1, l * c0);
  l += __shfl_xor(l, 32, kWave);
  if (q >= T) return;
  const float inv = l > 0.f ? 1.f / l : 0.f;
  half_t* dst = ctx + ((int64_t)b * T + q) * H * HD + (int64_t)h * HD;
#pragma unroll
  for (int t = 0; t < VT; ++t)
#pragma unroll
    for (int i = 0; i < 16; i += 4) {
      half4_t out;
#pragma unroll
      for (int e = 0; e < 4; ++e) out[e] = (half_t)(__builtin_fmaf(mg[(t * 16 + i + e) * 256], c1, o[t][i + e] * c0) * inv);
      *reinterpret_cast<half4_t*>(dst + t * 32 + 2 * i + 4 * hh) = out;
    }
}

}  // namespace dv
