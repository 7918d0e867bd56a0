// Causal softmax attention of a portion of a prompt on the matrix cores (bf16 operands, fp32 scores and sums):
// grouped key/value heads, different query/key and value sizes, optional sliding window or chunks, bias by distance,
// sink and output gate.
//
// A workgroup takes 128 queries of one head, a wave 32 of them.  Scores are computed transposed (keys x queries),
// so a lane holds the scores of ONE query: the softmax is lane-local but for one exchange between the half waves,
// and the weights are already in the operand layout of the second product when its keys are taken in the order
// the accumulator has them (key permutation 0-3, 8-11 | 4-7, 12-15 inside 16).  Values stay in LDS as they are in memory and
// are read transposed; pairing keys by hand took eight 4-byte stores for each 16-byte one, and with the sums rescaled for
// every tile, not only where a maximum has grown, 32 heads of 128 and 2048 tokens took 98 us instead of 89, 4096 tokens 331
// instead of 304.  Two buffers with one barrier a tile were slower (96).  Bound by the chain of a tile: LDS reads, two products, the
// softmax.  So two groups of four waves share a query tile (where two_groups says), the even and the odd key tiles: the last queries' chain is half as long, a SIMD
// has two waves whatever the grid (alone a wave takes 328 registers, one to a SIMD; two in a group's kernel 238), and a long workgroup and
// a short one make the same 17 steps on every compute unit.  us, one group / two, 32 heads of 128: 300 / 777 / 2048 / 4096 / 8192
// tokens 16.5 / 13.6, 35.1 / 25.7, 92 / 69, 308 / 217, 1172 / 713, a window of 1024 and 8 key heads 91.5 / 64.7 (2048), 352 / 251 (8192); 16 heads 33.6 / 24.3 (777),
// 79.5 / 53.8 (2048).
#pragma once
#include "attn_rows.hpp"

namespace dv {

constexpr int kTileQ = 128, kTileK = 64;

// DT: query/key tiles of 16, VT: value tiles of 32.  Grid: H * ceil(n / 128), head fastest, last queries first.
// KS: groups of four waves that take a query tile's key tiles in turn, each with its own softmax; their sums meet at the end.
template <int DT, int VT, int KS>
__global__ __launch_bounds__(256 * KS) void attn_tiles_kernel(AttnArgs a, int keys /* rows behind k and v */) {
  typedef short tr_t __attribute__((ext_vector_type(4)));
  typedef __attribute__((address_space(3))) tr_t* tr_ptr_t;
  constexpr int DL = DT * 16 + 8, VL = VT * 32;  // LDS row lengths
  constexpr size_t KB = kTileK * DL * sizeof(bf16_t), VB = kTileK * VL * sizeof(bf16_t), MERGE = KS > 1 ? (size_t)(KS - 1) * 256 * (VT * 16 + 2) * 4 : 0;
  __shared__ __attribute__((aligned(16))) unsigned char smem[KS * (KB + VB) > MERGE ? KS * (KB + VB) : MERGE];
  __shared__ float biases[KS][kTileQ + kTileK];
  const int group = KS > 1 ? __builtin_amdgcn_readfirstlane(threadIdx.x >> 8) : 0;
  bf16_t* const ks = reinterpret_cast<bf16_t*>(smem + group * (KB + VB));
  bf16_t* const vs = reinterpret_cast<bf16_t*>(smem + group * (KB + VB) + KB);
  float* const rs = biases[group];  // biases of a tile: entry i is the distance off + q0 - k0 - (kTileK - 1) + i
  const int tid = threadIdx.x & 255, lane = tid & 63, wave = tid >> 6, l32 = lane & 31, hh = lane >> 5;
  const int head = blockIdx.x % a.H, g = head / (a.H / a.G);
  const int nblk = (a.n + kTileQ - 1) / kTileQ;
  const int q0 = (nblk - 1 - (int)(blockIdx.x / a.H)) * kTileQ;
  const int off = a.pos_host - a.base;  // key slot of query 0
  const bf16_t* K = reinterpret_cast<const bf16_t*>(a.k) + (int64_t)g * a.k_head;
  const bf16_t* V = reinterpret_cast<const bf16_t*>(a.v) + (int64_t)g * a.v_head;

  const int qi = q0 + wave * 32 + l32;  // this lane's query
  bf16x8_t qf[DT];
  {
    const bf16_t* q = reinterpret_cast<const bf16_t*>(a.q) + (int64_t)(qi < a.n ? qi : 0) * a.ldq + (int64_t)head * a.dim_s;
#pragma unroll
    for (int t = 0; t < DT; ++t) {
      const int d = t * 16 + hh * 8;
      uint4_t z = {0, 0, 0, 0};
      if (qi < a.n && d < a.dim_s) z = *reinterpret_cast<const uint4_t*>(q + d);
      qf[t] = __builtin_bit_cast(bf16x8_t, z);
    }
  }
  const int qslot = off + qi;
  auto oldest_slot = [&](int q) { return max(0, oldest_key(a, a.pos_host + q) - a.base); };
  const int klo = oldest_slot(min(qi, a.n - 1));
  const int wklo = __builtin_amdgcn_readfirstlane(klo);
  const int wkhi = oldest_slot(min(q0 + wave * 32 + 31, a.n - 1));
  const int wlo = off + q0 + wave * 32, whi = min(off + q0 + wave * 32 + 31, off + a.n - 1);  // slots of the wave
  const int bhi = min(off + q0 + kTileQ - 1, off + a.n - 1);
  const int first = oldest_slot(q0) / kTileK * kTileK;
  const float* rel = a.rel ? a.rel + (int64_t)head * a.rel_len : nullptr;
  constexpr float kLog2e = 1.44269504088896340736f;
  const float rel_far = rel ? rel[a.rel_len - 1] * kLog2e : 0.f;
  float rr = 0.f;
  const int last = bhi;

  constexpr int KV = (kTileK * DT * 2 + 255) / 256;       // 16-byte loads of K per thread
  constexpr int VV = kTileK * VT * 4 / 256;               // and of V
  // 16-byte piece p of row r of V: the rows of a transposed read are on different banks
  auto piece = [](int r, int p) { return p ^ ((VT == 1 ? 0 : VT == 2 ? (r >> 1) & 1 : r & 3) << 2); };
  uint4_t kr[KV], vr[VV];
  auto fetch = [&](int k0) {
    if (rel) rr = rel[min(max(off + q0 - k0 - (kTileK - 1) + tid, 0), a.rel_len - 1)] * kLog2e;
    // past the last key the weights are zero; past the last channel the queries are, or nothing is stored
#pragma unroll
    for (int i = 0; i < KV; ++i) {
      const int at = i * 256 + tid, r = at / (DT * 2), d = at % (DT * 2) * 8;
      kr[i] = *reinterpret_cast<const uint4_t*>(K + (int64_t)min(k0 + r, keys - 1) * a.ldk + min(d, a.dim_s - 8));
    }
#pragma unroll
    for (int i = 0; i < VV; ++i) {
      const int at = i * 256 + tid, r = at / (VT * 4), d = min(at % (VT * 4) * 8, a.vdim_s - 8);
      vr[i] = *reinterpret_cast<const uint4_t*>(V + (int64_t)min(k0 + r, keys - 1) * a.ldv + d);
    }
  };
  auto put = [&]() {
    if (rel && tid < kTileQ + kTileK) rs[tid] = rr;
#pragma unroll
    for (int i = 0; i < KV; ++i) {
      const int at = i * 256 + tid, r = at / (DT * 2), d = at % (DT * 2) * 8;
      if (r < kTileK) *reinterpret_cast<uint4_t*>(&ks[r * DL + d]) = kr[i];
    }
#pragma unroll
    for (int i = 0; i < VV; ++i) {
      const int at = i * 256 + tid, r = at / (VT * 4);
      *reinterpret_cast<uint4_t*>(&vs[r * VL + piece(r, at % (VT * 4)) * 8]) = vr[i];
    }
  };

  float16_t o[VT];
#pragma unroll
  for (int t = 0; t < VT; ++t)
#pragma unroll
    for (int i = 0; i < 16; ++i) o[t][i] = 0.f;
  float m = -1e30f, l = 0.f;  // l: this half wave's share
  const float sc = a.scale * kLog2e;
  const int tr_row = 4 * hh + ((lane & 15) >> 2), tr_col = 16 * ((lane >> 4) & 1) + (lane & 3) * 4;

  const int mine = first + group * kTileK;
  fetch(mine);
  for (int b0 = first; b0 <= last; b0 += KS * kTileK) {
    const int k0 = b0 + group * kTileK;  // (a group may be past the last tile)
    __syncthreads();
    put();
    __syncthreads();
    if (k0 + KS * kTileK <= last) fetch(k0 + KS * kTileK);
    const bool seen = k0 <= whi && k0 + kTileK - 1 >= wklo;
    if (!seen) continue;
    float16_t s[2];
#pragma unroll
    for (int kt = 0; kt < 2; ++kt) {
#pragma unroll
      for (int i = 0; i < 16; ++i) s[kt][i] = 0.f;
#pragma unroll
      for (int t = 0; t < DT; ++t) {
        const bf16x8_t kf = *reinterpret_cast<const bf16x8_t*>(&ks[(kt * 32 + l32) * DL + t * 16 + hh * 8]);
        s[kt] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(kf, qf[t], s[kt], 0, 0, 0);
      }
    }
    const bool full = k0 + kTileK - 1 <= wlo && k0 >= wkhi;
    if (rel && wlo - (k0 + kTileK - 1) < a.rel_len - 1) {
      const float* rp = rs + wave * 32 + l32 + kTileK - 1 - 4 * hh;
#pragma unroll
      for (int kt = 0; kt < 2; ++kt)
#pragma unroll
        for (int i = 0; i < 16; ++i) s[kt][i] = __builtin_fmaf(s[kt][i], sc, rp[-(kt * 32 + 8 * (i >> 2) + (i & 3))]);
    } else {  // no bias, or one for all
#pragma unroll
      for (int kt = 0; kt < 2; ++kt)
#pragma unroll
        for (int i = 0; i < 16; ++i) s[kt][i] = __builtin_fmaf(s[kt][i], sc, rel_far);
    }
    float mx = -INFINITY;
#pragma unroll
    for (int kt = 0; kt < 2; ++kt)
#pragma unroll
      for (int i = 0; i < 16; ++i) {
        float x = s[kt][i];
        if (!full) {
          const int key = k0 + kt * 32 + 8 * (i >> 2) + 4 * hh + (i & 3);
          if (key > qslot || key < klo) x = -INFINITY;
        }
        s[kt][i] = x;
        mx = fmaxf(mx, x);
      }
    mx = fmaxf(mx, __shfl_xor(mx, 32, kWave));
    const float m1 = fmaxf(m, mx);
    const float c = __builtin_amdgcn_exp2f(m - m1);
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
      bf16x8_t pf;
#pragma unroll
      for (int e = 0; e < 8; ++e) pf[e] = (bf16_t)s[ks4 >> 1][8 * (ks4 & 1) + e];
#pragma unroll
      for (int t = 0; t < VT; ++t) {
        union {
          tr_t part[2];
          bf16x8_t all;
        } w;
#pragma unroll
        for (int u = 0; u < 2; ++u) {
          const int r = ks4 * 16 + u * 8 + tr_row, col = t * 32 + tr_col;
          w.part[u] = __builtin_amdgcn_ds_read_tr16_b64_v4i16((tr_ptr_t)(&vs[r * VL + piece(r, col >> 3) * 8 + (col & 7)]));
        }
        o[t] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(w.all, pf, o[t], 0, 0, 0);
      }
    }
  }
  if constexpr (KS > 1) {
    float* mg = reinterpret_cast<float*>(smem) + tid;
    __syncthreads();
    if (group > 0) {
      mg += (group - 1) * 256 * (VT * 16 + 2);
#pragma unroll
      for (int t = 0; t < VT; ++t)
#pragma unroll
        for (int i = 0; i < 16; ++i) mg[(t * 16 + i) * 256] = o[t][i];
      mg[VT * 16 * 256] = m;
      mg[(VT * 16 + 1) * 256] = l;
    }
    __syncthreads();
    if (group > 0) return;
#pragma unroll
    for (int k = 1; k < KS; ++k, mg += 256 * (VT * 16 + 2)) {
      const float mo = mg[VT * 16 * 256], m1 = fmaxf(m, mo), c0 = __builtin_amdgcn_exp2f(m - m1), c1 = __builtin_amdgcn_exp2f(mo - m1);
      m = m1;
      l = __builtin_fmaf(mg[(VT * 16 + 1) * 256], c1, l * c0);
#pragma unroll
      for (int t = 0; t < VT; ++t)
#pragma unroll
        for (int i = 0; i < 16; ++i) o[t][i] = __builtin_fmaf(mg[(t * 16 + i) * 256], c1, o[t][i] * c0);
    }
  }
  l += __shfl_xor(l, 32, kWave);
  if (qi >= a.n) return;
  m *= 0.69314718055994530942f;  // back to natural units
  float c;
  const float f = attn_factor<bf16_t>(a, qi, head, m, l, &c) * c;
  bf16_t* out = reinterpret_cast<bf16_t*>(a.out) + ((int64_t)qi * a.H + head) * a.vdim_s;
#pragma unroll
  for (int t = 0; t < VT; ++t)
#pragma unroll
    for (int i = 0; i < 16; i += 4) {
      const int d = t * 32 + 2 * i + 4 * hh;
      if (d < a.vdim_s) {
        bf16x4_t w = {(bf16_t)(o[t][i] * f), (bf16_t)(o[t][i + 1] * f), (bf16_t)(o[t][i + 2] * f), (bf16_t)(o[t][i + 3] * f)};
        *reinterpret_cast<bf16x4_t*>(out + d) = w;
      }
    }
}

}  // namespace dv
