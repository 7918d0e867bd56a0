// Products of up to a few hundred rows with a weight on the matrix cores where the weight's bytes bound them, not the
// operations: out(m, n) = sum_k W[rows(m), k] X[n, k], 16-bit operands, fp32 sums.
//
// A tile is MB rows of W by NB rows of X.  Both operands go from memory straight into a ring of ST LDS slots (no registers
// on the way) ST - 1 chunks of KC columns ahead of their use: a wave's load covers 256 or 128 contiguous bytes of a row,
// where loads in the matrix instruction's own layout cover 64 (a plain read of 22016 x 4096 in these pieces: 6.0, 5.2 and
// 4.3 TB/s).  Where the tiles are fewer than the chip's workgroups, K is split over the grid and a second launch adds the
// sums up; adding them up in the first one, by the workgroup that ends last, costs more (each hand-over between compute
// dies 5 us, fences 40 us).
//
// 47 rows by 4096 x 4096 / 4096 x 11008 / 22016 x 4096: 11.1 / 22 / 33.5 us (loads in operand layout, 24 at a time: 24 / 47 /
// 74); 16 rows 10.8 / 20 / 31.8 us (13 / 43 / 51).  Bound by the stream: 33.5 us are 5.4 TB/s beside a plain read's 6.
#pragma once
#include "common.hpp"

namespace dv {

typedef const __attribute__((address_space(1))) void* global_ptr_t;
typedef __attribute__((address_space(3))) void* lds_ptr_t;
typedef unsigned ring_word_t __attribute__((ext_vector_type(4)));  // eight elements

// Waits until at most N of this wave's loads are still on their way.
template <int N>
__device__ __forceinline__ void wait_loads() {
  asm volatile("s_waitcnt vmcnt(%0)" ::"i"(N) : "memory");
}

template <typename T>
__device__ __forceinline__ float4_t ring_mfma(ring_word_t w, ring_word_t x, float4_t acc) {
  typedef T vec_t __attribute__((ext_vector_type(8)));
  const vec_t a = __builtin_bit_cast(vec_t, w), b = __builtin_bit_cast(vec_t, x);
  if constexpr (__is_same(T, half_t)) return __builtin_amdgcn_mfma_f32_16x16x32_f16(a, b, acc, 0, 0, 0);
  else return __builtin_amdgcn_mfma_f32_16x16x32_bf16(a, b, acc, 0, 0, 0);
}

template <typename T>
struct RingOperands {
  const T* X;
  int64_t ldx;
  const T* W;
  int64_t ldw;
  int n, M, K;  // K, ldx, ldw % 8 == 0, X and W on 16-byte boundaries
};

// Rows 0 .. M - 1 of the weight.
struct PlainRows {
  static constexpr bool kPastCaches = true;
  static constexpr int kMostCols = 256;  // the widest tile that is launched for them
  __device__ __forceinline__ int64_t operator()(int m) const { return m; }
};

// As the output of a product: the splits' sums as rows of M floats (M % 4 == 0), one split after the other, for a launch that adds them up
// with what follows, a workgroup a row.
struct RingRowParts {
  float* part;
  int64_t rows;
  int M;
  __device__ __forceinline__ void operator()(int m, int n, const float4_t& v) const {
    *reinterpret_cast<float4_t*>(part + (blockIdx.z * rows + n) * M + m) = v;
  }
};

struct RingPlan {
  int mb, nb;        // tile: rows of W, rows of X
  int rows, cols;    // tiles
  int splits;        // of K
  size_t workspace_bytes() const { return splits > 1 ? (size_t)splits * rows * cols * mb * nb * sizeof(float) : 0; }
};

// Up to 64 rows: tiles are as narrow as the rows allow and of 64 weight rows for small weights.  Beyond, taller ones fetch X less
// often and split K into a round of workgroups with less left over (us, 64 weight rows a tile against 128, 47 rows: 6144 x 4096 17.4 /
// 14.3, 8512 x 4096 25 / 18.7, 12288 x 4096 25 / 22.2, but 4096 x 4096 11.1 / 12.1 and 6400 x 2048 12.0 / 12.6; 30 rows: 8512 x 4096 21 / 17.5,
// 22016 x 4096 39 / 31.8, 11264 x 2048 15.6 / 12.7); of 33 to 64 rows with more than a round of 64, 96 (22016 x 4096: 33.5 us, 128
// weight rows 34.2, 64 51), but 128 where these still make one round (32768 x 4096: 57 / 43.7).
// K is split until there are about as many workgroups as compute units (4096 x 11008 with 47 rows: 1, 2, 4, 8 splits of 64
// weight rows take 52, 32, 24.5, 27 us; 8512 x 4096 3 and 4 splits of 128, 201 and 268 workgroups, 18.7 and 26); the narrowest tiles'
// workgroups are small, so they go on to two per unit.
// More rows: 128 rows of W, so that X is fetched less often (5120 x 20480 with 96 rows: 53 us, 60 with 64 rows of W),
// where that leaves 32 tiles and K is long enough to split (but 64 where these make one round and K is short: 16384 x 4096 with
// 72 / 128 rows 41.5 / 45 us, in two splits 47.5 / 48; and for small weights, of whose K tiles of 128 have an eighth each: 4096 x 4096 with 72 / 100 /
// 128 rows 13.5 / 14.0 / 14.5, 16.9 / 17.9 / 18.2, a prompt of 68 to 127 tokens with such a product a layer 1 to 2 % less; 4096 x
// 4608 / 5632 1.04 / 1.00 to 1.04 times the speed, but 6144 0.98 to 1.01, 6656 to 8064 0.93 to 1.00); 192 where they fill the chip better (20480 x 5120 with 96 rows:
// 107 tiles in 2 splits take 53 us, 160 tiles of 128 rows 59) or spare a round of it (36864 x 12288 with 128 rows: 192
// tiles against 288).  257 to 384 rows are two tiles of 192, not of 256 (320 rows: QKV of 24 heads of 9216 97 against 147 us, of
// 32 heads of 12288 141 against 195).
// A split has at least 256 columns.
// The row counts 14336 and 16384 of these are what 224 and 256 of `units`, the device's compute units, take in a round.
inline RingPlan plan_ring(int n, int M, int K, int units) {
  RingPlan p;
  p.nb = n <= 16 ? 16 : n <= 32 ? 32 : n <= 64 ? 64 : n <= 128 ? 128 : n <= 192 || (n > 256 && n <= 384) ? 192 : 256;
  auto lay = [&](int mb) {
    p.mb = mb;
    p.rows = (M + mb - 1) / mb;
    p.cols = (n + p.nb - 1) / p.nb;
    const int64_t tiles = (int64_t)p.rows * p.cols;
    int64_t s = p.nb == 16 ? (tiles >= units ? 1 : tiles >= units / 2 ? 4 : 8) : (p.nb <= 64 && mb == 64 ? units * 9 / 8 : units) / tiles;
    if (s > K / 256) s = K / 256;
    p.splits = (int)(s < 1 ? 1 : s > 8 ? 8 : s);
    return (int64_t)p.splits * tiles;
  };
  if (p.nb <= 64) {
    const bool taller = M >= units * 24 && K >= (p.nb == 32 ? 2048 : 4096);
    if (p.nb == 16) lay(32);
    else if (p.nb == 64 && M >= units * 64) lay((M + 95) / 96 > units && (M + 127) / 128 <= units ? 128 : 96);
    else lay(taller && (p.nb == 32 || M <= units * 60) ? 128 : 64);  // (33 to 64 rows: not where 64 make a round)
  } else if (M < 32 * 128 || K < 2048 || (p.nb == 128 && K <= 4096 && M > units * 56 && M <= units * 64) ||
             (p.nb == 128 && K >= 4096 && K < 6144 && M <= units * 16)) {
    lay(64);
  } else {
    const bool tall = p.nb < 256 && K >= 4096;
    const int64_t groups = lay(128);
    if (tall) {
      const int64_t more = lay(192), rounds = (groups + units - 1) / units, tall_rounds = (more + units - 1) / units;
      const bool fuller = groups <= units ? more <= units && more * 10 > groups * 11 : tall_rounds * 192 < rounds * 128;
      if (!fuller) lay(128);
    }
  }
  return p;
}

// NT_W: the weight bypasses the caches: worth 10 % where the rows of X are few and the weight comes from memory (128 rows by
// 20480 x 5120 and its like, of a prompt's layer: 235 us the layer, 223), but a small weight (17 rows by 1024 x 5120: 7.2, 7.7
// us) and the chosen heads' rows of a block (192 rows a tile, 128 of X, 9216 columns: 39.2, 40.7) stay in the last cache from
// one call to the next.  These rows also gain nothing by beginning at different columns (kPastCaches of the rows).
// One tile: rows of W from m0 on, columns n0 .. of the n that `cols` makes rows of X of.  Splits of K: blockIdx.z of gridDim.z.
// Out: called with (m, row of X, sums of rows m .. m + 3), m % 4 == 0, m < M.
// part: with several splits, this tile's sums [value][thread] of this split.
template <typename T, int MB, int NB, int KC, int ST, int WM, int WN, bool NT_W, bool ROUND, typename Rows, typename Cols, typename Out>
__device__ __forceinline__ void ring_tile(const RingOperands<T>& a, const Rows& rows, const Cols& cols, const Out& out, int m0, int n0, int n_cols,
                                          float4_t* __restrict__ part, unsigned char* slots) {
  constexpr int WAVES = WM * WN, THREADS = WAVES * 64;
  constexpr int CH = KC / 8;               // 16-byte pieces of a row's chunk
  constexpr int RPL = 64 / CH;             // rows per load of a wave
  constexpr int SWAP = (CH < 16 ? CH : 16) - 1;
  constexpr int LI = (MB + NB) / RPL / WAVES;
  constexpr int SLOT = (MB + NB) * KC * 2;
  constexpr int RT = MB / WM / 16, NT = NB / WN / 16, KS = KC / 32;
  static_assert((MB + NB) % (RPL * WAVES) == 0 && MB % RPL == 0, "loads do not tile");
  const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int wm = wave % WM, wn = wave / WM, l16 = lane & 15, g = lane >> 4;
  const int nch = (a.K + KC - 1) / KC;
  const int c0 = nch * blockIdx.z / gridDim.z, len = nch * (blockIdx.z + 1) / gridDim.z - c0;
  // ROUND: the columns are taken in parts, and workgroups begin with different ones and go round: all of them at the same
  // column, of rows that are a power of two apart, wait for the same few channels of the memory.  The parts' sums are added in
  // the columns' order (two: in any) wherever the workgroup began, so a row's result does not depend on its place.  (A different
  // chunk for each instead: the same time, other bits.)
  // us without and with: 47 rows by 22016 x 4096 37.7, 32.2; 22016 x 6144 60.0, 47.1; 16 rows by 22016 x 4096 37.3, 31.8; 100 rows by
  // 16384 x 4096 40.2, 35.7, 12288 x 4096 31.8, 29.0; 128 rows by 15360 x 5120 46.5, 44.1, four parts 44.3; 5120 x 20480 55.1, 55.7,
  // four parts 65.  But tiles of 64 weight rows (12288 x 4096, 47 rows) 25.2, 30.1, more rows of X the same time either way, and a
  // split of a few chunks (16 rows by 1024 x 4096 in eight) 5.4, 5.7.
  constexpr int PARTS = !ROUND ? 1 : NB == 128 ? 2 : 4, CHAINS = 4 / PARTS;  // sums of a part
  const int id = blockIdx.x + gridDim.x * (blockIdx.y + gridDim.y * blockIdx.z);  // (these go round the eight dies)
  const int begin = PARTS == 4 ? id / 8 % 4 : PARTS == 2 ? id / 16 % 2 : 0;
  const int part_len = (len + PARTS - 1) / PARTS, chain_len = ((PARTS == 1 ? nch : part_len) + CHAINS - 1) / CHAINS;
  const int first = begin * part_len < len ? begin * part_len : 0;
  auto chunk = [&](int i) { return c0 + (i + first < len ? i + first : i + first - len); };

  // A row's pieces lie in LDS at places exchanged by the row (place = piece ^ row), so that 16 rows' pieces are read
  // from different banks; the lanes fetch them in that order.
  const T* src[LI];
  int piece[LI];
#pragma unroll
  for (int i = 0; i < LI; ++i) {
    const int row = (wave * LI + i) * RPL + lane / CH;
    piece[i] = (lane % CH) ^ (row & SWAP);
    src[i] = row < MB ? a.W + rows(min(m0 + row, a.M - 1)) * a.ldw : a.X + (int64_t)cols(min(n0 + row - MB, n_cols - 1)) * a.ldx;
  }
  const int pieces = a.K / 8;
  auto load = [&](int at, int slot) {
    const int c = chunk(at);
    // past the last piece: that one again (set to zero when it is used); past the last chunk: into a slot that is not read
#pragma unroll
    for (int i = 0; i < LI; ++i) {
      const global_ptr_t from = (global_ptr_t)(src[i] + min(c * CH + piece[i], pieces - 1) * 8);
      const lds_ptr_t to = (lds_ptr_t)(slots + slot * SLOT + (wave * LI + i) * 1024);
      if (NT_W && (wave * LI + i) * RPL < MB) __builtin_amdgcn_global_load_lds(from, to, 16, 0, 2 /* read once */);
      else __builtin_amdgcn_global_load_lds(from, to, 16, 0, 0);
    }
  };
#pragma unroll
  for (int d = 0; d < ST - 1; ++d) load(d, d);

  // The instruction adds its products one after the other, so no sum has more than a quarter of K: one over all of 4096
  // columns is 3.95e-7 from its value in 64 bits, four are 1.9e-7.  (A sum for each step of a chunk instead, side by side:
  // 0.3 us more for the smallest products, whose time is that of fetching the instructions.)
  float4_t acc[RT][NT], sums[PARTS][RT][NT];
#pragma unroll
  for (auto& sum : sums)
#pragma unroll
    for (int i = 0; i < RT; ++i)
#pragma unroll
      for (int j = 0; j < NT; ++j) sum[i][j] = float4_t{0.f, 0.f, 0.f, 0.f};
  int slot = 0;
  for (int at = 0, step = 0; PARTS == 1 ? at < len : step < 4; ++step) {
    const int in_part = min(part_len, len - (begin + step / CHAINS) % PARTS * part_len) - step % CHAINS * chain_len;
    const int stop = PARTS == 1 ? min(at + chain_len, len) : at + max(min(chain_len, in_part), 0);
#pragma unroll
    for (int i = 0; i < RT; ++i)
#pragma unroll
      for (int j = 0; j < NT; ++j) acc[i][j] = float4_t{0.f, 0.f, 0.f, 0.f};
    for (; at < stop; ++at) {
      const int c = chunk(at);
      // Everybody's part of the slot is there, and nobody still reads the slot before it, which is loaded next: the reads have
      // to have returned, which the barrier itself does not wait for and the instructions that use them need not come before.
      asm volatile("s_waitcnt vmcnt(%0) lgkmcnt(0)" ::"i"(LI * (ST - 2)) : "memory");
      __builtin_amdgcn_s_barrier();
      asm volatile("" ::: "memory");
      load(at + ST - 1, slot == 0 ? ST - 1 : slot - 1);
      const unsigned char* wb = slots + slot * SLOT + (wm * RT * 16 + l16) * KC * 2;
      const unsigned char* xb = slots + slot * SLOT + (MB + wn * NT * 16 + l16) * KC * 2;
#pragma unroll
      for (int ks = 0; ks < KS; ++ks) {
        const int place = ((ks * 4 + g) ^ (l16 & SWAP)) * 16;
        ring_word_t w[RT], x[NT];
#pragma unroll
        for (int i = 0; i < RT; ++i) w[i] = *reinterpret_cast<const ring_word_t*>(wb + i * 16 * KC * 2 + place);
#pragma unroll
        for (int j = 0; j < NT; ++j) x[j] = *reinterpret_cast<const ring_word_t*>(xb + j * 16 * KC * 2 + place);
        if ((c + 1) * CH > pieces && c * CH + ks * 4 + g >= pieces) {  // past the end of the rows
#pragma unroll
          for (int i = 0; i < RT; ++i) w[i] = ring_word_t{0, 0, 0, 0};
#pragma unroll
          for (int j = 0; j < NT; ++j) x[j] = ring_word_t{0, 0, 0, 0};
        }
#pragma unroll
        for (int i = 0; i < RT; ++i)
#pragma unroll
          for (int j = 0; j < NT; ++j) acc[i][j] = ring_mfma<T>(w[i], x[j], acc[i][j]);
      }
      slot = slot == ST - 1 ? 0 : slot + 1;
      if constexpr (RT * NT == 1) {
        // The instruction's sums are there eight states after it.  The compiler has been seen to read the first of them two
        // after it behind this loop, and a copy of this kernel in which that was one got the sum without its last products.
        __builtin_amdgcn_sched_barrier(0);
        asm volatile("s_nop 7\n\ts_nop 1" ::: "memory");
      }
    }
#pragma unroll
    for (int i = 0; i < RT; ++i)
#pragma unroll
      for (int j = 0; j < NT; ++j) {
        if (PARTS > 1 && step % CHAINS == 0) {
#pragma unroll
          for (int k = 1; k < PARTS; ++k) sums[k - 1][i][j] = sums[k][i][j];
          sums[PARTS - 1][i][j] = acc[i][j];
        } else {
          sums[PARTS - 1][i][j] += acc[i][j];
        }
      }
  }
  if constexpr (PARTS == 4) {
    for (int r = begin; r > 0; --r)  // the columns' order
#pragma unroll
      for (int i = 0; i < RT; ++i)
#pragma unroll
        for (int j = 0; j < NT; ++j) {
          const float4_t last = sums[3][i][j];
          sums[3][i][j] = sums[2][i][j], sums[2][i][j] = sums[1][i][j], sums[1][i][j] = sums[0][i][j], sums[0][i][j] = last;
        }
  }
#pragma unroll
  for (int k = 1; k < PARTS; ++k)
#pragma unroll
    for (int i = 0; i < RT; ++i)
#pragma unroll
      for (int j = 0; j < NT; ++j) sums[0][i][j] += sums[k][i][j];
  if (!__is_same(Out, RingRowParts) && gridDim.z > 1) {
    float4_t* p = part + threadIdx.x;
#pragma unroll
    for (int i = 0; i < RT; ++i)
#pragma unroll
      for (int j = 0; j < NT; ++j) p[(i * NT + j) * THREADS] = sums[0][i][j];
  } else {
#pragma unroll
    for (int i = 0; i < RT; ++i)
#pragma unroll
      for (int j = 0; j < NT; ++j) {
        const int m = m0 + (wm * RT + i) * 16 + g * 4, n = n0 + (wn * NT + j) * 16 + l16;
        if (m < a.M && n < n_cols) out(m, cols(n), sums[0][i][j]);
      }
  }
  wait_loads<0>();  // no load into LDS outlives the workgroup
}

struct PlainCols {
  __device__ __forceinline__ int operator()(int n) const { return n; }
};

// Grid: (tiles of W, tiles of X, splits of K).  part: with several splits, the sums [split][tile][value][thread].
template <typename T, int MB, int NB, int KC, int ST, int WM, int WN, bool NT_W, typename Rows, typename Out,
          bool ROUND = MB != 64 && NB <= 128>
__global__ __launch_bounds__(WM * WN * 64) void gemm_ring_kernel(RingOperands<T> a, Rows rows, Out out, float4_t* __restrict__ part) {
  extern __shared__ __attribute__((aligned(16))) unsigned char slots[];
  ring_tile<T, MB, NB, KC, ST, WM, WN, NT_W, ROUND>(
      a, rows, PlainCols{}, out, blockIdx.x * MB, blockIdx.y * NB, a.n,
      part + (((int64_t)blockIdx.z * gridDim.y + blockIdx.y) * gridDim.x + blockIdx.x) * (MB * NB / 4), slots);
}

// Adds the splits' sums up, in their order.  Grid: (tiles of W, tiles of X, values of a thread).
template <int MB, int NB, int WM, int WN, typename Out>
__global__ __launch_bounds__(WM * WN * 64) void gemm_ring_sum_kernel(int n_rows, int M, Out out, const float4_t* __restrict__ part, int splits) {
  constexpr int THREADS = WM * WN * 64, RT = MB / WM / 16, NT = NB / WN / 16;
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6, wm = wave % WM, wn = wave / WM;
  const int i = blockIdx.z / NT, j = blockIdx.z % NT;
  const int m = blockIdx.x * MB + (wm * RT + i) * 16 + (lane >> 4) * 4, n = blockIdx.y * NB + (wn * NT + j) * 16 + (lane & 15);
  if (n >= n_rows || m >= M) return;
  const int64_t step = (int64_t)gridDim.y * gridDim.x * (MB * NB / 4);
  const float4_t* p = part + ((int64_t)blockIdx.y * gridDim.x + blockIdx.x) * (MB * NB / 4) + blockIdx.z * THREADS + threadIdx.x;
  float4_t v = p[0];
  for (int s = 1; s < splits; ++s) v += p[s * step];
  out(m, n, v);
}

// launch(kernel as a template argument, grid, threads, LDS bytes, arguments) is the library's own way to launch with more
// than 48 KiB of LDS.
template <typename T, int MB, int NB, int KC, int ST, int WM, int WN, bool NT_W, bool ROUND, typename Rows, typename Out, typename Launch>
int gemm_ring_tiles(const RingPlan& p, const RingOperands<T>& a, const Rows& rows, const Out& out, void* workspace, hipStream_t s,
                    const Launch& launch) {
  float4_t* part = reinterpret_cast<float4_t*>(workspace);
  const dim3 threads(WM * WN * 64);
  const int rc = launch.template operator()<gemm_ring_kernel<T, MB, NB, KC, ST, WM, WN, NT_W, Rows, Out, ROUND>>(
      dim3(p.rows, p.cols, p.splits), threads, (size_t)ST * (MB + NB) * KC * 2, s, a, rows, out, part);
  if (rc != 0 || p.splits == 1) return rc;
  if constexpr (!__is_same(Out, RingRowParts)) {
  constexpr int values = (MB / WM / 16) * (NB / WN / 16);
  return launch.template operator()<gemm_ring_sum_kernel<MB, NB, WM, WN, Out>>(dim3(p.rows, p.cols, values), threads, 0, s, a.n, a.M, out,
                                                                               (const float4_t*)part, p.splits);
  } else {
    return rc;
  }
}

template <typename T, typename Rows, typename Out, typename Launch>
int gemm_ring(const RingPlan& p, const RingOperands<T>& a, const Rows& rows, const Out& out, void* workspace, hipStream_t s,
              const Launch& launch) {
  constexpr bool kPast = Rows::kPastCaches;
#define DV_RING(MB, NB, KC, ST, WM, WN, NT_W, ROUND) gemm_ring_tiles<T, MB, NB, KC, ST, WM, WN, NT_W, ROUND>(p, a, rows, out, workspace, s, launch)
  switch (p.nb) {
    case 16: return p.splits == 8 ? DV_RING(32, 16, 128, 4, 2, 1, true, false) : DV_RING(32, 16, 128, 4, 2, 1, true, true);
    case 32: return p.mb == 128 ? DV_RING(128, 32, 64, 4, 4, 1, kPast, true) : DV_RING(64, 32, 64, 4, 4, 1, false, false);
    case 64: return p.mb == 128 ? DV_RING(128, 64, 64, 4, 4, 2, kPast, true)
                    : p.mb == 96 ? DV_RING(96, 64, 64, 4, 2, 2, kPast, true) : DV_RING(64, 64, 64, 4, 2, 2, false, false);
  }
  if constexpr (Rows::kMostCols > 64) switch (p.nb) {
    case 128: return p.mb == 64 ? DV_RING(64, 128, 64, 3, 2, 4, false, false)
                     : p.mb == 128 ? DV_RING(128, 128, 64, 4, 2, 4, kPast, kPast) : DV_RING(192, 128, 64, 3, 2, 4, kPast, kPast);
    case 192: return p.mb == 64 ? DV_RING(64, 192, 64, 4, 2, 4, false, false)
                     : p.mb == 128 ? DV_RING(128, 192, 64, 3, 2, 4, false, false) : DV_RING(192, 192, 64, 3, 2, 4, false, false);
    default: return p.mb == 64 ? DV_RING(64, 256, 64, 3, 2, 4, false, false) : DV_RING(128, 256, 64, 3, 2, 4, false, false);
  }
  return -2;  // DV_ERR_UNSUPPORTED
#undef DV_RING
}

}  // namespace dv
