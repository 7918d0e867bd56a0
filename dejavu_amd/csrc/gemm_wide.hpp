// Products of many rows with a weight where the operations bound them: out(m, n) = sum_k W[m, k] X[n, k], 16-bit operands, fp32
// sums, tiles of 256 rows of W by NB rows of X, one workgroup of four waves (one per SIMD) per compute unit.
//
// A wave keeps 128 x NB / 2 sums in the accumulation registers and both halves of its operands of a chunk of 64 columns in vector
// registers: while it multiplies one half, the other one is read from LDS, two reads a row of instructions, so the matrix unit
// waits for nothing but one barrier a chunk.  (Eight waves of 128 x 64 that take turns, which stood here before, read half as much
// again from LDS, and with what arrives there that was all that LDS delivers.)
// LDS holds five operands of a chunk, W and X in turn (160 KB): W of chunk c + 2 arrives while chunk c is multiplied, X of c + 2
// from the last quarter of c's time on, a load or so a row of instructions.  What that is worth (2048 rows by 16384 x 4096, two rounds of
// tiles): two whole chunks instead 249 us, all loads right behind the barrier 231, spread out 225.  A compute unit takes 100 B/ns
// in pieces of 128 contiguous bytes of a row, 60 in pieces of 64 (chunks of 32 columns in five places: 262 us).
// The sums leave by way of LDS, so that a store covers whole lines of a row: a tile's end 10.5 -> 4.2 us.
//
// 2048 rows by 22016 x 4096 338 -> 296 us, 1999 by 18560 x 4096 310 -> 276, 2048 by 8192 x 8192 233 -> 208.  Bound by power: a chunk is 2048 cycles of
// matrix instructions and takes 2460 at 1.81 GHz with all compute units at work, at 2.1 GHz with half of them; fewer cycles come at a
// lower clock (32 x 32 instructions: 2470 at 1.66).
// Tiles too few for the chip share a split of K each (plan_wide_split), whose sums go to memory as rows of fp32 and are added up by the
// launch behind, together with what it is for: 777 rows by 4096 x 16384 192 us in 64 tiles, 113 in four splits (the library 146).
// A sum is one chain over all of K (of a split's part of it), as the library's is: of 16-bit results as many are not the nearest to 64 bits up to 8192 columns (fp16, random
// values: 0.14 % at 2048, 0.27 % at 8192); of 20480, which the library splits, 0.32 % for its 0.24, with the same error to five digits.
#pragma once
#include "gemm_ring.hpp"

namespace dv {

constexpr int kWideRows = 256, kWideChunk = 64;
constexpr size_t kWideLds = (size_t)5 * kWideRows * kWideChunk * 2;
constexpr int64_t kWideMaxStride = 1 << 25;  // 64 rows' bytes are counted in 32 bits

// NB whose rounds of tiles take least: a round takes as NB + 60, one that is not full three quarters of it and a quarter of its share (fewer compute
// units at work have a higher clock).  Over 634 products of 257..8192 rows with cold weights of 9 to 340 million values and 1024 to 36864 columns, every
// width measured, the choice takes 0.1 % longer than the best one and 6 % at most.  (NB + 12 and a half: 0.9 % and 28 %; 1024 rows by 36864 x 9216 739 us,
// now 622, the library 584; 2048 by 28672 x 7168 802 / 718 / 672; 1152 by 27648 x 5120, gated, 379 / 323 / 295.)
inline int plan_wide(int n, int M, int units) {
  int best = 0;
  double least = 0.0;
  for (int nb = 256; nb >= 128; nb -= 32) {
    const int64_t tiles = ((int64_t)M + kWideRows - 1) / kWideRows * (((int64_t)n + nb - 1) / nb), rest = tiles % units;
    const double t = (nb + 60) * ((double)(tiles / units) + (rest ? 0.75 + 0.25 * rest / units : 0.0));
    if (best == 0 || t < least) best = nb, least = t;
  }
  return best;
}

struct WideSplit {
  int nb, splits;
  size_t workspace_bytes(int n, int M) const { return (size_t)splits * n * M * sizeof(float); }
};

// The same with K in up to six parts, one round of workgroups at most: a chunk takes as NB + 166 (fewer columns share the chunk of W, and cold
// weights arrive slower than they are multiplied), a workgroup's ends as 7400, a part's sums as 3.6e-4 each, to memory and back.  From whole
// prompts of 300 to 1900 tokens, every choice for their down projections or fc2 in turn (4096 x 11008, 4096 x 16384, 5120 x 20480): the prompt
// takes 0.1 % longer than with the best one, 1.2 % at most, and 1.00 to 1.29 times less than with the library's products.  (By the products alone, back
// to back, where the clock is lower than beside other kernels, more parts look better than they are: 0.5 % and 3.3 %.)
inline WideSplit plan_wide_split(int n, int M, int K, int units) {
  WideSplit best{256, 1};
  double least = 0.0;
  const int chunks = K / kWideChunk;
  // Up to 256 rows one column of tiles, as many parts as nearly fill the chip: the stream of the weights bounds them, which does not run at its
  // speed with fewer workgroups (128 rows by 20480 x 5120 in 2 / 3 parts 69 / 57 us, 256 in 1 / 2 / 3 99 / 84 / 77).
  if (n <= 256) {
    const int nb = n <= 128 ? 128 : (n + 31) / 32 * 32;
    const int64_t tiles = ((int64_t)M + kWideRows - 1) / kWideRows;
    int64_t s = units * 15 / 16 / tiles;
    if (s > chunks / 8) s = chunks / 8;
    return {nb, (int)(s < 1 ? 1 : s > 6 ? 6 : s)};
  }
  for (int nb = 256; nb >= 128; nb -= 32) {
    const int64_t tiles = ((int64_t)M + kWideRows - 1) / kWideRows * (((int64_t)n + nb - 1) / nb);
    for (int splits = 1; splits <= 6; ++splits) {
      if (splits > 1 && (tiles * splits > units || chunks < splits * 8)) break;
      const int64_t rest = tiles * splits % units;
      const double rounds = (double)(tiles * splits / units) + (rest ? 0.5 + 0.5 * rest / units : 0.0);
      const double t = rounds * (((chunks + splits - 1) / splits) * (double)(nb + 166) + 7400.0) + 3.6e-4 * splits * n * (double)M;
      if (least == 0.0 || t < least) best = {nb, splits}, least = t;
    }
  }
  return best;
}

// Four values of a vector of M from place m on (past its end: its last one), m % 4 == 0.
template <typename T>
struct WideBias {
  typedef T vec_t __attribute__((ext_vector_type(4)));
  vec_t v;
  __device__ __forceinline__ void load(const T* p, int M, int m) {
    v = vec_t{(T)0.f, (T)0.f, (T)0.f, (T)0.f};
    if (p == nullptr) return;
    if (m + 3 < M && (reinterpret_cast<uintptr_t>(p) & 7) == 0) {
      v = *reinterpret_cast<const vec_t*>(p + m);
    } else {
#pragma unroll
      for (int e = 0; e < 4; ++e) v[e] = p[min(m + e, M - 1)];
    }
  }
};

// A part's sums: rows of M floats (M % 4 == 0), one part after the other.
struct WidePart {
  struct Row {};
  float* part;
  int64_t rows;
  int M;
  __device__ __forceinline__ void store(int m, int row, const float4_t& v) const {
    *reinterpret_cast<float4_t*>(part + (blockIdx.y * rows + row) * M + m) = v;
  }
};

// The sums stay where they are: the compiler copies them from one set of registers to another when left to itself.
template <typename T>
__device__ __forceinline__ void wide_mfma(float4_t& acc, const ring_word_t& w, const ring_word_t& x) {
  if constexpr (__is_same(T, half_t)) asm volatile("v_mfma_f32_16x16x32_f16 %0, %1, %2, %0" : "+a"(acc) : "v"(w), "v"(x));
  else asm volatile("v_mfma_f32_16x16x32_bf16 %0, %1, %2, %0" : "+a"(acc) : "v"(w), "v"(x));
}

// Out: kOuts results (of type T, columns kOuts / 4 * m ..) of the sums of rows m .. m + 3, by make(row(m), sums) for any m below the
// tile's end; row(m), what a row's results need beside their sums, is asked for before the loop (a bias read behind it: 69 instead of
// 63 us, 2048 rows by 4096 x 4096); base, ld, columns: where they go.
// WidePart: part blockIdx.y of gridDim.y of K.
// Grid: row_tiles * col_tiles (256 rows of W, NB rows of X).  K, ldx, ldw % 8 == 0, X and W on 16-byte boundaries.
template <typename T, int NB, typename Out>
__global__ __launch_bounds__(256, 1) void gemm_wide_kernel(RingOperands<T> a, Out out, int row_tiles, int col_tiles) {
#if defined(__HIP_DEVICE_COMPILE__)  // (the loads' resources have no type on the host)
  extern __shared__ __attribute__((aligned(16))) unsigned char slots[];
  constexpr bool PART = __is_same(Out, WidePart);
  constexpr int MB = kWideRows, KC = kWideChunk, CH = KC / 8, RPL = 64 / CH, UNIT = MB * KC * 2;
  constexpr int RT = MB / 32, NT = NB / 32;                      // tiles of 16 rows a wave
  constexpr int LW = MB / RPL / 4, LX = NB / RPL / 4;            // loads of a wave
  static_assert(NB % 32 == 0 && NB <= MB, "tile");
  const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int wm = wave & 1, wn = wave >> 1, l16 = lane & 15, g = lane >> 4;
  // Consecutive workgroups go round the eight compute dies: each die is given a stretch of the tiles, taken in blocks of
  // eight row tiles by all columns, so that its L2 serves an operand's later uses.
  int bm, bn;
  {
    const int tiles = row_tiles * col_tiles, die = blockIdx.x & 7, k = blockIdx.x >> 3;
    const int id = die * (tiles >> 3) + min(die, tiles & 7) + k;
    const int block = id / (8 * col_tiles), at = id - block * 8 * col_tiles, tall = min(8, row_tiles - block * 8);
    bm = block * 8 + at % tall;
    bn = at / tall;
  }
  const int m0 = bm * MB, n0 = bn * NB, chunks = a.K / KC;  // (the columns behind the whole chunks are the last part's)
  const int c0 = PART ? chunks * (int)blockIdx.y / (int)gridDim.y : 0;
  const int nch = (PART ? chunks * ((int)blockIdx.y + 1) / (int)gridDim.y : chunks) - c0;

  // A wave loads 64 rows of W and NB / 4 of X, eight rows at a time; rows past the end are the last one again.  A row's pieces of
  // 16 bytes lie in LDS at places exchanged by the row (place = piece ^ row): 16 rows' pieces are read from different banks.
  const int w_row = min(m0 + wave * LW * RPL, a.M - 1), x_row = min(n0 + wave * LX * RPL, a.n - 1);
  const auto wr = __builtin_amdgcn_make_buffer_rsrc(const_cast<T*>(a.W) + w_row * a.ldw, 0,
                                                    (int)((unsigned)(min(LW * RPL, a.M - w_row) - 1) * (unsigned)a.ldw * 2u + a.K * 2u), 0x00020000);
  const auto xr = __builtin_amdgcn_make_buffer_rsrc(const_cast<T*>(a.X) + x_row * a.ldx, 0,
                                                    (int)((unsigned)(min(LX * RPL, a.n - x_row) - 1) * (unsigned)a.ldx * 2u + a.K * 2u), 0x00020000);
  const int piece = (lane % CH) ^ (lane / CH);
  unsigned w_at[LW], x_at[LX];
#pragma unroll
  for (int i = 0; i < LW; ++i)
    w_at[i] = (unsigned)(min(m0 + (wave * LW + i) * RPL + lane / CH, a.M - 1) - w_row) * (unsigned)a.ldw * 2u + piece * 16;
#pragma unroll
  for (int i = 0; i < LX; ++i)
    x_at[i] = (unsigned)(min(n0 + (wave * LX + i) * RPL + lane / CH, a.n - 1) - x_row) * (unsigned)a.ldx * 2u + piece * 16;
  auto load_w = [&](int c, int unit, int i) {
    __builtin_amdgcn_raw_ptr_buffer_load_lds(wr, (lds_ptr_t)(slots + unit * UNIT + (wave * LW + i) * 1024), 16, w_at[i], (c0 + c) * KC * 2, 0, 0);
  };
  auto load_x = [&](int c, int unit, int i) {
    __builtin_amdgcn_raw_ptr_buffer_load_lds(xr, (lds_ptr_t)(slots + unit * UNIT + (wave * LX + i) * 1024), 16, x_at[i], (c0 + c) * KC * 2, 0, 0);
  };

  typename Out::Row rows[PART ? 1 : RT];
  if constexpr (!PART)
#pragma unroll
    for (int i = 0; i < RT; ++i) rows[i] = out.row(m0 + (wm * RT + i) * 16 + g * 4);
  ring_word_t w[2][RT], x[2][NT];
  float4_t acc[RT][NT];
#pragma unroll
  for (int i = 0; i < RT; ++i)
#pragma unroll
    for (int j = 0; j < NT; ++j) acc[i][j] = float4_t{0.f, 0.f, 0.f, 0.f};
  const unsigned char* wb = slots + (wm * RT * 16 + l16) * KC * 2;
  const unsigned char* xb = slots + (wn * NT * 16 + l16) * KC * 2;
  const int half_at[2] = {(g ^ (l16 & 7)) * 16, ((4 + g) ^ (l16 & 7)) * 16};
  auto read = [&](int w_unit, int x_unit, int half, int i) {  // x first: all of it is needed at once
    if (i < NT) x[half][i] = *reinterpret_cast<const ring_word_t*>(xb + i * 16 * KC * 2 + half_at[half] + x_unit * UNIT);
    else if (i < NT + RT) w[half][i - NT] = *reinterpret_cast<const ring_word_t*>(wb + (i - NT) * 16 * KC * 2 + half_at[half] + w_unit * UNIT);
  };
  auto multiply = [&](int half, int i) {
    __builtin_amdgcn_sched_barrier(0);
#pragma unroll
    for (int j = 0; j < NT; ++j) wide_mfma<T>(acc[i][j], w[half][i], x[half][j]);
    __builtin_amdgcn_sched_barrier(0);
  };
  auto reads_back = [&]() {
    asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
    __builtin_amdgcn_sched_barrier(0);
  };
  auto all_here = [&]() {  // nobody reads LDS any more, nothing is on its way there
    asm volatile("s_waitcnt vmcnt(0) lgkmcnt(0)" ::: "memory");
    __builtin_amdgcn_s_barrier();
    asm volatile("" ::: "memory");
  };

  if (nch > 0) {
    const int last = nch - 1;  // (past it: that chunk again, into places that are not read)
#pragma unroll
    for (int i = 0; i < LW; ++i) load_w(0, 0, i);
#pragma unroll
    for (int i = 0; i < LX; ++i) load_x(0, 1, i);
#pragma unroll
    for (int i = 0; i < LW; ++i) load_w(min(1, last), 2, i);
#pragma unroll
    for (int i = 0; i < LX; ++i) load_x(min(1, last), 3, i);
    asm volatile("s_waitcnt vmcnt(%0)" ::"i"(LW + LX) : "memory");
    __builtin_amdgcn_s_barrier();
    asm volatile("" ::: "memory");
#pragma unroll
    for (int i = 0; i < RT + NT; ++i) read(0, 1, 0, i);
    reads_back();
    int wu = 0, free_unit = 4;  // W of chunk c is in unit 2 c mod 5, X in the one behind it; the fifth is the one that X of c - 1 had
    for (int c = 0; c < nch; ++c) {
      const int xu = wu == 4 ? 0 : wu + 1, next_wu = wu >= 3 ? wu - 3 : wu + 2, next_xu = xu >= 3 ? xu - 3 : xu + 2;
      const int ahead = min(c + 2, last);
#pragma unroll
      for (int i = 0; i < RT; ++i) {
        read(wu, xu, 1, 2 * i), read(wu, xu, 1, 2 * i + 1);
        load_w(ahead, free_unit, i);
        multiply(0, i);
      }
      // Everybody's part of chunk c + 1 is there (the loads just asked for are the only ones that need not be), and nobody
      // reads chunk c any more.
      asm volatile("s_waitcnt vmcnt(%0) lgkmcnt(0)" ::"i"(LW) : "memory");
      __builtin_amdgcn_s_barrier();
      asm volatile("" ::: "memory");
      __builtin_amdgcn_sched_barrier(0);
#pragma unroll
      for (int i = 0; i < RT; ++i) {
        read(next_wu, next_xu, 0, 2 * i), read(next_wu, next_xu, 0, 2 * i + 1);
        if (i < LX) load_x(ahead, wu, i);
        multiply(1, i);
      }
      reads_back();
      free_unit = xu;
      wu = next_wu;
    }
  }
  static_assert(LW == RT && LX <= RT && RT + NT <= 2 * RT, "a row of instructions has one load and two reads");
  if (a.K % KC != 0 && (!PART || blockIdx.y + 1 == gridDim.y)) {  // the columns behind the whole chunks, zeros past the rows' end
    all_here();
    const unsigned back = max(chunks * KC + piece * 8 - (a.K - 8), 0) * 2;
#pragma unroll
    for (int i = 0; i < LW; ++i) w_at[i] -= back, load_w(nch, 0, i);  // (chunk nch of this part: c0 + nch == chunks)
#pragma unroll
    for (int i = 0; i < LX; ++i) x_at[i] -= back, load_x(nch, 1, i);
    all_here();
#pragma unroll
    for (int half = 0; half < 2; ++half) {
#pragma unroll
      for (int i = 0; i < RT + NT; ++i) read(0, 1, half, i);
      reads_back();
      if (chunks * CH + half * 4 + g >= a.K / 8) {
#pragma unroll
        for (int i = 0; i < RT; ++i) w[half][i] = ring_word_t{0, 0, 0, 0};
#pragma unroll
        for (int j = 0; j < NT; ++j) x[half][j] = ring_word_t{0, 0, 0, 0};
      }
      __builtin_amdgcn_sched_barrier(0);
      asm volatile("s_nop 4" ::: "memory");  // between these writes and the matrix instructions
#pragma unroll
      for (int i = 0; i < RT; ++i) multiply(half, i);
    }
  }
  asm volatile("s_nop 15" ::: "memory");  // the last sums are there
  __builtin_amdgcn_sched_barrier(0);

  if constexpr (PART) {
#pragma unroll
    for (int i = 0; i < RT; ++i)
#pragma unroll
      for (int j = 0; j < NT; ++j) {
        const int m = m0 + (wm * RT + i) * 16 + g * 4, row = n0 + (wn * NT + j) * 16 + l16;
        if (m < a.M && row < a.n) out.store(m, row, acc[i][j]);
      }
    wait_loads<0>();  // no load into LDS outlives the workgroup
    return;
  } else {
  typedef T out_t __attribute__((ext_vector_type(Out::kOuts)));
  T* const base = out.base();
  const int64_t ld = out.ld();
  const int columns = out.columns();
  constexpr int PER = Out::kOuts;  // of four rows of W
  if (ld % 8 == 0 && (reinterpret_cast<uintptr_t>(base) & 15) == 0) {
    constexpr int ROW = 128 * PER / 4 * 2, P = ROW / 16;  // bytes of a wave's row, pieces of it
    all_here();
    unsigned char* mine = slots + wave * (NB / 2 * ROW);
#pragma unroll
    for (int i = 0; i < RT; ++i)
#pragma unroll
      for (int j = 0; j < NT; ++j) {
        const int at = (i * 16 + g * 4) * PER / 4 * 2, n = j * 16 + l16;  // bytes
        *reinterpret_cast<out_t*>(mine + n * ROW + (((at >> 4) ^ (n & (P - 1))) << 4) + (at & 15)) = out.make(rows[i], acc[i][j]);
      }
    reads_back();  // (a wave reads what it wrote itself)
#pragma unroll 8
    for (int r = 0; r < NB / 2 * P / 64; ++r) {
      const int n = r * (64 / P) + lane / P, p = lane % P;
      const ring_word_t v = *reinterpret_cast<const ring_word_t*>(mine + n * ROW + ((p ^ (n & (P - 1))) << 4));
      const int col = (m0 + wm * 128) * PER / 4 + p * 8, row = n0 + wn * (NB / 2) + n;
      if (row >= a.n) continue;
      T* o = base + row * ld + col;
      if (col + 8 <= columns) {
        *reinterpret_cast<ring_word_t*>(o) = v;
      } else {
        typedef T vec_t __attribute__((ext_vector_type(8)));
        const vec_t e = __builtin_bit_cast(vec_t, v);
#pragma unroll
        for (int k = 0; k < 8; ++k)
          if (col + k < columns) o[k] = e[k];
      }
    }
  } else {
#pragma unroll
    for (int i = 0; i < RT; ++i)
#pragma unroll
      for (int j = 0; j < NT; ++j) {
        const int m = m0 + (wm * RT + i) * 16 + g * 4, row = n0 + (wn * NT + j) * 16 + l16, col = m * PER / 4;
        const out_t v = out.make(rows[i], acc[i][j]);
#pragma unroll
        for (int k = 0; k < PER; ++k)
          if (row < a.n && col + k < columns) base[row * ld + col + k] = v[k];
      }
  }
  wait_loads<0>();
  }
#endif
}

// Adds the parts up in their order.  done(row, m, sums of rows m .. m + 3 of W, ready(row, m)); ready asks for what is needed beside them.
template <int SPLITS, typename Done>
__global__ __launch_bounds__(256) void wide_sum_kernel(const float* __restrict__ part, int64_t rows, int M, Done done) {
  const int64_t quads = rows * M / 4;
  const float4_t* p = reinterpret_cast<const float4_t*>(part);
  for (int64_t q = (int64_t)blockIdx.x * 256 + threadIdx.x; q < quads; q += (int64_t)gridDim.x * 256) {
    const int64_t row = q * 4 / M;
    const int m = (int)(q * 4 - row * M);
    float4_t v[SPLITS];
#pragma unroll
    for (int k = 0; k < SPLITS; ++k) v[k] = p[k * quads + q];
    const auto ready = done.ready(row, m);
#pragma unroll
    for (int k = 1; k < SPLITS; ++k) v[0] += v[k];
    done(row, m, v[0], ready);
  }
}

template <typename Done, typename Launch>
int wide_sum(int splits, const float* part, int64_t rows, int M, const Done& done, hipStream_t s, const Launch& launch) {
  const int64_t blocks = (rows * M / 4 + 255) / 256;
  const dim3 grid((unsigned)(blocks < 8192 ? blocks : 8192)), threads(256);
#define DV_SUM(S) launch.template operator()<wide_sum_kernel<S, Done>>(grid, threads, (size_t)0, s, part, rows, M, done)
  switch (splits) {
    case 2: return DV_SUM(2);
    case 3: return DV_SUM(3);
    case 4: return DV_SUM(4);
    case 5: return DV_SUM(5);
    default: return DV_SUM(6);
  }
#undef DV_SUM
}

// launch as for gemm_ring
template <typename T, typename Out, typename Launch>
int gemm_wide(int nb, const RingOperands<T>& a, const Out& out, hipStream_t s, const Launch& launch, int splits = 1) {
  const int64_t rows = ((int64_t)a.M + kWideRows - 1) / kWideRows, cols = ((int64_t)a.n + nb - 1) / nb;
  const dim3 grid((unsigned)(rows * cols), (unsigned)splits), threads(256);
#define DV_WIDE(NB) launch.template operator()<gemm_wide_kernel<T, NB, Out>>(grid, threads, kWideLds, s, a, out, (int)rows, (int)cols)
  switch (nb) {
    case 128: return DV_WIDE(128);
    case 160: return DV_WIDE(160);
    case 192: return DV_WIDE(192);
    case 224: return DV_WIDE(224);
    default: return DV_WIDE(256);
  }
#undef DV_WIDE
}

}  // namespace dv
