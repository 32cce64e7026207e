// Float32 matrix products out [M, N] (+)= a [M, K] w[N, K]^T (+ bias) on the matrix cores.
//
// The float32 matrix instruction multiplies and adds float32 values as fused multiply-adds in ascending k, subnormal
// numbers included: 16x16x4 gives, bit for bit, the chain of fmaf that a thread would make (checked over normal products,
// subnormal products and subnormal inputs).  K is divided into F32_PARTS runs of whole 128s (f32_part, common.h), a chain each from
// zero, whose sums are added first to last: four short chains at once where rows are few, and a bound of the
// error that is a quarter of one chain's (measured, K up to 3,072: farthest from 64 bits 4.9e-6 for 5.7e-6).  So every output here is the same sum whatever kernel, tile or number of rows made it, and equals the tiled
// kernel's in gemm.hip, which serves what this file does not take (K no multiple of 32, rows not 16-byte aligned): a row's result
// does not depend on what else is in the batch.
#include "common.h"

#include <type_traits>

int lrs_gemm_f32(float* out, bool add, const float* a, const float* w, const float* bias, int m, int n, int k, int lda, int ldc, hipStream_t s);

namespace {

// Memory straight into LDS as fetch_to_lds (common.h) has it, for a base that the compiler holds in scalar registers already: no wait
// for a vector instruction that wrote it (the waits cost 0.3 % of a float32 prompt here; tests/test_wait_states.py reads the built library).
__device__ __forceinline__ void fetch_from(uint64_t base, unsigned lane_offset, unsigned lds_address) {
  asm volatile("s_mov_b32 m0, %0\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %1, %2" :: "s"(lds_address), "v"(lane_offset), "s"(base) : "memory");
}

// WN x WM waves side by side along weight rows and input rows, TN x TM tiles of 16 x 16 outputs a wave; slices of BK of both
// operands lie in LDS, written there by memory itself (STAGES slices).  A tile's rows lie piece by piece, the 16 bytes of its
// rows at one place of K after each other: the 64 single floats that a fragment read takes (16 rows, four consecutive k) meet
// every bank once, and all of a slice's reads go by one address register.  QUADS, where memory and not the matrix unit sets the pace: four
// neighbouring lanes of a fetch bring 64 bytes of one row, since a lane a row costs the compute unit's L1 four times as many looks at its
// tags (8 rows, N 1,024 K 3,072 11.5 us for 7.6); 64 bytes of all of a tile's rows lie together, and a row's four pieces of 16 bytes are
// turned round by a quarter of its number, for the banks.  That is four address registers an operand to work out for every slice: 8
// rows, N 4,096 K 1,024 in one chain 7.6 us so 8.9, 509 rows N 1,024 K 2,048 27 so 29.  A slice's fragments are read into registers while
// the slice before is multiplied, between the products: what a wave does besides them has to fit the 32 cycles of a 16x16x4,
// for a wave whose sums are one chain has nothing else to wait for (K = 3,072 in 64 workgroups: 54 cycles a product with an
// address worked out for every read and fetch).
// PARTS: 1, or F32_PARTS groups of waves that take a run of K each, one wave a group, with slices of its own that no barrier guards;
// their sums meet in LDS at the end.  (With 1 a wave adds each run's sum to those before.)  A wave a SIMD: a 16x16x4 is as long in the
// matrix unit as its sum is on its way, so two chains on a SIMD take turns.
// WR, AR: 8 where a tile has only 8 rows of weights or inputs to bring (its other outputs are copies that nobody stores).
// A wave's fragment of the weights is the instruction's first operand: its lanes end with four consecutive output columns.
template <bool GATED, bool QUADS, int BK, int PARTS, int WN, int WM, int TN, int TM, int STAGES, int WR, int AR>
__global__ __launch_bounds__(PARTS * WN * WM * WAVE) void gemm_f32_mfma_kernel(const float* __restrict__ a, const float* __restrict__ w, int m, int n, int k,
                                                                       int lda, int tiles_m, int tiles, float* __restrict__ out, int add, int ldc,
                                                                       const float* __restrict__ bias, int wide_stores) {
  // (the arguments that lead to the first fetches come first: they are in registers when a wave begins, the file is compiled so)
  static_assert((BK == 32 || BK == 64) && (WR == 8 || WR == 16) && (AR == 8 || AR == 16), "what the layout is made for");
  static_assert(PARTS == 1 || (PARTS == F32_PARTS && WN * WM == 1), "one group of waves for all of K, or a wave for each run of it");
  constexpr int WAVES = WN * WM, BN = WN * TN * WR, BM = WM * TM * AR;
  constexpr int CHUNKS = BK / 4;                                           // a row's pieces of 16 bytes
  constexpr int STAGE = (BN + BM) * BK, EACH = (BN + BM) * BK / 256 / WAVES;   // floats; fetches a wave and slice (a fetch brings 64 pieces)
  constexpr int W_FETCHES = CHUNKS * WR / 64, A_FETCHES = CHUNKS * AR / 64;    // for the rows of a tile
  static_assert((BN + BM) * BK / 256 % WAVES == 0 && STAGES * EACH < 64, "every wave brings as much, counted in vmcnt");
  __shared__ __attribute__((aligned(128))) float all_slices[PARTS * STAGES * STAGE];
  const int tid = threadIdx.x, lane = tid % WAVE, wave = WAVES == 1 ? 0 : __builtin_amdgcn_readfirstlane(tid / WAVE);
  const int part = PARTS == 1 ? 0 : __builtin_amdgcn_readfirstlane(tid / WAVE);
  float* const slices = all_slices + part * (STAGES * STAGE);
  int id = blockIdx.x;
  if (tiles % 8 == 0) id = (id % 8) * (tiles / 8) + id / 8;        // an XCD takes neighbouring weight rows, which it then reads once
  const int m0 = (id % tiles_m) * BM, n0 = (id / tiles_m) * BN;
  unsigned offset[EACH];
#pragma unroll
  for (int i = 0; i < EACH; ++i) {
    const int fetch = wave + i * WAVES;                                    // the weights' tiles first, then the inputs'
    if (fetch < BN / WR * W_FETCHES) {
      const int of_tile = QUADS ? lane / 4 % WR : lane % WR, last = n - 1 - n0, piece = fetch % W_FETCHES;
      const int row = fetch / W_FETCHES * WR + of_tile;
      const int chunk = QUADS ? (piece * (16 / WR) + lane / (4 * WR)) * 4 + (lane % 4 ^ (of_tile >> 2)) : piece * (64 / WR) + lane / WR;
      offset[i] = ((unsigned)(row < last ? row : last) * (unsigned)k + (unsigned)chunk * 4u) * 4u;
    } else {
      const int mine = fetch - BN / WR * W_FETCHES;
      const int of_tile = QUADS ? lane / 4 % AR : lane % AR, last = m - 1 - m0, piece = mine % A_FETCHES;
      const int row = mine / A_FETCHES * AR + of_tile;
      const int chunk = QUADS ? (piece * (16 / AR) + lane / (4 * AR)) * 4 + (lane % 4 ^ (of_tile >> 2)) : piece * (64 / AR) + lane / AR;
      offset[i] = ((unsigned)(row < last ? row : last) * (unsigned)lda + (unsigned)chunk * 4u) * 4u;
    }
  }
  // this wave's slices: all, or its run's (none where K is too short for so many runs: it fetches the last and multiplies nothing)
  const int run = f32_part(k) / BK, all = k / BK, first = PARTS == 1 ? 0 : part * run < all ? part * run : all - 1;
  const int steps = PARTS == 1 ? all : part * run >= all ? 0 : all - first < run ? all - first : run;
  const unsigned slices_address = (unsigned)(uintptr_t)(__attribute__((address_space(3))) float*)all_slices + (unsigned)(part * (STAGES * STAGE * 4) + wave * 1024);
  uint64_t w_at = (uint64_t)(uintptr_t)(w + (int64_t)n0 * k + first * BK), a_at = (uint64_t)(uintptr_t)(a + (int64_t)m0 * lda + first * BK);   // of the slice to fetch next
  auto slice_there = [&](auto pending) {                                   // and read by every wave that shares it
    if constexpr (PARTS == 1) fetched_and_read_then_barrier<decltype(pending)::value>();
    else asm volatile("s_waitcnt vmcnt(%0) lgkmcnt(0)" :: "n"(decltype(pending)::value) : "memory");
  };
  auto fetch = [&](int stage, int i) {
    const uint64_t base = wave + i * WAVES < BN / WR * W_FETCHES ? w_at : a_at;
    fetch_from(base, offset[i], slices_address + (unsigned)(stage * (STAGE * 4) + i * WAVES * 1024));
  };
  auto advance = [&](int kt) {                                             // kt: the slice to fetch next; past the end the last one once more, read by nobody
    const unsigned by = kt < steps ? BK * 4u : 0u;
    w_at += by, a_at += by;
  };
  struct Fragments {
    float w[CHUNKS][TN], a[CHUNKS][TM];
  };
  const int r = lane & 15, g = lane >> 4;
  const int wave_n = (wave % WN) * TN * WR, wave_m = (wave / WN) * TM * AR;
  // this lane's value of a tile's rows in the pieces c, c + 4, .. (QUADS; else in piece 0), in floats from the tile's first
  int w_at_chunk[QUADS ? 4 : 1], a_at_chunk[QUADS ? 4 : 1];
#pragma unroll
  for (int c = 0; c < (QUADS ? 4 : 1); ++c) {
    const int wr = r % WR, ar = r % AR;
    w_at_chunk[c] = wave_n * BK + (QUADS ? wr * 16 + (c ^ (wr >> 2)) * 4 : wr * 4) + g;
    a_at_chunk[c] = (BN + wave_m) * BK + (QUADS ? ar * 16 + (c ^ (ar >> 2)) * 4 : ar * 4) + g;
  }
  auto read = [&](int stage, int c, Fragments& f) {                       // four k of a slice
#pragma unroll
    for (int i = 0; i < TN; ++i) f.w[c][i] = slices[w_at_chunk[QUADS ? c % 4 : 0] + stage * STAGE + i * WR * BK + (QUADS ? c / 4 * WR * 16 : c * WR * 4)];
#pragma unroll
    for (int j = 0; j < TM; ++j) f.a[c][j] = slices[a_at_chunk[QUADS ? c % 4 : 0] + stage * STAGE + j * AR * BK + (QUADS ? c / 4 * AR * 16 : c * AR * 4)];
  };
  floatx4 acc[TN][TM], total[TN][TM];
#pragma unroll
  for (int i = 0; i < TN; ++i)
#pragma unroll
    for (int j = 0; j < TM; ++j) acc[i][j] = total[i][j] = floatx4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
  for (int kt = 0; kt < STAGES; ++kt) {
#pragma unroll
    for (int i = 0; i < EACH; ++i) fetch(kt, i);
    advance(kt + 1);
  }
  Fragments even, odd;
  slice_there(std::integral_constant<int, (STAGES - 1) * EACH>());
#pragma unroll
  for (int c = 0; c < CHUNKS; ++c) read(0, c, even);
  int stage = 0;                                                           // of slice kt
  // first: slice kt begins a run of K.  What the run before left is added to the sums before it beside the first products, which begin
  // from zero.  As a pass over the sums between two runs, with the matrix units waiting, and with the gated epilogue's instructions in
  // every kernel, 2,048 rows of N 4,096 K 1,024 took 140.5 us (134.6 so, 134.3 in one chain) and 509 rows of N 2,048 K 6,144 108.5 (107.1, 106.2).
  auto turn = [&](int kt, const Fragments& now, Fragments& next, auto first) {
    // slice kt + 1 is there, and every wave holds slice kt in registers: its stage may be filled again
    slice_there(std::integral_constant<int, (STAGES - 2) * EACH>());
    const int free = stage;
    stage = stage == STAGES - 1 ? 0 : stage + 1;
#pragma unroll
    for (int c = 0; c < CHUNKS; ++c) {
      // the matrix unit works on these while the wave asks for the rest: reads in the first half, so that they are there by the end
#pragma unroll
      for (int i = 0; i < TN; ++i)
#pragma unroll
        for (int j = 0; j < TM; ++j) {
          if (decltype(first)::value && c == 0) {
            total[i][j] += acc[i][j];
            asm volatile("" : "+v"(total[i][j]));                          // here, not in a block between two runs
            __builtin_amdgcn_sched_barrier(0);
            acc[i][j] = __builtin_amdgcn_mfma_f32_16x16x4f32(now.w[c][i], now.a[c][j], floatx4{0.f, 0.f, 0.f, 0.f}, 0, 0, 0);
          } else {
            acc[i][j] = __builtin_amdgcn_mfma_f32_16x16x4f32(now.w[c][i], now.a[c][j], acc[i][j], 0, 0, 0);
          }
        }
      __builtin_amdgcn_sched_barrier(0);
      if (c < CHUNKS / 2) read(stage, 2 * c, next), read(stage, 2 * c + 1, next);
#pragma unroll
      for (int i = c; i < EACH; i += CHUNKS) fetch(free, i);
      __builtin_amdgcn_sched_barrier(0);
    }
    advance(kt + STAGES + 1);
  };
  const std::true_type begins;
  const std::false_type goes_on;
  int kt = 0;
  auto walk = [&](int end) {
    for (; kt < end; kt += 2) {
      turn(kt, even, odd, goes_on);
      if (kt + 1 < end) turn(kt + 1, odd, even, goes_on);
    }
  };
  if constexpr (PARTS == 1) {
    while (kt < steps) {                                                   // a run has an even number of slices, but for the last
      const int end = steps - kt > run ? kt + run : steps;
      turn(kt, even, odd, begins);
      if (kt + 1 < end) turn(kt + 1, odd, even, goes_on);
      kt += 2;
      walk(end);
    }
  } else {
    walk(steps);
  }
  asm volatile("s_waitcnt vmcnt(0)" ::: "memory");                         // the fetches past K
  if constexpr (PARTS == 1) {
#pragma unroll
    for (int i = 0; i < TN; ++i)
#pragma unroll
      for (int j = 0; j < TM; ++j) acc[i][j] = total[i][j] + acc[i][j];    // the last run's
  } else {
    // every wave's fetches are done and its slices read: its sums go where they were
    if (part > 0) {
#pragma unroll
      for (int i = 0; i < TN; ++i)
#pragma unroll
        for (int j = 0; j < TM; ++j) *(floatx4*)(slices + ((i * TM + j) * WAVE + lane) * 4) = acc[i][j];
    }
    __syncthreads();
    if (part > 0) return;
#pragma unroll
    for (int p = 1; p < PARTS; ++p)
#pragma unroll
      for (int i = 0; i < TN; ++i)
#pragma unroll
        for (int j = 0; j < TM; ++j) acc[i][j] += *(const floatx4*)(all_slices + p * (STAGES * STAGE) + ((i * TM + j) * WAVE + lane) * 4);
  }
#pragma unroll
  for (int j = 0; j < TM; ++j) {
    const int token = m0 + wave_m + j * AR + r;
    if (token >= m || r >= AR) continue;
#pragma unroll
    for (int i = 0; i < TN; ++i) {
      const int col = n0 + wave_n + i * WR + 4 * g;
      if (4 * g >= WR) continue;
      floatx4 v = acc[i][j];
      if constexpr (GATED) {
        // a tile's 16 weight rows are 8 gate rows and the 8 up rows of the same features, which the lane 32 further on holds (n % 16 == 0)
        floatx4 up;
#pragma unroll
        for (int e = 0; e < 4; ++e) up[e] = __shfl(v[e], (lane + 32) % WAVE, WAVE);
        if (g < 2 && col < n) {
#pragma unroll
          for (int e = 0; e < 4; ++e) v[e] = v[e] / (1.0f + expf(-v[e])) * up[e];
          *(floatx4*)(out + (int64_t)token * ldc + (col - 4 * g) / 2 + 4 * g) = v;
        }
        continue;
      }
      float* to = out + (int64_t)token * ldc + col;
      if (wide_stores && col + 3 < n) {
        if (bias)
#pragma unroll
          for (int e = 0; e < 4; ++e) v[e] += bias[col + e];
        if (add) v = *(const floatx4*)to + v;
        *(floatx4*)to = v;
      } else {
#pragma unroll
        for (int e = 0; e < 4; ++e) {
          if (col + e >= n) break;
          float x = v[e];
          if (bias) x += bias[col + e];
          to[e] = add ? to[e] + x : x;
        }
      }
    }
  }
}

// Measured on the MI355X, us now and before runs of K, fetches of four lanes a row and the tiles for them (in a graph, weights in turn):
//   rows 8: N 4,096 K 1,024 5.7 (7.6), N 1,024 K 2,048 6.5 (11.7) and K 3,072 7.7 (16.0), N 6,144 K 1,024 7.9 (10.5), N 151,936 K 1,024 119 (139);
//   rows 32: 7.7 (10.1), 9.9 (15.1), 12.7 (20.4), 13.0 (17.1); rows 256: 23 (23), 18 (28), 24 (38), 38 (45);
//   rows 509: 39 (38), 23 (27), 32 (38), 53 (53); rows 2,048: N 24,576 K 4,096 2,978, 138 TFLOP/s of the 139 that the instruction alone reaches.
// What bounds them: many rows the matrix units; few rows the node of a graph, a trip for the first slices and the chains of a run, 13.3 ns
// for four k; the head memory (6.2 TB/s would make 100).
// What a launch of BN x BM tiles costs, by the outputs of the compute unit that has the most of them; `per_output` is how much
// longer a small tile takes an output (it reads more from the L2s for each).
int tile_cost(int m, int n, int bn, int bm, int per_output) {
  const int tiles = ((n + bn - 1) / bn) * ((m + bm - 1) / bm);
  return (tiles + 255) / 256 * (bn * bm / 64) * per_output;
}

}  // namespace

// The tile of a product of more than 16 rows, weight rows times 1,024 plus input rows: the one whose busiest compute unit has least to
// do, small tiles marked up by what they measured.
LRS_API int lrs_gemm_f32_tile(int m, int n) {
  const int small = tile_cost(m, n, 16, 32, 18), middle = tile_cost(m, n, 64, 32, 13), large = tile_cost(m, n, 64, 64, 11), largest = tile_cost(m, n, 128, 128, 10);
  if (small <= middle && small <= large && small <= largest) return 16 * 1024 + 32;
  if (middle <= large && middle <= largest) return 64 * 1024 + 32;
  return large <= largest ? 64 * 1024 + 64 : 128 * 1024 + 128;
}

// K % 32 == 0; a, w and rows of lda floats 16-byte aligned.  GATED: silu(gate) * up of weight rows interleaved in groups of 8, out [m, n / 2].
template <bool GATED>
static int launch_f32(float* out, bool add, const float* a, const float* w, const float* bias, int m, int n, int k, int lda, int ldc, hipStream_t s) {
  const int wide_stores = ldc % 4 == 0 && (uintptr_t)out % 16 == 0;
#define TILES(QUADS, BK, PARTS, WN, WM, TN, TM, STAGES, WR, AR)                                                                           \
  do {                                                                                                                             \
    const int tiles_m = (m + WM * TM * AR - 1) / (WM * TM * AR), tiles_n = (n + WN * TN * WR - 1) / (WN * TN * WR);                \
    gemm_f32_mfma_kernel<GATED, QUADS, BK, PARTS, WN, WM, TN, TM, STAGES, WR, AR><<<tiles_m * tiles_n, PARTS * WN * WM * WAVE, 0, s>>>(   \
        a, w, m, n, k, lda, tiles_m, tiles_m * tiles_n, out, add, ldc, bias, wide_stores);                                                \
  } while (0)
  if (m <= 16) {
    // Few rows: memory and the chains bound it.  As many workgroups as there are tiles of 16 weight rows, of 8 where those are
    // fewer than half the compute units (N under 2,048), a wave for each run of K; a head's many rows in workgroups of
    // 64, which share the input rows (119 us; a wave for each run and 16 weight rows 137).
    const bool pairs = k % 64 == 0, half = m <= 8;
    // Gated products take a wave for each run further, until the rows of every workgroup weigh more than the weights (shared / a wave for each
    // run: N 24,576 K 4,096 8 rows 84.2 / 78.8, 12 81.4 / 80.3, 16 82.6 / 87; N 34,816 K 5,120 8 rows 164 / 148, 12 162 / 165, 16 163 / 181;
    // N 51,200 K 5,120 4 rows 206 / 195, 8 202 / 206, 16 211 / 262; N 17,408 K 4,096 16 rows 82 / 72).
    const bool shared = n > 16384 && (!GATED || (int64_t)m * n >= 24 * 16384);
    if (shared && pairs) TILES(true, 64, 1, 4, 1, 1, 1, 4, 16, 16);
    else if (!pairs) TILES(false, 32, 1, 1, 1, 1, 1, 15, 16, 16);
    else if (n >= 2048 || GATED) { if (half) TILES(true, 64, 4, 1, 1, 1, 1, 3, 16, 8); else TILES(true, 32, 4, 1, 1, 1, 1, 4, 16, 16); }
    else if constexpr (!GATED) {
      if (half) TILES(true, 64, 4, 1, 1, 1, 1, 8, 8, 8);
      else TILES(true, 64, 4, 1, 1, 1, 1, 6, 8, 16);
    }
  } else {
    switch (lrs_gemm_f32_tile(m, n)) {
      case 16 * 1024 + 32:
        // a wave for each run of K with two chains, where K is long enough for more than one run (K 3,072, 17 to 128 rows: 12-14 us for 17-21)
        if (f32_part(k) < k) TILES(true, 32, 4, 1, 1, 1, 2, 6, 16, 16);
        else TILES(false, 32, 1, 1, 2, 1, 1, 12, 16, 16);
        break;
      case 64 * 1024 + 32:
        // a wave for each run with eight chains, no barrier in the walk: K 3,072, 509 rows 34 us for 39
        if (f32_part(k) < k) TILES(true, 32, 4, 1, 1, 4, 2, 3, 16, 16);
        else TILES(false, 32, 1, 2, 2, 2, 1, 8, 16, 16);
        break;
      case 64 * 1024 + 64: TILES(false, 32, 1, 2, 2, 2, 2, 3, 16, 16); break;
      default: TILES(false, 32, 1, 2, 4, 4, 2, 3, 16, 16);
    }
  }
#undef TILES
  return 0;
}

int lrs_gemm_f32(float* out, bool add, const float* a, const float* w, const float* bias, int m, int n, int k, int lda, int ldc, hipStream_t s) {
  return launch_f32<false>(out, add, a, w, bias, m, n, k, lda, ldc, s);
}

// out [M, N / 2] (row stride ldc) = silu(gate) * up, float32, where a [M, K] (row stride lda) times w[N, K]^T gives 8 gate columns, then the 8 up
// columns of the same features, and so on: the sums and the activation of lrs_gemm and lrs_silu_mul, bit for bit, without the
// kernel between and its two trips through memory (8 rows of N 6,144: 5 us a layer; 509 rows 6).
LRS_API int lrs_gemm_f32_gated(float* out, const float* a, const float* w, int m, int n, int k, int lda, int ldc, void* stream) {
  LRS_REQUIRE(m > 0 && n > 0 && k > 0 && n % 16 == 0 && k % 32 == 0 && lda >= k && ldc >= n / 2, "gemm_f32_gated: takes N %% 16 == 0 and K %% 32 == 0, got m=%d n=%d k=%d lda=%d ldc=%d", m, n, k, lda, ldc);
  LRS_REQUIRE(lda % 4 == 0 && ldc % 4 == 0 && (((uintptr_t)out | (uintptr_t)a | (uintptr_t)w) % 16) == 0 && (int64_t)128 * (lda > k ? lda : k) < (1ll << 30),
              "gemm_f32_gated: needs 16-byte aligned rows (lda=%d ldc=%d)", lda, ldc);
  if (int rc = launch_f32<true>(out, false, a, w, nullptr, m, n, k, lda, ldc, (hipStream_t)stream)) return rc;
  return lrs_check_launch("gemm_f32_gated");
}
