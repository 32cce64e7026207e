// bf16 products of many rows: y = x W^T with both operands through LDS in slices of 64 k (whole 128-byte lines of every row), tiles of
// 256 or 128 tokens x 64 to 256 weight rows, two groups of four waves in turn.
#include "gemm_tiles.h"

#include "lines_walk.h"

// A workgroup of eight waves owns WM * JT * 16 tokens x (8 / WM) * IT * 16 weight rows; a wave JT x IT tiles of the 16x16x32 product.
// K is walked in slices of 64 * PANELS, whole or in two halves of the wave's tokens (HALVES), STAGES of them in LDS (lines_walk.h).
//
// What bounds it: the large tiles by the matrix cores' power.  8B gate_up at 2,048 rows (three rounds of 256 x 256) 291 us (1.42 PFLOP/s; 327
// before), on another card 317, there without fetches 280, without reads as well 262, the matrix instructions alone 259 (1.59); with
// operands of zeros 259, 229, 218 and 215: what is left is the clock, not a wait.  The L2s hand out 22-26 TB/s to such fetches.  4B gate_up at
// 512 rows (244 tiles of 256 x 160) 51 us (72), 8B down at 512 rows (256 x 128, K in four) with its norm 59 (66), 1.7B gate_up at
// 2,048 (256 x 192) 90 (104).  32x32x16 products instead: a tenth slower.  The small tiles by their steps' beginnings, which is why
// they take slices of 128 whole: 1.7B q/k/v at 256 rows (64 x 64) 12.2 us, in slices of 64 14.0, of 128 x 64 in halves 18.2.
//
// Rows past a matrix are read from its last row and never written.
// Needs K % (64 * PANELS) == 0, 16-byte aligned rows, N % 4 == 0, matrices of fewer than 2^31 elements.
// With K divided (splits > 1) a workgroup walks its part of the slices and leaves its sums in part `split` of out [splits, m, ldc].
// The sums of an output are one chain over its K in steps of 32, whatever the tile: bits depend on the parts alone.
__device__ __forceinline__ float silu_of(float v) { return v / (1.f + __expf(-v)); }

template <int WM, int JT, int IT, int PANELS, int HALVES, int STAGES>
__global__ __launch_bounds__(512, 1) void gemm_bf16_tiles_kernel(const bf16* __restrict__ x, const bf16* __restrict__ w, int m, int n, int k, int lda,
                                                                 int tiles_m, int tiles_n, int splits, int chunk, void* __restrict__ out, int form, int ldc) {
  constexpr int WN = 8 / WM, BM = WM * JT * 16, BN = WN * IT * 16, BK = 64 * PANELS;
  constexpr int X_BLOCKS = BM / 8 / HALVES, W_BLOCKS = BN / 8;   // blocks of 8 rows of a panel: of a part of the tokens, of the weights
  static_assert(X_BLOCKS * PANELS % 8 == 0 && JT % HALVES == 0, "a part of the tokens is dealt evenly to eight waves");
  constexpr int NX = X_BLOCKS * PANELS / 8, NW = W_BLOCKS * PANELS / 8, REST = W_BLOCKS * PANELS % 8;   // fetches a wave; REST: one more of the weights for the first waves
  constexpr int STAGE_ELEMENTS = (BM + BN) * BK;
  __shared__ __attribute__((aligned(64))) bf16 slices[STAGES * STAGE_ELEMENTS];   // a stage: the tokens' panels, then the weights'
  const int tid = threadIdx.x, lane = tid % WAVE, wave = __builtin_amdgcn_readfirstlane(tid / WAVE);
  const int r = lane & 15, g = lane >> 4;
  int id = (blockIdx.x % 8) * chunk + blockIdx.x / 8;            // consecutive workgroups go to different XCDs: a run of tiles to each
  const int tiles = tiles_m * tiles_n;
  if (id >= tiles * splits) return;
  const int split = id / tiles;
  id -= split * tiles;
  const int band = id / (4 * tiles_n), within = id % (4 * tiles_n);
  const int band_rows = tiles_m - band * 4 < 4 ? tiles_m - band * 4 : 4;
  const int m0 = (band * 4 + within % band_rows) * BM, n0 = (within / band_rows) * BN;
  const int wm = wave / WN, wn = wave % WN;
  const int place_row = lines_place_row(lane), place_chunk = lines_place_chunk(lane);
  unsigned x_off[HALVES][NX], x_to[HALVES][NX], w_off[NW + 1];   // bytes from the matrix's first element, from the stage's first
#pragma unroll
  for (int h = 0; h < HALVES; ++h)
#pragma unroll
    for (int i = 0; i < NX; ++i) {
      const int b = wave + 8 * i, panel = b / X_BLOCKS, of = b % X_BLOCKS;
      const int first = HALVES == 2 ? ((of / JT) * 2 + h) * 8 * JT + (of % JT) * 8 : of * 8;   // a wave's half is JT blocks
      const int row = m0 + first + place_row;
      x_to[h][i] = (panel * BM + first) * 128;
      x_off[h][i] = ((unsigned)(row < m ? row : m - 1) * (unsigned)lda + panel * 64 + place_chunk * 8) * 2u;
    }
#pragma unroll
  for (int i = 0; i < NW + (REST ? 1 : 0); ++i) {
    const int b = wave + 8 * i, panel = b / W_BLOCKS, row = n0 + 8 * (b % W_BLOCKS) + place_row;
    w_off[i] = ((unsigned)(row < n ? row : n - 1) * (unsigned)k + panel * 64 + place_chunk * 8) * 2u;
  }
  floatx4 acc[IT][JT];
#pragma unroll
  for (int it = 0; it < IT; ++it)
#pragma unroll
    for (int jt = 0; jt < JT; ++jt) acc[it][jt] = floatx4{0.f, 0.f, 0.f, 0.f};
  const int steps_of_k = k / BK, steps_each = (steps_of_k + splits - 1) / splits, step0 = split * steps_each;
  const int steps = steps_of_k - step0 < steps_each ? steps_of_k - step0 : steps_each;
  const unsigned slices_address = (unsigned)(uintptr_t)(__attribute__((address_space(3))) bf16*)slices;
  const bool one_more = REST != 0 && wave < REST;
  auto fetch_x = [&](int h, int s, int stage) {
    const int at = (step0 + s) * BK * 2;
    const unsigned to = slices_address + (unsigned)(stage * STAGE_ELEMENTS * 2);
#pragma unroll
    for (int i = 0; i < NX; ++i) fetch_to_lds((const char*)x + at, x_off[h][i], to + x_to[h][i]);
  };
  auto fetch_w = [&](int s, int stage) {
    const int at = (step0 + s) * BK * 2;
    const unsigned to = slices_address + (unsigned)((stage * STAGE_ELEMENTS + BM * BK) * 2 + wave * 1024);
#pragma unroll
    for (int i = 0; i < NW; ++i) fetch_to_lds((const char*)w + at, w_off[i], to + (unsigned)(i * 8192));
    if (REST != 0 && one_more) fetch_to_lds((const char*)w + at, w_off[NW], to + (unsigned)(NW * 8192));
  };
  walk_in_turns<HALVES, PANELS, STAGES, NX, NW, REST != 0>(acc, slices, BM, BN, wm * JT * 16, wn * IT * 16, steps, one_more, fetch_x, fetch_w);
  int m0_opaque = m0;                                              // nothing of what follows is worked out before the loop ends
  asm volatile("" : "+s"(ldc), "+s"(m0_opaque));
#pragma unroll
  for (int jt = 0; jt < JT; ++jt) {
    const int token = m0_opaque + (wm * JT + jt) * 16 + r;
    const int64_t row_at = ((int64_t)split * m + token) * ldc;
#pragma unroll
    for (int it = 0; it < IT; ++it) {
      const int tile0 = n0 + (wn * IT + it) * 16, row0 = tile0 + 4 * g;   // this lane's four weight rows = output columns
      const floatx4 v = acc[it][jt];
      if (form == TILES_GATED) {
        // a tile's 16 weight rows are 8 gate rows and the 8 up rows of the same features: the up values of a lane's gate rows are
        // held by the lane 32 further on
        floatx4 up;
#pragma unroll
        for (int i = 0; i < 4; ++i) up[i] = __shfl(v[i], (lane + 32) % WAVE, WAVE);
        if (g < 2 && token < m && tile0 + 15 < n)
          *(bf16x4*)((bf16*)out + row_at + tile0 / 2 + 4 * g) =
              bf16x4{(bf16)(silu_of(v[0]) * up[0]), (bf16)(silu_of(v[1]) * up[1]), (bf16)(silu_of(v[2]) * up[2]), (bf16)(silu_of(v[3]) * up[3])};
      } else if (token < m && row0 < n) {
        if (form == TILES_STORE) *(bf16x4*)((bf16*)out + row_at + row0) = bf16x4{(bf16)v[0], (bf16)v[1], (bf16)v[2], (bf16)v[3]};
        else if (form == TILES_STORE_F32) *(floatx4*)((float*)out + row_at + row0) = v;
        else *(floatx4*)((float*)out + row_at + row0) = *(const floatx4*)((const float*)out + row_at + row0) + v;
      }
      __builtin_amdgcn_sched_barrier(0);
    }
  }
}

// The tiles, and what a launch of them takes: us = rounds of the chip * (fixed + slices of 64 k * (slice + crowd * share of the chip in use)),
// fitted to 106 to 617 launches of each, at 144 to 2,048 rows of the 0.6B, 1.7B, 4B and 8B layers' products with K in 1 to 8 parts (half
// of them within 5 %, nine in ten within 12 %; a fuller chip runs slower: its clock).  What the least of these takes is within 0.3 % of
// the best of all launches on the mean, 6 % at most (weights from memory, 140 to 256 rows of q/k/v and o: 4 % on the mean, 13 % at most).  Outside the fit: 65 to 128
// rows of seven sizes whose K is no multiple of 256, 1.3 to 7 times as fast as in the slices of 32 of gemm_bf16_wide; beyond 2,048 rows see lrs_gemm_tiles_pay.  panels: slices of 64 k
// a step (K a multiple of so many).  Worked out at every launch that is not recorded: under 1 us of the host.
struct TileShape { int bm, bn, panels; float fixed, slice, crowd; };
constexpr TileShape TILES[] = {{256, 256, 1, 12.0f, 0.81f, 0.66f}, {256, 192, 1, 9.7f, 0.69f, 0.51f}, {256, 160, 1, 8.9f, 0.58f, 0.45f},
                               {256, 128, 1, 7.7f, 0.50f, 0.38f}, {128, 256, 1, 8.1f, 0.52f, 0.37f}, {128, 192, 1, 6.5f, 0.48f, 0.25f},
                               {128, 128, 2, 5.8f, 0.37f, 0.17f}, {64, 128, 2, 4.1f, 0.28f, 0.08f}, {64, 64, 2, 3.0f, 0.23f, 0.03f}};
// Sums of parts: a kernel more, or more work for the one that adds the residual, and every part's sums written and read once, most of it in the caches.
constexpr float PARTS_FIXED = 2.f, PARTS_BYTES_A_US = 14e6f;

bool tiles_take_few_outputs(int m, int k) { return (m > 4096 && k >= 512) || (m == 4096 && k >= 4096); }

// Few outputs (up to STREAM_OUTPUTS) of rows that the memory-side cache does not hold are a matter of reading those rows.  Parts that begin a multiple of 4 KB
// into a row read them more slowly (K 8,192, 16,384 rows of 192 and 256 outputs in four parts of 4 KB 97 and 108 us, whole 76 and 87; 32,768 rows in two of 8 KB
// 167 and 180, whole 146 and 170), and parts that promise less than a tenth are no faster (28,000 rows of K 5,120, 128 outputs in two 80, whole 70).  Others
// are: 17,000 rows of K 8,192 in three parts 85 and 98, whole 97 and 117; 5,000 of K 28,672 in six 86 and 97, whole 133 and 182; 8 outputs 52, whole 108.
constexpr int64_t CACHED_BYTES = 256ll << 20;
constexpr int STREAM_OUTPUTS = 256, SLOW_APART = 32;               // SLOW_APART: slices
constexpr float STREAM_GAIN = 1.1f;

TilesChoice choose_tiles(int m, int n, int k, size_t sums_bytes) {
  const int units = lrs_compute_units() > 0 ? lrs_compute_units() : 256, steps = k / 64;
  // Up to FEW_OUTPUTS have the same parts, those of so many, and none where some of them go to gemm_bf16_narrow: a router's logits keep the bits
  // that they have beside more weight rows.
  const bool few = n <= FEW_OUTPUTS;
  const bool whole = few && !tiles_take_few_outputs(m, k), streams = n <= STREAM_OUTPUTS && (int64_t)m * k * 2 >= CACHED_BYTES;
  // the least for n outputs with 1 to `most` parts
  auto least = [&](int n, int most) {
    TilesChoice best{0, 1, 0.f};
    for (int t = 0; t < (int)(sizeof(TILES) / sizeof(TILES[0])); ++t) {
      const TileShape& shape = TILES[t];
      if (k % (64 * shape.panels) != 0) continue;
      const int64_t tiles = (int64_t)((m + shape.bm - 1) / shape.bm) * ((n + shape.bn - 1) / shape.bn);
      for (int parts = 1; parts <= most; ++parts) {
        const int each = (steps / shape.panels + parts - 1) / parts * shape.panels;   // slices of the longest part
        const double sums = (double)parts * m * n * sizeof(float);
        // every part has work, and eight slices of it: shorter walks are mostly beginnings
        if (parts > 1 && (each < 8 || (parts - 1) * each >= steps || sums > (double)sums_bytes || tiles * parts > units || (streams && each % SLOW_APART == 0))) continue;
        const int64_t rounds = (tiles * parts + units - 1) / units;
        const float share = (float)(tiles * parts) / (float)(rounds * units);
        float us = (float)rounds * (shape.fixed + (float)each * (shape.slice + shape.crowd * share));
        if (parts > 1) us += PARTS_FIXED + 2.f * (float)sums / PARTS_BYTES_A_US;
        if (best.us == 0.f || us < best.us) {
          best = TilesChoice{t, parts, us, (float)((double)parts * m * n / ((double)rounds * units * shape.bm * shape.bn))};
        }
      }
    }
    return best;
  };
  const int counted = few ? FEW_OUTPUTS : n;
  TilesChoice best = least(counted, whole ? 1 : 8);
  if (streams && best.splits > 1) {
    const TilesChoice undivided = least(counted, 1);
    if (undivided.us <= STREAM_GAIN * best.us) best = undivided;
  }
  return few && best.splits == 1 ? least(n, 1) : best;            // (a sum's bits are the parts' alone: undivided, fewer outputs may take smaller tiles)
}

void launch_tiles(const TilesChoice& choice, void* out, int form, const bf16* x, const bf16* w, int m, int n, int k, int lda, int ldc, hipStream_t s) {
  const TileShape& shape = TILES[choice.tile];
  const int tiles_m = (m + shape.bm - 1) / shape.bm, tiles_n = (n + shape.bn - 1) / shape.bn, chunk = (tiles_m * tiles_n * choice.splits + 7) / 8;
#define TILES_OF(...) gemm_bf16_tiles_kernel<__VA_ARGS__><<<chunk * 8, 512, 0, s>>>(x, w, m, n, k, lda, tiles_m, tiles_n, choice.splits, chunk, out, form, ldc)
  switch (choice.tile) {
    case 0: TILES_OF(2, 8, 4, 1, 2, 2); break;
    case 1: TILES_OF(2, 8, 3, 1, 2, 2); break;
    case 2: TILES_OF(4, 4, 5, 1, 1, 3); break;
    case 3: TILES_OF(4, 4, 4, 1, 1, 3); break;
    case 4: TILES_OF(2, 4, 4, 1, 1, 3); break;
    case 5: TILES_OF(2, 4, 3, 1, 1, 4); break;
    case 6: TILES_OF(2, 4, 2, 2, 2, 2); break;
    case 7: TILES_OF(2, 2, 2, 2, 1, 3); break;
    default: TILES_OF(4, 1, 2, 2, 1, 4); break;
  }
#undef TILES_OF
}

// (tokens, weight rows) of the tile and the parts of K for a product, with `sums_bytes` of room for the parts' sums; a choice of this process's
// device, the same at every call.
LRS_API int lrs_gemm_tiles_choice(int m, int n, int k, int64_t sums_bytes, int* bm, int* bn, int* splits) {
  LRS_REQUIRE(m > 0 && n > 0 && k > 0 && k % 64 == 0 && sums_bytes >= 0 && bm && bn && splits, "gemm_tiles_choice: takes positive sizes, K %% 64 == 0, got m=%d n=%d k=%d", m, n, k);
  const TilesChoice choice = choose_tiles(m, n, k, (size_t)sums_bytes);
  *bm = TILES[choice.tile].bm, *bn = TILES[choice.tile].bn, *splits = choice.splits;
  return 0;
}
