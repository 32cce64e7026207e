// bf16 products of many rows in tiles (gemm_tiles.hip): which tile and how many parts of K, and the launch.
#pragma once

#include "common.h"

extern "C" int lrs_compute_units();

// What becomes of an output: stored as bf16, stored as float32, added into float32, or silu(gate) * up of weight rows interleaved in
// groups of 8, stored as bf16.  The first three are the modes of lrs_gemm.
enum { TILES_STORE = 0, TILES_STORE_F32 = 1, TILES_ADD_F32 = 2, TILES_GATED = 3 };

struct TilesChoice {
  int tile, splits;
  float us;                                                       // what it is expected to take, the kernel that adds up the parts included
  float useful;                                                   // of what the chip makes in the rounds of such a launch, the product's own outputs
};
// Products of up to 64 outputs that tiles take rather than gemm_bf16_narrow, whose workgroups of 16 rows and all outputs are one round of the chip up
// to 4,096 rows.  us, narrow / tiles: K 4,096 8 outputs 4,096 rows 11.4 / 13.3, 8,192 19.7 / 17.7; 32 outputs 4,096 rows 17.3 / 13.9, 64 24.4 / 14.1; K 2,048
// 4,096 rows 8 outputs 7.9 / 11.5, 6,000 13.3 / 11.7; K 8,192 4,096 rows 8 outputs 16.9 / 18.4, 64 41 / 19.4.
constexpr int FEW_OUTPUTS = 128;
bool tiles_take_few_outputs(int m, int k);

// The least by measured costs; sums_bytes: room for the parts' sums.  Depends on its arguments and the number of compute units alone.
TilesChoice choose_tiles(int m, int n, int k, size_t sums_bytes);
// x [m, k] (row stride lda), w [n, k]; with splits > 1 out is [splits, m, ldc] float32 and form TILES_STORE_F32.
void launch_tiles(const TilesChoice& choice, void* out, int form, const bf16* x, const bf16* w, int m, int n, int k, int lda, int ldc, hipStream_t s);
