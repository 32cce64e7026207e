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
};
// The least by measured costs; sums_bytes: room for the parts' sums.  Depends on its arguments and the number of compute units alone.
TilesChoice choose_tiles(int m, int n, int k, size_t sums_bytes);
// x [m, k] (row stride lda), w [n, k]; with splits > 1 out is [splits, m, ldc] float32 and form TILES_STORE_F32.
void launch_tiles(const TilesChoice& choice, void* out, int form, const bf16* x, const bf16* w, int m, int n, int k, int lda, int ldc, hipStream_t s);
