// A walk over K for products of many bf16 rows (the routed experts', moe.hip): a workgroup's tile of x rows times weight rows, slices of
// 64 of K, so that every fetch brings whole 128-byte lines, brought into LDS by memory itself (fetch_to_lds).
//
// (In the dense products of gemm.hip, whose tiles have this layout too, the walk made no difference: 8192^3 865 us for 867, where the
// clock is what bounds them; up to 1,024 rows 5-10 % less at tiles of 256 x 256, which go to the vendor library, and 2-5 % more at 256 x 128.)
//
// Where chunk c (8 k, 16 bytes) of tile row q lies in a stage: rows are 128 bytes, eight to a block of 1,024 bytes (one fetch of one
// wave, whose lane l fills place l), and the chunks of a row are turned round by twice (q / 2) % 4, so that the lanes LDS serves
// together (eight consecutive rows, chunks g and g + 1) meet every bank once: place (q % 8) * 8 + (c ^ ((q >> 1 & 3) << 1)) of block
// q / 8.  The x rows come first, the weight rows behind them.
#pragma once

#include "common.h"

constexpr int LINES_BK = 64;

// The row and the chunk that lane l of a fetch brings: place l of its block of eight rows.
__device__ __forceinline__ int lines_place_row(int lane) { return lane >> 3; }
__device__ __forceinline__ int lines_place_chunk(int lane) { return (lane & 7) ^ ((lane >> 4 & 3) << 1); }

// acc[it][jt] += the products of weight rows wn + 16 it .. and x rows wm + 16 jt .. over slices 0 .. steps - 1.
// fetch(slice, stage) asks for this wave's EACH pieces of a slice (of the last one for slices past it).
//
// A turn multiplies the two halves of a slice (32 of K each).  While the first half's products run, the second half's fragments are
// read; then every wave has read the slice, and the barrier stands here, in the middle: behind it the slice's stage is filled again,
// the next slice is there, and its first half's fragments are read while the second half's products run, whose operands are in
// registers already.  With the barrier between two slices every wave began each of them with nothing to multiply until its first
// fragments came from LDS, and reads and products took turns inside.
template <int STAGES, int EACH, int IT, int JT, typename Fetch>
__device__ __forceinline__ void lines_walk(floatx4 (&acc)[IT][JT], const bf16* slices, int x_rows, int w_rows, int wm, int wn, int steps, Fetch&& fetch) {
  const int lane = threadIdx.x % WAVE, r = lane & 15, g = lane >> 4;
  const int stage_elements = (x_rows + w_rows) * LINES_BK;
  // this lane's fragment of rows 16 j .. 16 j + 15, k half c: row r, chunk 4 c + g
  const int frag_row = (r >> 3) * 512 + (r & 7) * 64, turn = ((r >> 1) & 3) << 1;
  const int frag[2] = {frag_row + ((g ^ turn) * 8), frag_row + (((4 + g) ^ turn) * 8)};
  struct Half {
    bf16x8 x[JT], w[IT];
  };
  Half first, second;
  constexpr int READS = IT + JT, GROUPS = IT > 1 ? IT - 1 : 1, PER_GROUP = (READS + GROUPS - 1) / GROUPS;
  auto read = [&](Half& to, int n, int stage, int half) {             // the nth fragment of a half
    const bf16* at = slices + stage * stage_elements + frag[half];
    if (n < JT) to.x[n] = *(const bf16x8*)(at + (wm + n * 16) * LINES_BK);
    else to.w[n - JT] = *(const bf16x8*)(at + (x_rows + wn + (n - JT) * 16) * LINES_BK);
  };
  auto multiply = [&](const Half& with, Half& next, int stage, int half) {
#pragma unroll
    for (int it = 0; it < IT; ++it) {
#pragma unroll
      for (int jt = 0; jt < JT; ++jt) acc[it][jt] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(with.w[it], with.x[jt], acc[it][jt], 0, 0, 0);
#pragma unroll
      for (int n = it * PER_GROUP; n < (it + 1) * PER_GROUP && n < READS; ++n) read(next, n, stage, half);
      __builtin_amdgcn_sched_barrier(0);
    }
  };
#pragma unroll
  for (int s = 0; s < STAGES; ++s) fetch(s, s);
  fetched_and_read_then_barrier<(STAGES - 1) * EACH>();
  int stage = 0;
#pragma unroll
  for (int n = 0; n < READS; ++n) read(first, n, 0, 0);
  for (int kt = 0; kt < steps; ++kt) {
    multiply(first, second, stage, 1);
    fetched_and_read_then_barrier<(STAGES - 2) * EACH>();
    fetch(kt + STAGES, stage);
    stage = stage == STAGES - 1 ? 0 : stage + 1;
    multiply(second, first, stage, 0);
  }
  asm volatile("s_waitcnt vmcnt(0)" ::: "memory");                    // the fetches past K that nobody reads
}
