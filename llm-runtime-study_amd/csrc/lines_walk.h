// A walk over K for products of many bf16 rows (gemm_tiles.hip, the routed experts' in moe.hip): a workgroup of eight waves, its tile of x
// rows times weight rows, slices of 64 * PANELS of K, so that every fetch brings whole 128-byte lines, brought into LDS by memory
// itself (fetch_to_lds).
//
// Where chunk c (8 k, 16 bytes) of tile row q lies in a panel (64 of K): rows are 128 bytes, eight to a block of 1,024 bytes (one fetch of
// one wave, whose lane l fills place l), and the chunks of a row are turned round by twice (q / 2) % 4, so that the lanes LDS serves
// together (eight consecutive rows, chunks g and g + 1) meet every bank once: place (q % 8) * 8 + (c ^ ((q >> 1 & 3) << 1)) of block
// q / 8.  A stage: the x rows' panels, then the weight rows'.
#pragma once

#include "common.h"

constexpr int LINES_BK = 64;

// The row and the chunk that lane l of a fetch brings: place l of its block of eight rows.
__device__ __forceinline__ int lines_place_row(int lane) { return lane >> 3; }
__device__ __forceinline__ int lines_place_chunk(int lane) { return (lane & 7) ^ ((lane >> 4 & 3) << 1); }

template <int N>
__device__ __forceinline__ void wait_fetches() {
  asm volatile("s_waitcnt vmcnt(%0)" :: "n"(N) : "memory");
}
__device__ __forceinline__ void have_read_then_barrier() { asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory"); }
__device__ __forceinline__ void barrier_alone() { asm volatile("s_barrier" ::: "memory"); }

// acc[it][jt] += the products of weight rows wn + 16 it .. and x rows wm + 16 jt .. over slices 0 .. steps - 1, in steps of 32 of K in order.
// fetch_x(h, s, stage) asks for this wave's NX pieces of slice s of the x rows of every wave's part h, fetch_w(s, stage) for its NW pieces of
// the weight rows, one more if `one_more` (SOME_MORE: of some waves).
//
// A slice is taken whole, or in two halves of the wave's x rows (HALVES; what the registers and LDS of the largest tiles ask for): a step
// of reading (the fragments; those of the weights stay in registers for the second half) and a step of multiplying, with a barrier
// behind each.  Waves 4..7 are one step behind waves 0..3, and a SIMD has one of either: while one multiplies, the other reads LDS and
// asks memory for a slice to come.  So neither kind of work waits for the other, where waves in step all read, then all multiplied
// (the dense products 8B gate_up 2,048 rows 327 us for 291; with the barrier in the middle of a slice, second-half reads among the
// first half's products, 320).
//
// What may be asked for when.  A wave has what it read before the barrier that ends its step of reading.
// Whole slices: waves 0..3 read slice s in step 2 s, waves 4..7 in step 2 s + 1.  Behind that its place is free, and every wave asks for
// slice s + STAGES in its next step of reading (steps 2 s + 2 and 2 s + 3).  Before the barrier that ends a step of reading, of slice s, a
// wave waits until only the last STAGES - 2 slices are on their way: slice s + 1 is then there (steps 2 s and 2 s + 1) before anyone reads
// it (step 2 s + 2).
// Halves: waves 0..3 read the first half of slice s in step 4 s and the second in step 4 s + 2, waves 4..7 in steps 4 s + 1 and 4 s + 3.  The
// first half of x and the weights of s are read by everybody when step 4 s + 1 ends, and every wave asks for those of s + STAGES when it
// reads the second half of s (steps 4 s + 2 and 4 s + 3); the second half of s is free when step 4 s + 3 ends, and is asked for again when
// the first half of s + 1 is read (steps 4 s + 4 and 4 s + 5).  A wave waits until only the last STAGES - 1 slices' worth is on its way: at
// the end of reading the second half of s (steps 4 s + 2 and 4 s + 3) the first half and the weights of s + 1 are there, read from step
// 4 s + 4 on; at the end of reading the first half of s + 1 (steps 4 s + 4 and 4 s + 5) its second half, read from step 4 s + 6 on.
// Once there are no more slices to ask for, a wave waits for all it has asked for.
// (Three stages of the weights, which come from memory, beside two of x: 8B gate_up 299 -> 312 us, routed experts the same times.)
template <int HALVES, int PANELS, int STAGES, int NX, int NW, bool SOME_MORE, int IT, int JT, typename FetchX, typename FetchW>
__device__ __forceinline__ void walk_in_turns(floatx4 (&acc)[IT][JT], const bf16* slices, int x_rows, int w_rows, int wm, int wn, int steps, bool one_more,
                                              FetchX&& fetch_x, FetchW&& fetch_w) {
  static_assert(HALVES == 2 ? STAGES >= 2 : STAGES >= 3, "slices on their way while one is multiplied");
  constexpr int JH = JT / HALVES, STEPS = 2 * PANELS, EACH = HALVES * NX + NW, AHEAD = HALVES == 2 ? STAGES - 1 : STAGES - 2;
  const int lane = threadIdx.x % WAVE, wave = __builtin_amdgcn_readfirstlane(threadIdx.x / WAVE), r = lane & 15, g = lane >> 4;
  const int stage_elements = (x_rows + w_rows) * LINES_BK * PANELS;
  // this lane's fragment of rows 16 j .. 16 j + 15, k half c of a panel: row r, chunk 4 c + g
  const int frag_row = (r >> 3) * 512 + (r & 7) * 64, turn = ((r >> 1) & 3) << 1;
  const int frag[2] = {frag_row + ((g ^ turn) * 8), frag_row + (((4 + g) ^ turn) * 8)};
  auto fetch_first = [&](int s, int stage) {
    if (s >= steps) return;
    fetch_x(0, s, stage);
    fetch_w(s, stage);
  };
  auto fetch_second = [&](int s, int stage) {
    if (s < steps) fetch_x(1, s, stage);
  };
  auto wait = [&](bool more_to_come) {
    if (!more_to_come) wait_fetches<0>();
    else if (SOME_MORE && one_more) wait_fetches<AHEAD * (EACH + 1)>();
    else wait_fetches<AHEAD * EACH>();
  };
#pragma unroll
  for (int s = 0; s < AHEAD + 1; ++s) {
    fetch_first(s, s);
    if (HALVES == 2 && s < AHEAD) fetch_second(s, s);
  }
  wait(AHEAD < steps);
  barrier_alone();
  if (wave >= 4) barrier_alone();                                  // a step behind from here on
  int stage = 0;
  bf16x8 wf[STEPS][IT], xf[STEPS][JH];
  auto multiply = [&](int first) {
    __builtin_amdgcn_sched_barrier(0);
#pragma unroll
    for (int c = 0; c < STEPS; ++c)
#pragma unroll
      for (int it = 0; it < IT; ++it)
#pragma unroll
        for (int jt = 0; jt < JH; ++jt) acc[it][first + jt] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(wf[c][it], xf[c][jt], acc[it][first + jt], 0, 0, 0);
    __builtin_amdgcn_sched_barrier(0);
    barrier_alone();
  };
  for (int s = 0; s < steps; ++s) {
    const bf16* xs = slices + stage * stage_elements;
    const bf16* ws = xs + x_rows * LINES_BK * PANELS;
    const int before = stage == 0 ? STAGES - 1 : stage - 1;
    auto read_x = [&](int first) {
#pragma unroll
      for (int c = 0; c < STEPS; ++c)
#pragma unroll
        for (int jt = 0; jt < JH; ++jt) xf[c][jt] = *(const bf16x8*)(xs + frag[c % 2] + (c / 2 * x_rows + wm + (first + jt) * 16) * LINES_BK);
    };
#pragma unroll
    for (int c = 0; c < STEPS; ++c)
#pragma unroll
      for (int it = 0; it < IT; ++it) wf[c][it] = *(const bf16x8*)(ws + frag[c % 2] + (c / 2 * w_rows + wn + it * 16) * LINES_BK);
    read_x(0);
    if constexpr (HALVES == 2) fetch_second(s + STAGES - 1, before);
    else fetch_first(s + STAGES - 1, before);
    wait(s + STAGES - 1 < steps);
    have_read_then_barrier();
    multiply(0);
    if constexpr (HALVES == 2) {
      read_x(JH);
      fetch_first(s + STAGES, stage);
      wait(s + STAGES < steps);
      have_read_then_barrier();
      multiply(JH);
    }
    stage = stage == STAGES - 1 ? 0 : stage + 1;
  }
  if (wave < 4) barrier_alone();                                   // as many barriers for every wave
}
