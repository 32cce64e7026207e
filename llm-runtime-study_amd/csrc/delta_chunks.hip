// The gated delta rule (delta.hip, one decay a head) over portions in bfloat16 runs: chunks of 64 tokens on the float32 matrix
// cores, the state carried from chunk to chunk.
//
// Within a chunk let D_ts be the product of the decays g behind token s up to token t (D_tt = 1), c_t that of all up to t and S0 the
// state before the chunk.  The rule of every token, u_t = beta_t (v_t - g_t S_{t-1}^T k_t), is a triangular system:
//     (1 + A) U = beta V - beta c K S0,   A_ts = beta_t D_ts (k_t . k_s) for s < t
//     O = c Q S0 + P U,                   P_ts = D_ts (q_t . k_s) for s <= t
//     S = c_L S0 + sum_s D_Ls k_s u_s^T
// What does not know S0 is made for all chunks at once: W' = -(1 + A)^-1 beta c K, V' = (1 + A)^-1 beta V, Q' = c Q + P W', O' = P V';
// left for the walk are U = V' + W' S0, O = O' + Q' S0 and the update of S.
//   delta_pack  per (chunk, head): those matrices, as operands of the walk's products;
//   delta_walk  per (request, head, 16 columns of S): walks the chunks with its part of S in accumulators.
// Precision: float32 as in the scan, sums in another order, and with it the queries' products with keys would make read-outs half as far
// again from those of 64 bits as the scan's.  So the nearest tokens' are made in 64 bits, a token's u is rounded as often as in the scan
// (exact_sum) and the state's update adds the last tokens one by one on top of the earlier ones (U's order).  Distance from 64 bits,
// here / in the scan, read-outs and states: a Nobodra layer's inputs (decays about 0.5) 6.4e-8 / 6.7e-8 and 4.8e-8 / 4.9e-8 (1.0e-7 and
// 6.6e-8 without all that); decays near one 1.5e-7 / 1.9e-7 and 1.1e-7 / 1.5e-7; keys that are nearly all alike under step sizes near one
// 4.2e-7 / 2.5e-7 and 5.9e-7 / 6.5e-7.  Decays are multiplied as the scan does and never divided, so decays of zero are no special case;
// the inverse holds products of contractions (1 - beta k k^T), none above one.
// A token whose inputs are infinite or NaN spoils itself and what comes after it, as in the scan, and no token before it.
//
// The matrix instructions are 16 x 16 x 4: of a block of 16 rows, lane 16 g + r gives or gets row r (column r) and, of every 16 of
// the inner size, the four 4 g .. 4 g + 3 in four instructions.  Sums come out with lane 16 g + r holding column r of the rows
// 4 g .. 4 g + 3, so a block of sums is at once a right operand of the next product.
//
// 32 heads of 128 x 128, one request of 2,048 tokens: 514 us in the scan, a chain of 2,048 turns with two lane sums each; here, inside a
// prompt, 84 us for the packs, some 5 of them for the precision above, and 105 for the walk.  Where the scan is the faster one (many
// portions, short ones) the part says.
#include "common.h"

extern "C" int lrs_delta_state_rows(int d);

namespace {

constexpr int L = 64;             // tokens of a chunk
constexpr int SPLIT = 16;         // lanes of a column in the state row's layout (delta.hip)
constexpr int BLOCK = 16 * 16;    // floats of a block of operands or sums

// A request's chunks lie side by side in the packs: request r's chunk c in slot cu[r] / L + r + c (requests never share one).
__device__ __forceinline__ int first_slot(const int* __restrict__ cu, int r) { return cu[r] / L + r; }

typedef double doublex4 __attribute__((ext_vector_type(4)));

__device__ __forceinline__ floatx4 mfma(float a, float b, floatx4 c) { return __builtin_amdgcn_mfma_f32_16x16x4f32(a, b, c, 0, 0, 0); }

// c + a b for a block of 16 x 16 x 16
__device__ __forceinline__ floatx4 product(const floatx4& a, const floatx4& b, floatx4 c) {
#pragma unroll
  for (int i = 0; i < 4; ++i) c = mfma(a[i], b[i], c);
  return c;
}

// A sum over many blocks, in four parts: a part's roundings are a quarter as many and of smaller numbers (with one chain the read-outs
// were twice as far from those of 64 bits as the scan's).
struct Sums {
  floatx4 part[4] = {};
  __device__ __forceinline__ void add(int j, const floatx4& a, const floatx4& b) { part[j % 4] = product(a, b, part[j % 4]); }
  // blocks j and j + 1, their instructions in turn: none waits for the one before it
  __device__ __forceinline__ void add_two(int j, const floatx4* a, const floatx4* b) {
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      part[j % 4] = mfma(a[j][i], b[j][i], part[j % 4]);
      part[(j + 1) % 4] = mfma(a[j + 1][i], b[j + 1][i], part[(j + 1) % 4]);
    }
  }
  __device__ __forceinline__ floatx4 total() const { return (part[0] + part[1]) + (part[2] + part[3]); }
};

// The four values of lane group g and the lane groups change places: value i of group g goes to value g of group i.
__device__ __forceinline__ floatx4 groups_for_values(floatx4 v) {
  typedef unsigned two __attribute__((ext_vector_type(2)));
  const two a = __builtin_amdgcn_permlane16_swap(__float_as_uint(v[0]), __float_as_uint(v[1]), false, false);
  const two b = __builtin_amdgcn_permlane16_swap(__float_as_uint(v[2]), __float_as_uint(v[3]), false, false);
  const two c = __builtin_amdgcn_permlane32_swap(a[0], b[0], false, false), d = __builtin_amdgcn_permlane32_swap(a[1], b[1], false, false);
  return floatx4{__uint_as_float(c[0]), __uint_as_float(d[0]), __uint_as_float(c[1]), __uint_as_float(d[1])};
}

// s times x plus c, as a sum and what its rounding left out of it.
struct Pair {
  float sum, rest;
};
__device__ __forceinline__ Pair exact_sum(float s, float x, float c) {
#pragma clang fp contract(off)
  const float p = s * x, p_rest = fmaf(s, x, -p), sum = p + c, back = sum - p;
  return Pair{sum, ((p - (sum - back)) + (c - back)) + p_rest};
}

// U's order: lane group g's value i of a block is token g + 4 i, so that the four tokens of a matrix instruction of the state's update
// are neighbours and the update adds them from the first to the last, as the scan does; W', V' and the keys are packed for that.
// A (slot, head)'s floats: W' and Q' [L / 16][DP / 16] blocks of left operands, D_Ls k_s by rows of S [DP / 16][L / 16] blocks of left
// operands, V' and O' [column blocks][L / 16] blocks of sums, and one line for c_L.
__host__ __device__ inline int64_t pack_floats(int dp, int blocks) { return (int64_t)3 * L * dp + (int64_t)2 * L * 16 * blocks + 64; }

// Four waves.  The products of keys with keys and queries (wave w takes row block w of the one and 3 - w of the other: ten blocks each
// in all, five a wave), the inverses of A's diagonal blocks (a wave one, a lane a column), and then every wave solves for columns of
// its own, block row by block row, each block of the solution at once an operand of the next.  480 matrix instructions a wave for
// heads of 128 x 128, 32 of them in 64 bits and twice as long, 7 us (139 TFLOP/s is what the float32 ones reach): 31 us for 1,024 heads of
// chunks if nothing else took time, 84 as it is inside a prompt, two workgroups a compute unit filling each other's waits.  11 of them are
// the stores of W' and Q' in pieces of 16 bytes; loads behind branches, one waited for after the other, had made it 40 more.
// WHOLE: every piece of four values is 16 bytes aligned.
template <int DP, bool WHOLE>
__global__ __launch_bounds__(256, 2) void delta_pack_kernel(const float* __restrict__ qkv, const float* __restrict__ gates,
                                                            const int* __restrict__ cu, int requests, int G, int H, int d, int dv,
                                                            float* __restrict__ packs) {
  constexpr int KB = DP / 16, LD = DP + 4, TLD = L + 4;        // rows four banks apart: 16-byte reads of 16 rows meet no conflict
  __shared__ __attribute__((aligned(16))) float ks[L * LD];
  __shared__ __attribute__((aligned(16))) float low[L * TLD];  // D, then -A off the diagonal blocks and the inverses less 1 in them
  __shared__ __attribute__((aligned(16))) float seen[L * TLD]; // D, then P
  __shared__ __attribute__((aligned(16))) float beta_of[L], decay_of[L], tail_of[L];
  const int slot = blockIdx.x, h = blockIdx.y, tid = threadIdx.x, lane = tid % WAVE, wave = __builtin_amdgcn_readfirstlane(tid / WAVE), col = lane & 15, g = lane >> 4;
  // the request whose chunk this slot is: the last one that begins at or before it
  int r = -1;
  for (int r0 = 0; r0 < requests; r0 += WAVE) {
    const bool before = r0 + lane < requests && first_slot(cu, r0 + lane) <= slot;
    r += __popcll(__ballot(before));
  }
  if (r < 0) return;
  const int chunk = slot - first_slot(cu, r), n = cu[r + 1] - cu[r];
  if (chunk * L >= n) return;
  const int token0 = cu[r] + chunk * L, count = min(L, n - chunk * L);
  const int channels = 2 * G * d + H * dv, hk = h / (H / G), blocks = (dv + 15) / 16;
  const float* q_rows = qkv + (int64_t)token0 * channels + hk * d;
  const float* k_rows = q_rows + G * d;
  const float* v_rows = qkv + (int64_t)token0 * channels + 2 * G * d + (int64_t)h * dv;
  // four values of a row from dim i on; zeros past the portion's end and the head's last dim.  (No branch around a load, here and below:
  // behind one, each load would be waited for by itself.  Past the end an address inside is read and the value not used.)
  auto piece = [&](const float* rows, int t, int i) {
    const float* from = rows + (int64_t)min(t, count - 1) * channels;
    floatx4 v;
    if constexpr (WHOLE) {
      v = *(const floatx4*)(from + min(i, d - 4));
    } else {
#pragma unroll
      for (int x = 0; x < 4; ++x) v[x] = from[min(i + x, d - 1)];
    }
#pragma unroll
    for (int x = 0; x < 4; ++x)
      if (t >= count || i + x >= d) v[x] = 0.f;
    return v;
  };
  float* own = packs + ((int64_t)slot * H + h) * pack_floats(DP, blocks);
  float* w_pack = own;
  float* q_pack = w_pack + L * DP;
  float* k_pack = q_pack + L * DP;
  float* v_pack = k_pack + L * DP;
  float* o_pack = v_pack + L * 16 * blocks;
  float* end_pack = o_pack + L * 16 * blocks;

  constexpr int KP = L * DP / 4 / 256, ROW_PIECES = DP / 4;
  floatx4 kp[KP], qa[KB];
  const int bq = 3 - wave;
  const float* gate = gates + (int64_t)(token0 + min(lane, count - 1)) * 2 * H + h;
  const float beta = lane < count ? gate[0] : 0.f, decay = lane < count ? gate[H] : 1.f;
#pragma unroll
  for (int p = 0; p < KP; ++p) kp[p] = piece(k_rows, (tid + p * 256) / ROW_PIECES, (tid + p * 256) % ROW_PIECES * 4);
#pragma unroll
  for (int j = 0; j < KB; ++j) qa[j] = piece(q_rows, bq * 16 + col, 16 * j + 4 * g);
  if (wave == 0) {
    float behind = 0.f, all = 1.f, mine = 0.f;
#pragma unroll 8
    for (int t = 0; t < L; ++t) {
      const float here = __int_as_float(__builtin_amdgcn_readlane(__float_as_int(decay), t));
      behind = lane < t ? behind * here : lane == t ? 1.f : 0.f;
      all *= here;
      if (lane == t) mine = all;
      low[t * TLD + lane] = behind;
      seen[t * TLD + lane] = behind;
    }
    beta_of[lane] = beta;
    decay_of[lane] = mine;
    tail_of[lane] = behind;
    if (lane == 0) end_pack[0] = all;
  }
#pragma unroll
  for (int p = 0; p < KP; ++p) *(floatx4*)(ks + (tid + p * 256) / ROW_PIECES * LD + (tid + p * 256) % ROW_PIECES * 4) = kp[p];
  __syncthreads();

  {
    floatx4 ka[KB];
#pragma unroll
    for (int j = 0; j < KB; ++j) ka[j] = *(const floatx4*)(ks + (wave * 16 + col) * LD + 16 * j + 4 * g);
    // the sums of one row block's rows with the keys of block b
    auto with_keys = [&](const floatx4 (&rows)[KB], int b) {
      floatx4 part[KB] = {}, keys[KB];
#pragma unroll
      for (int j = 0; j < KB; ++j) keys[j] = *(const floatx4*)(ks + (b * 16 + col) * LD + 16 * j + 4 * g);
#pragma unroll
      for (int i = 0; i < 4; ++i)
#pragma unroll
        for (int j = 0; j < KB; ++j) part[j] = mfma(rows[j][i], keys[j][i], part[j]);
#pragma unroll
      for (int apart = 1; apart < KB; apart *= 2)
#pragma unroll
        for (int j = 0; j < KB; j += 2 * apart) part[j] += part[j + apart];
      return part[0];
    };
    for (int b = 0; b <= wave; ++b) {
      const floatx4 sums = with_keys(ka, b), beta4 = *(const floatx4*)(beta_of + wave * 16 + 4 * g);
      const int s = b * 16 + col;
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        const int t = wave * 16 + 4 * g + i;
        const float a = beta4[i] * low[t * TLD + s] * sums[i];
        low[t * TLD + s] = b < wave ? -a : s < t ? a : 0.f;
      }
    }
    for (int b = 0; b < bq; ++b) {
      const floatx4 sums = with_keys(qa, b);
#pragma unroll
      for (int i = 0; i < 4; ++i) seen[(bq * 16 + 4 * g + i) * TLD + b * 16 + col] *= sums[i];
    }
    // The last block in 64 bits: a query's product with a key is where the terms cancel most, and the nearest tokens' are what
    // read-outs are mostly made of.  (Sums come out with lane 16 g + r holding column r of the rows g, g + 4, g + 8 and g + 12.)
    doublex4 sums[2] = {};
#pragma unroll
    for (int j = 0; j < KB; ++j) {
      const floatx4 keys = *(const floatx4*)(ks + (bq * 16 + col) * LD + 16 * j + 4 * g);
#pragma unroll
      for (int i = 0; i < 4; ++i) sums[i % 2] = __builtin_amdgcn_mfma_f64_16x16x4f64((double)qa[j][i], (double)keys[i], sums[i % 2], 0, 0, 0);
    }
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      const int row = g + 4 * i;
      float* at = seen + (bq * 16 + row) * TLD + bq * 16 + col;
      *at = col <= row ? (float)((double)*at * (sums[0][i] + sums[1][i])) : 0.f;
    }
  }
  __syncthreads();
  {
    // column `col` of the inverse of 1 + A's block (wave, wave) by substitution from the top; what is kept is the inverse less 1
    const float* a = low + (wave * 16) * TLD + wave * 16;
    float x[16];
#pragma unroll
    for (int t = 0; t < 16; ++t) {
      x[t] = t == col ? 1.f : 0.f;
      floatx4 row[4];
#pragma unroll
      for (int s4 = 0; s4 < 4; ++s4) row[s4] = *(const floatx4*)(a + t * TLD + 4 * s4);
#pragma unroll
      for (int s = 0; s < t; ++s) x[t] = fmaf(-row[s / 4][s % 4], x[s], x[t]);
    }
    __syncthreads();
#pragma unroll
    for (int t = 0; t < 16; ++t)
      if (t / 4 == g) low[(wave * 16 + t) * TLD + wave * 16 + col] = t == col ? 0.f : x[t];
  }
  __syncthreads();

  // the blocks of both triangles, held for all columns: block (b, c) at b (b + 1) / 2 + c
  floatx4 la[10], pa[10];
#pragma unroll
  for (int b = 0; b < 4; ++b)
#pragma unroll
    for (int c = 0; c <= b; ++c) {
      la[b * (b + 1) / 2 + c] = *(const floatx4*)(low + (b * 16 + col) * TLD + c * 16 + 4 * g);
      pa[b * (b + 1) / 2 + c] = *(const floatx4*)(seen + (b * 16 + col) * TLD + c * 16 + 4 * g);
    }
  // A diagonal block of either triangle times a block of x, added to c.  A product multiplies the zeros above the diagonal with the
  // rows of later tokens as well, which makes NaN of an infinity or NaN there: a column of x with one in it is then worked out value by
  // value, below the diagonal only, so that it reaches no token before its own, as in the scan.
  auto on_diagonal = [&](const float* triangle, int b, const floatx4& block, const floatx4& rows, floatx4 c) {
    const float probe = fmaf(rows[0], 0.f, fmaf(rows[1], 0.f, fmaf(rows[2], 0.f, rows[3] * 0.f)));      // 0, or NaN
    if (__builtin_amdgcn_ballot_w64(probe != 0.f) == 0) return product(block, rows, c);
    const float* a = triangle + (b * 16 + 4 * g) * TLD + b * 16;
#pragma unroll 1
    for (int from = 0; from < 4; ++from)
#pragma unroll
      for (int j = 0; j < 4; ++j) {
        const float row = __shfl(rows[j], from * 16 + col, WAVE);
#pragma unroll
        for (int i = 0; i < 4; ++i)
          if (4 * from + j <= 4 * g + i) c[i] = fmaf(a[i * TLD + 4 * from + j], row, c[i]);
      }
    return c;
  };
  // a tile's queries (W' and Q') or values (V' and O'), asked for a tile ahead
  floatx4 next[4];
  auto fetch = [&](int tile) {
    const bool is_w = tile < KB;
    const float* from = is_w ? q_rows + min(tile * 16 + col, d - 1) : v_rows + min((tile - KB) * 16 + col, dv - 1);
#pragma unroll
    for (int b = 0; b < 4; ++b)
#pragma unroll
      for (int i = 0; i < 4; ++i) next[b][i] = from[(int64_t)min(b * 16 + 4 * g + i, count - 1) * channels];
  };
  fetch(wave);
  for (int tile = wave; tile < KB + blocks; tile += 4) {
    const bool is_w = tile < KB;
    const int column = (is_w ? tile : tile - KB) * 16 + col, width = is_w ? d : dv;
    floatx4 x[4], y[4];
#pragma unroll
    for (int b = 0; b < 4; ++b) {
      const int t0 = b * 16 + 4 * g;
      const floatx4 kept = *(const floatx4*)(decay_of + t0);
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        const float value = t0 + i < count && column < width ? next[b][i] : 0.f;
        x[b][i] = is_w ? kept[i] * ks[(t0 + i) * LD + min(column, DP - 1)] : value;       // (times the step sizes below)
        y[b][i] = is_w ? kept[i] * value : 0.f;
      }
    }
    fetch(min(tile + 4, KB + blocks - 1));
    __builtin_amdgcn_sched_barrier(0);
#pragma unroll
    for (int b = 0; b < 4; ++b) {
      Sums above, read;
#pragma unroll
      for (int c = 0; c < b; ++c) above.add(c, la[b * (b + 1) / 2 + c], x[c]);
      // The right side less what the blocks above take of it, rounded and what the rounding left out, which joins the smaller part of
      // the product with the inverse: a token's u is rounded twice, as in the scan.
      const floatx4 steps = *(const floatx4*)(beta_of + b * 16 + 4 * g), taken = above.total();
      floatx4 rest;
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        const Pair right = exact_sum(is_w ? -steps[i] : steps[i], x[b][i], taken[i]);
        x[b][i] = right.sum, rest[i] = right.rest;
      }
      x[b] += on_diagonal(low, b, la[b * (b + 1) / 2 + b], x[b], rest);
#pragma unroll
      for (int c = 0; c < b; ++c) read.add(c, pa[b * (b + 1) / 2 + c], x[c]);
      read.part[b] = on_diagonal(seen, b, pa[b * (b + 1) / 2 + b], x[b], read.part[b]);
      y[b] += read.total();
    }
#pragma unroll
    for (int b = 0; b < 4; ++b) {
      if (is_w) {
        // as left operands: row 4 g + i (of W' row 4 i + g: see U's order), and column col of the block is lane group col / 4's value col % 4
#pragma unroll
        for (int i = 0; i < 4; ++i) {
          const int at = (b * KB + tile) * BLOCK + col / 4 * 64 + col % 4;
          w_pack[at + (4 * i + g) * 4] = x[b][i];
          q_pack[at + (4 * g + i) * 4] = y[b][i];
        }
      } else {
        const int at = ((tile - KB) * 4 + b) * BLOCK + lane * 4;
        *(floatx4*)(v_pack + at) = groups_for_values(x[b]);
        *(floatx4*)(o_pack + at) = y[b];
      }
    }
  }
  for (int b = wave; b < KB; b += 4)
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      floatx4 v;
#pragma unroll
      for (int i = 0; i < 4; ++i) v[i] = ks[(16 * j + g + 4 * i) * LD + 16 * b + col] * tail_of[16 * j + g + 4 * i];
      *(floatx4*)(k_pack + (b * 4 + j) * BLOCK + lane * 4) = v;
    }
}

// Four waves: wave w makes U and O of the chunk's tokens 16 w .. 16 w + 15 and updates the rows of S of its DP / 64 blocks.  U and the
// new S go through LDS, a barrier each; half of O's products stand before either barrier, with the old S still in registers.  A
// chunk's operands (a wave's rows of the packs, 1,024 bytes a load) are asked for a chunk ahead, into a second set of registers: with
// one wave a SIMD there are enough.  96 matrix instructions a wave and chunk, 3,072 cycles: 47 us for
// 32 chunks, 95 by itself and 105 inside a prompt: 71 without the loads (96 KB a chunk and compute unit, 44 bytes a nanosecond; fetches into LDS that the L2s
// answer bring a unit 86-100 in gemm_tiles.hip, which has not been tried here), the rest the two barriers with a trip through LDS each.  Left to itself the compiler moves the loads to where
// their registers are cheapest: 106 us.
template <int DP>
__global__ __launch_bounds__(256, 1) void delta_walk_kernel(const float* __restrict__ packs, const int* __restrict__ cu,
                                                            const int* __restrict__ slot_ids, float* __restrict__ state,
                                                            int64_t state_stride, int H, int dv, float* __restrict__ raw) {
  constexpr int KB = DP / 16, SB = KB / 4, ROWS = DP / SPLIT;
  __shared__ floatx4 s_room[KB * WAVE], u_room[4 * WAVE];
  const int r = blockIdx.x, h = blockIdx.y, z = blockIdx.z, c0 = z * 16, tid = threadIdx.x, lane = tid % WAVE, wave = __builtin_amdgcn_readfirstlane(tid / WAVE);
  const int col = lane & 15, g = lane >> 4, blocks = (dv + 15) / 16;
  const int start = cu[r], n = cu[r + 1] - start, chunks = (n + L - 1) / L;
  if (n <= 0) return;
  const int64_t stride = pack_floats(DP, blocks), step = (int64_t)H * stride;
  const float* own = packs + (int64_t)first_slot(cu, r) * step + (int64_t)h * stride;
  float* st = state + (int64_t)slot_ids[r] * state_stride + (int64_t)h * ROWS * dv * SPLIT;

  // row k of S lies in block k / 16 with lane group k % 16 / 4; the state row runs over columns and 16ths of the rows
  auto place = [&](int row, int s, int cc) {
    const int k = s * ROWS + row;
    return (k / 16 * WAVE + k % 16 / 4 * 16 + cc) * 4 + k % 4;
  };
  for (int e = tid; e < ROWS * 16 * SPLIT; e += 256) {
    const int row = e / (16 * SPLIT), cc = e / SPLIT % 16, s = e % SPLIT;
    ((float*)s_room)[place(row, s, cc)] = c0 + cc < dv ? st[((int64_t)row * dv + c0 + cc) * SPLIT + s] : 0.f;
  }
  __syncthreads();
  floatx4 S[SB], old[KB];
#pragma unroll
  for (int b = 0; b < SB; ++b) S[b] = s_room[(wave * SB + b) * WAVE + lane];
#pragma unroll
  for (int j = 0; j < KB; ++j) old[j] = s_room[j * WAVE + lane];

  struct Operands {
    floatx4 w[KB], q[KB], k[SB][4], v, o;
    float end;
  };
  auto fetch = [&](Operands& x, int chunk) {
    const float* from = own + min(chunk, chunks - 1) * step;
    const float* q_from = from + L * DP;
    const float* k_from = q_from + L * DP;
    const float* v_from = k_from + L * DP;
    const float* o_from = v_from + L * 16 * blocks;
    x.v = *(const floatx4*)(v_from + (z * 4 + wave) * BLOCK + lane * 4);
#pragma unroll
    for (int j = 0; j < KB; ++j) x.w[j] = *(const floatx4*)(from + (wave * KB + j) * BLOCK + lane * 4);
    x.o = *(const floatx4*)(o_from + (z * 4 + wave) * BLOCK + lane * 4);
#pragma unroll
    for (int j = 0; j < KB; ++j) x.q[j] = *(const floatx4*)(q_from + (wave * KB + j) * BLOCK + lane * 4);
#pragma unroll
    for (int b = 0; b < SB; ++b)
#pragma unroll
      for (int j = 0; j < 4; ++j) x.k[b][j] = *(const floatx4*)(k_from + ((wave * SB + b) * 4 + j) * BLOCK + lane * 4);
    x.end = o_from[L * 16 * blocks];
  };
  auto turn = [&](const Operands& x, int chunk) {
    Sums u, o, s[SB];
    // a quarter of O's products at a time, where the others would wait for LDS or for each other
    auto read_out = [&](int quarter) {
      __builtin_amdgcn_sched_barrier(0);
      if constexpr (KB >= 8) {
#pragma unroll
        for (int j = 0; j < KB / 4; j += 2) o.add_two(quarter * (KB / 4) + j, x.q, old);
      } else {
        o.add(quarter, x.q[quarter], old[quarter]);
      }
      __builtin_amdgcn_sched_barrier(0);
    };
#pragma unroll
    for (int j = 0; j < KB; j += 2) u.add_two(j, x.w, old);
    u_room[wave * WAVE + lane] = x.v + u.total();
    read_out(0);
    __syncthreads();
    floatx4 all[4];
#pragma unroll
    for (int j = 0; j < 4; ++j) all[j] = u_room[j * WAVE + lane];
    read_out(1);
    // the state and the first three blocks of tokens, each summed by itself, and the last block's chain, mostly the largest, on top
#pragma unroll
    for (int b = 0; b < SB; ++b) s[b].add_two(0, x.k[b], all);
#pragma unroll
    for (int b = 0; b < SB; ++b) s[b].add(2, x.k[b][2], all[2]);
#pragma unroll
    for (int b = 0; b < SB; ++b) S[b] = x.end * S[b] + ((s[b].part[0] + s[b].part[1]) + s[b].part[2]);
#pragma unroll
    for (int i = 0; i < 4; ++i)
#pragma unroll
      for (int b = 0; b < SB; ++b) S[b] = mfma(x.k[b][3][i], all[3][i], S[b]);
#pragma unroll
    for (int b = 0; b < SB; ++b) s_room[(wave * SB + b) * WAVE + lane] = S[b];
    read_out(2);
    __syncthreads();
    floatx4 now[KB];
#pragma unroll
    for (int j = 0; j < KB; ++j) now[j] = s_room[j * WAVE + lane];
    read_out(3);
#pragma unroll
    for (int j = 0; j < KB; ++j) old[j] = now[j];
    const int t0 = chunk * L + wave * 16 + 4 * g;
    const floatx4 read = x.o + o.total();
    float* row = raw + ((int64_t)(start + t0) * H + h) * dv + c0 + col;
#pragma unroll
    for (int i = 0; i < 4; ++i)
      if (t0 + i < n && c0 + col < dv) row[(int64_t)i * H * dv] = read[i];
  };
  Operands a, b;
  fetch(a, 0);
  for (int chunk = 0; chunk < chunks; chunk += 2) {
    fetch(b, chunk + 1);
    __builtin_amdgcn_sched_barrier(0);      // (the loads here, not where their registers would be cheapest)
    turn(a, chunk);
    if (chunk + 1 >= chunks) break;
    fetch(a, chunk + 2);
    __builtin_amdgcn_sched_barrier(0);
    turn(b, chunk + 1);
  }
  for (int e = tid; e < ROWS * 16 * SPLIT; e += 256) {
    const int row = e / (16 * SPLIT), cc = e / SPLIT % 16, s = e % SPLIT;
    if (c0 + cc < dv) st[((int64_t)row * dv + c0 + cc) * SPLIT + s] = ((const float*)s_room)[place(row, s, cc)];
  }
}

}  // namespace

// Floats of the packs that a step of so many tokens needs, `requests` of whose requests take the form in chunks.
LRS_API int64_t lrs_delta_pack_floats(int tokens, int requests, int H, int d, int dv) {
  return (int64_t)(tokens / L + requests + 1) * H * pack_floats(SPLIT * lrs_delta_state_rows(d), (dv + 15) / 16);
}

// The recurrence of the requests that cu and slot_ids name, from the prepared rows of qkv and gates to raw (delta.hip); d at most 128.
void lrs_delta_chunk_walk(const float* qkv, const float* gates, const int* cu, const int* slot_ids, int tokens, int requests, float* state,
                          int64_t state_stride, int G, int H, int d, int dv, float* raw, float* packs, hipStream_t s) {
  const dim3 pgrid(tokens / L + requests + 1, H), grid(requests, H, (dv + 15) / 16);
  const bool whole = d % 4 == 0 && H * dv % 4 == 0;
#define RUN(DP)                                                                                                  \
  do {                                                                                                           \
    if (whole) delta_pack_kernel<DP, true><<<pgrid, 256, 0, s>>>(qkv, gates, cu, requests, G, H, d, dv, packs);  \
    else delta_pack_kernel<DP, false><<<pgrid, 256, 0, s>>>(qkv, gates, cu, requests, G, H, d, dv, packs);       \
    delta_walk_kernel<DP><<<grid, 256, 0, s>>>(packs, cu, slot_ids, state, state_stride, H, dv, raw);            \
  } while (0)
  if (d <= 64) RUN(64);
  else RUN(128);
#undef RUN
}
