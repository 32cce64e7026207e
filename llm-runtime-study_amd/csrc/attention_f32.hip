// Float32 attention over the paged cache on the matrix cores (the rules of attention.hip: what a token sees, the pages'
// layout, rounding that depends on positions alone).
//
// The keys of a sequence are cut into pieces of 64 positions counted from position 0.  A wave takes a piece for up to 16
// queries (tokens times the kv group's heads, the columns of its products): scores, their maximum, weights and weighted sum of
// that piece alone, as if there were no other.  A query's result is its pieces' partial results merged one after the
// other in the order of their positions, by the same operations however many queries
// share a workgroup's waves (eight, or fewer over short contexts), which take a piece each at a time.
//
// A piece is 256 products of 32 cycles at 128 dims whatever columns are in use, 6.8 us for the two waves of a SIMD: that bounds a
// prompt (2,048 tokens, 16 heads of 128: 305 us, 56 TFLOP/s; 3,174 us with a workgroup a (token, head) and plain FMAs) and,
// with one trip to memory before it, a decode step (8 tokens at 509: 16.6 us, 18.5 before; 509 tokens of a prompt 33, 39 before).  A block of 16 keys, and one of
// values, is asked for while the one before is multiplied.  Memory writes it into the wave's part of LDS, 64 bytes of a row by
// four neighbouring lanes: loaded as the products' operands lie, a lane a row, a block costs the compute unit's L1 four times as many
// looks at its tags, and a decode step's 512 KB for a compute unit took 15 us to come.
#include "common.h"

#include <type_traits>

LRS_API int lrs_compute_units();

int lrs_attention_f32(float* out, int out_stride, const float* q, int q_stride, const float* k_pages, const float* v_pages, const int* block_table,
                      int table_stride, const int* token_request, const int* positions, int tokens, int nq, int nkv, int d, int page_size,
                      float scale, int window, int together, int longest, hipStream_t s);
bool lrs_attention_f32_takes(const void* out, int out_stride, const void* q, int q_stride, const void* k_pages, const void* v_pages, int nq, int nkv,
                             int d, int dv, int page_size);

namespace {

typedef float floatx2 __attribute__((ext_vector_type(2)));
constexpr int PIECE = 64, COLUMNS = 16, FEW = 4;

// What is left of a partial result when its reference point moves to `top`.
__device__ __forceinline__ float moved(float from, float top) { return from == -INFINITY ? 0.f : expf(from - top); }

// 16 keys' weighted values where some values are not finite (perhaps in slots that nothing was written to): such a value counts
// only where its weight is not zero, which a product of tiles cannot tell.  It is left out of the products, and three more
// products say which sums see an infinity or a NaN.
__device__ __forceinline__ void add_odd_values(floatx4 values, floatx4 weights, floatx4& acc) {
  floatx4 plus = {0.f, 0.f, 0.f, 0.f}, minus = plus, none = plus;
#pragma unroll
  for (int t = 0; t < 4; ++t) {
    const float v = values[t], seen = weights[t] != 0.f ? 1.f : 0.f;
    acc = __builtin_amdgcn_mfma_f32_16x16x4f32(isfinite(v) ? v : 0.f, weights[t], acc, 0, 0, 0);
    plus = __builtin_amdgcn_mfma_f32_16x16x4f32(v == INFINITY ? 1.f : 0.f, seen, plus, 0, 0, 0);
    minus = __builtin_amdgcn_mfma_f32_16x16x4f32(v == -INFINITY ? 1.f : 0.f, seen, minus, 0, 0, 0);
    none = __builtin_amdgcn_mfma_f32_16x16x4f32(v != v ? 1.f : 0.f, seen, none, 0, 0, 0);
  }
#pragma unroll
  for (int e = 0; e < 4; ++e) {
    if (plus[e] > 0.f) acc[e] += INFINITY;
    if (minus[e] > 0.f) acc[e] -= INFINITY;
    if (none[e] > 0.f) acc[e] = NAN;
  }
  __builtin_amdgcn_sched_barrier(0);
}

// SHORT: blocks of 16 keys that nobody sees are left out rather than multiplied with weights of zero.
// DIRECT: keys and values into registers as the products' operands lie, not into LDS first: a trip shorter, which a wave of one piece waits
// for (lrs_attention_f32 says when).
// One workgroup: `together` tokens (as many as fit 16 columns with the kv group's heads) of one kv head, taken request by
// request should they not all belong to one.
template <int D, int WAVES, bool SHORT, bool DIRECT>
__global__ __launch_bounds__(WAVES * WAVE, WAVES == 8 ? 1 : 2) void attention_f32_mfma_kernel(
    const int* __restrict__ positions, const int* __restrict__ token_request, const int* __restrict__ block_table, const float* __restrict__ q,
    int table_stride, int q_stride, int tokens, int together, int heads, int groups, const float* __restrict__ k_pages,
    const float* __restrict__ v_pages, float* __restrict__ out, int out_stride, int nkv, int page_size, float scale, int window) {
  // (what leads to the first keys comes first: those arguments are in registers when a wave begins, the file is compiled so)
  constexpr int PITCH = D + 4, TILES = D / 16;   // floats from column to column of a partial result; its tiles of 16 dims
  constexpr int BLOCK = 16 * D, ROOM = !DIRECT && 2 * BLOCK > COLUMNS * PITCH ? 2 * BLOCK : COLUMNS * PITCH;   // floats: 16 keys or their values; a wave's two, or its partial result
  __shared__ __attribute__((aligned(128))) float parts[WAVES * ROOM];
  __shared__ float maxima[WAVES * COLUMNS * 2];                            // maxima and sums
  const int columns = together * heads;
  const int tid = threadIdx.x, lane = tid % WAVE, wave = __builtin_amdgcn_readfirstlane(tid / WAVE);
  const int r = lane & 15, g = lane >> 4;
  const int kv_head = blockIdx.y;
  // the last tokens of a prompt, which see most, begin first
  const int begin = (groups - 1 - (int)blockIdx.x) * together, end = begin + together < tokens ? begin + together : tokens;
  // A fetch brings 16 bytes of each of 16 rows four times over (rows of 16 dims of a key, or of 16 keys of a value's dim): lane l the
  // piece at place l, row l / 4; a row's pieces are turned round so that 16-byte reads of the operands meet every bank once.
  const int place_row = lane / 4, place_piece = lane % 4 ^ (place_row >> 2 & 1) << 1;
  const unsigned key_lane = (unsigned)(place_row * D + 4 * place_piece) * 4u, value_lane = (unsigned)(place_row * page_size + 4 * place_piece) * 4u;   // bytes
  float* const blocks = parts + wave * ROOM;
  const unsigned blocks_address = (unsigned)(uintptr_t)(__attribute__((address_space(3))) float*)parts + (unsigned)(wave * ROOM * 4);
  const float* const operand = blocks + r * 16 + (g ^ (r >> 2 & 1) << 1) * 4;
  const int my_token = begin + r / heads;                                  // of this lane's column
  // the thread that merges: column and four dims
  const int item = tid, item_column = item / (D / 4), item_dim = item % (D / 4) * 4;
  for (int first = begin; first < end;) {
    const int request = token_request[first];
    int last = first + 1, highest = positions[first], lowest = first_seen(highest, window);
    for (; last < end && token_request[last] == request; ++last) {
      const int pos = positions[last], from = first_seen(pos, window);
      highest = pos > highest ? pos : highest, lowest = from < lowest ? from : lowest;
    }
    const bool mine = r < columns && my_token >= first && my_token < last;
    const int token = mine ? my_token : first, head = kv_head * heads + (mine ? r % heads : 0);
    const int pos = mine ? positions[token] : -1, from = mine ? first_seen(pos, window) : 0;
    const int* table = block_table + (int64_t)request * table_stride;
    // the query, as the products' second operand: product 4 j + t multiplies dims 16 j + 4 g + t
    floatx4 qf[TILES];
#pragma unroll
    for (int j = 0; j < TILES; ++j) qf[j] = *(const floatx4*)(q + (int64_t)token * q_stride + head * D + 16 * j + 4 * g);
    float run_max = -INFINITY, run_sum = 0.f;
    floatx4 run = {0.f, 0.f, 0.f, 0.f};
    const int last_piece = highest / PIECE;
    for (int piece0 = lowest / PIECE; piece0 <= last_piece; piece0 += WAVES) {
      const int piece = piece0 + wave;
      if (piece <= last_piece) {
        floatx4 score[4];
        int64_t page[4];                                                   // the (page, kv head) block of 16 keys, and the slot they begin at
        int slot[4];
        bool seen[4];
#pragma unroll
        for (int b = 0; b < 4; ++b) {
          // a block that nobody sees (perhaps without a page) stands for the nearest that somebody does: its weights will be zero
          int key0 = piece * PIECE + b * 16;
          seen[b] = !SHORT || (key0 <= highest && key0 + 15 >= lowest);
          key0 = key0 < (lowest & ~15) ? lowest & ~15 : key0 > (highest & ~15) ? highest & ~15 : key0;
          page[b] = (int64_t)table[key0 / page_size] * nkv + kv_head;
          slot[b] = key0 % page_size;
        }
        // 16 keys, or their values, are asked for a block ahead, into LDS once the wave has what it read from their place
        floatx4 held[DIRECT ? 2 : 1][TILES];
        auto have_read = [] { asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory"); };
        auto load_keys = [&](int b) {
          const float* keys = k_pages + (page[b] * page_size + slot[b]) * D;
          if constexpr (DIRECT) {
#pragma unroll
            for (int j = 0; j < TILES; ++j) held[b & 1][j] = *(const floatx4*)(keys + (unsigned)(r * D + 4 * g) + 16 * j);
          } else {
            have_read();
#pragma unroll
            for (int j = 0; j < TILES; ++j) fetch_to_lds(keys + 16 * j, key_lane, blocks_address + (unsigned)(((b & 1) * BLOCK + j * 256) * 4));
          }
        };
        auto load_values = [&](int b) {
          const float* values = v_pages + page[b] * D * page_size + slot[b];                      // [dim][slot]
          if constexpr (DIRECT) {
#pragma unroll
            for (int i = 0; i < TILES; ++i) held[b & 1][i] = *(const floatx4*)(values + (int64_t)(16 * i) * page_size + (unsigned)(r * page_size + 4 * g));
          } else {
            have_read();
#pragma unroll
            for (int i = 0; i < TILES; ++i) fetch_to_lds(values + 16 * i * page_size, value_lane, blocks_address + (unsigned)(((b & 1) * BLOCK + i * 256) * 4));
          }
        };
        auto take = [&](int b, auto pending) {                             // block b, with so many fetches still on their way
          if constexpr (!DIRECT) {
            asm volatile("s_waitcnt vmcnt(%0)" :: "n"(decltype(pending)::value) : "memory");
#pragma unroll
            for (int j = 0; j < TILES; ++j) held[0][j] = *(const floatx4*)(operand + (b & 1) * BLOCK + j * 256);
          }
        };
        typedef std::integral_constant<int, TILES> NextBlock;
        load_keys(0);
#pragma unroll
        for (int b = 0; b < 4; ++b) {
          if (b < 3) load_keys(b + 1);
          else load_values(0);
          take(b, NextBlock());
          __builtin_amdgcn_sched_barrier(0);
          score[b] = floatx4{0.f, 0.f, 0.f, 0.f};
          if (seen[b])
#pragma unroll
            for (int j = 0; j < TILES; ++j)
#pragma unroll
              for (int t = 0; t < 4; ++t) score[b] = __builtin_amdgcn_mfma_f32_16x16x4f32(held[DIRECT ? b & 1 : 0][j][t], qf[j][t], score[b], 0, 0, 0);
          __builtin_amdgcn_sched_barrier(0);
        }
        // this lane: keys 16 b + 4 g + t of its column
        float top = -INFINITY;
#pragma unroll
        for (int b = 0; b < 4; ++b)
#pragma unroll
          for (int t = 0; t < 4; ++t) {
            const int key = piece * PIECE + b * 16 + 4 * g + t;
            score[b][t] = key <= pos && key >= from ? score[b][t] * scale : -INFINITY;
            top = fmaxf(top, score[b][t]);
          }
        top = fmaxf(top, __shfl_xor(top, 16, WAVE));
        top = fmaxf(top, __shfl_xor(top, 32, WAVE));
        const float ref = top == -INFINITY ? 0.f : top;                    // all that is seen of the piece scores minus infinity: no weight
        float sum = 0.f;
#pragma unroll
        for (int b = 0; b < 4; ++b)
#pragma unroll
          for (int t = 0; t < 4; ++t) {
            const int key = piece * PIECE + b * 16 + 4 * g + t;
            score[b][t] = key <= pos && key >= from ? expf(score[b][t] - ref) : 0.f;
            sum += score[b][t];
            if (t == 3) __builtin_amdgcn_sched_barrier(0);
          }
        sum += __shfl_xor(sum, 16, WAVE);
        sum += __shfl_xor(sum, 32, WAVE);
        floatx4 acc[TILES];
#pragma unroll
        for (int i = 0; i < TILES; ++i) acc[i] = floatx4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
        for (int b = 0; b < 4; ++b) {
          if (b < 3) {
            load_values(b + 1);
            take(b, NextBlock());
          } else {
            take(b, std::integral_constant<int, 0>());
          }
          __builtin_amdgcn_sched_barrier(0);
          if (seen[b]) {
            const floatx4(&vf)[TILES] = held[DIRECT ? b & 1 : 0];
            float finite = 0.f;
#pragma unroll
            for (int i = 0; i < TILES; ++i)
#pragma unroll
              for (int t = 0; t < 4; ++t) finite = fmaf(vf[i][t], 0.f, finite);
            if (__any(finite != 0.f)) {
#pragma unroll
              for (int i = 0; i < TILES; ++i) add_odd_values(vf[i], score[b], acc[i]);
            } else {
#pragma unroll
              for (int t = 0; t < 4; ++t)
#pragma unroll
                for (int i = 0; i < TILES; ++i) acc[i] = __builtin_amdgcn_mfma_f32_16x16x4f32(vf[i][t], score[b][t], acc[i], 0, 0, 0);
            }
          }
          __builtin_amdgcn_sched_barrier(0);
        }
        if (r < columns) {
          float* to = blocks + r * PITCH + 4 * g;
#pragma unroll
          for (int i = 0; i < TILES; ++i) *(floatx4*)(to + 16 * i) = acc[i];
          if (g == 0) maxima[(wave * COLUMNS + r) * 2] = top, maxima[(wave * COLUMNS + r) * 2 + 1] = sum;
        }
      }
      __syncthreads();
      if (item_column < columns) {
        const int here = last_piece - piece0 + 1 < WAVES ? last_piece - piece0 + 1 : WAVES;
        for (int p = 0; p < here; ++p) {
          const float top = maxima[(p * COLUMNS + item_column) * 2], sum = maxima[(p * COLUMNS + item_column) * 2 + 1];
          const floatx4 part = *(const floatx4*)(parts + p * ROOM + item_column * PITCH + item_dim);
          const float now = fmaxf(run_max, top), keep = moved(run_max, now), take = moved(top, now);
          run_sum = fmaf(run_sum, keep, sum * take);
#pragma unroll
          for (int e = 0; e < 4; ++e) run[e] = fmaf(run[e], keep, part[e] * take);
          run_max = now;
        }
      }
      __syncthreads();
    }
    const int item_token = begin + item_column / heads;
    if (item_column < columns && item_token >= first && item_token < last) {
      const float inv = 1.f / run_sum;
      *(floatx4*)(out + (int64_t)item_token * out_stride + (kv_head * heads + item_column % heads) * D + item_dim) = run * inv;
    }
    first = last;
  }
}

// f(0), f(1) .. f(N - 1), each as a constant.
template <typename F, int... X>
__device__ __forceinline__ void each_of(F&& f, std::integer_sequence<int, X...>) { (f(std::integral_constant<int, X>()), ...); }
template <int N, typename F>
__device__ __forceinline__ void each(F&& f) { each_of(f, std::make_integer_sequence<int, N>()); }

// acc += column i of `a`'s block ABID (lanes 4 ABID + i) times every lane's b: element i of a lane is its own sum for column i.
template <int ABID>
__device__ __forceinline__ void add_few(floatx4& acc, float a, float b) {
  acc = __builtin_amdgcn_mfma_f32_4x4x1f32(a, b, acc, 4, ABID, 0);
}
// 16 keys' weighted values where some are not finite (add_odd_values): key 4 g + t is v[g][t], its weight for column i in lane 16 `block` + 4 g + i of w[t].
__device__ __forceinline__ void add_few_odd_values(const floatx4 (&v)[4], floatx4 w, int block, floatx4& acc) {
  for (int i = 0; i < FEW; ++i) {
    bool plus = false, minus = false, none = false;
    float sum = acc[i];
#pragma unroll
    for (int t = 0; t < 4; ++t)
#pragma unroll
      for (int g = 0; g < 4; ++g) {
        const float x = v[g][t], weight = __shfl(w[t], 16 * block + 4 * g + i, WAVE);
        sum = fmaf(isfinite(x) ? x : 0.f, weight, sum);
        plus |= x == INFINITY && weight != 0.f;
        minus |= x == -INFINITY && weight != 0.f;
        none |= x != x && weight != 0.f;
      }
    if (plus) sum += INFINITY;
    if (minus) sum -= INFINITY;
    if (none) sum = NAN;
    acc[i] = sum;
  }
}

// A step in which every request brings one token and at most four heads share a kv head: the pieces of a (token, kv head) go round `divided`
// workgroups of one wave, piece p, counted from the first that the token sees, to place p of `slots` of sums [tokens, heads of all, slots, D] and
// maxima [..., 2], which attention_f32_merge_kernel merges.  The same operations in the same order as above, so the same bits, but on
// 4x4x1 products, whose sixteen blocks are 64 keys (then 64 dims) for four columns, where 16x16x4 multiplies sixteen whatever is in
// use: a quarter of the time.  All of a piece is asked for at once (64 KB of LDS at 128 dims, two workgroups a unit), the next
// one's keys and values as soon as their place is free.
// What bounds it: one (token, kv head) its trips to memory and the merge's launch (8 of 128 dims at 509 tokens 15.3 -> 10.0 us), many and long ones
// two waves' fetches a unit (64 at 4,000 tokens 116 -> 73 us, 3.6 TB/s).  With 16x16x4 products instead 91 us, 16.2 for 13.7 at 509.
template <int D>
__global__ __launch_bounds__(WAVE, 1) void attention_f32_few_kernel(
    const int* __restrict__ positions, const int* __restrict__ token_request, const int* __restrict__ block_table, const float* __restrict__ q, int table_stride,
    int q_stride, int heads, int divided, const float* __restrict__ k_pages, const float* __restrict__ v_pages, float* __restrict__ sums, float* __restrict__ maxima,
    int slots, int nkv, int page_size, float scale, int window) {
  constexpr int TILES = D / 16, BLOCK = 16 * D, PITCH = PIECE + 4, HALVES = D / 64;
  __shared__ __attribute__((aligned(128))) float blocks[8 * BLOCK];        // 16 keys each, then 16 keys' values each
  __shared__ __attribute__((aligned(16))) float share[FEW * PITCH];        // scores, then weights
  __shared__ __attribute__((aligned(16))) float queries[FEW * D];
  const int lane = threadIdx.x, r = lane & 15, g = lane >> 4, column = r & 3;
  const int token = blockIdx.x, kv_head = blockIdx.y;
  const int pos = positions[token], from = first_seen(pos, window), last_piece = pos / PIECE, first_piece = from / PIECE;
  int piece = first_piece + (int)blockIdx.z;
  if (piece > last_piece) return;
  const int* table = block_table + (int64_t)token_request[token] * table_stride;
  // places of a row's pieces of 16 bytes (fetches as above), turned round so that a lane a row meets every bank once
  const int place_row = lane / 4, place_piece = lane % 4 ^ (place_row >> 2 & 3);
  const unsigned key_lane = (unsigned)(place_row * D + 4 * place_piece) * 4u, value_lane = (unsigned)(place_row * page_size + 4 * place_piece) * 4u;   // bytes
  const unsigned blocks_address = (unsigned)(uintptr_t)(__attribute__((address_space(3))) float*)blocks;
  const int turn = r >> 2 & 3;
  auto have_read = [] { asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory"); };
  auto block_of = [&](int at, int b, int64_t& page, int& slot) {           // the (page, kv head) block of 16 keys of piece `at`, and the slot they begin at
    int key0 = at * PIECE + b * 16;                                        // one that is not seen stands for the nearest that is
    key0 = key0 < (from & ~15) ? from & ~15 : key0 > (pos & ~15) ? pos & ~15 : key0;
    page = (int64_t)table[key0 / page_size] * nkv + kv_head;
    slot = key0 % page_size;
  };
  auto load_keys = [&](int at) {                                           // 16 dims of all, then the next
    const float* keys[4];
#pragma unroll
    for (int b = 0; b < 4; ++b) {
      int64_t page;
      int slot;
      block_of(at, b, page, slot);
      keys[b] = k_pages + (page * page_size + slot) * D;
    }
    have_read();
#pragma unroll
    for (int j = 0; j < TILES; ++j)
#pragma unroll
      for (int b = 0; b < 4; ++b) fetch_to_lds(keys[b] + 16 * j, key_lane, blocks_address + (unsigned)((b * BLOCK + j * 256) * 4));
  };
  auto load_values = [&](int at) {
    const float* values[4];                                                // [dim][slot]
#pragma unroll
    for (int b = 0; b < 4; ++b) {
      int64_t page;
      int slot;
      block_of(at, b, page, slot);
      values[b] = v_pages + page * D * page_size + slot;
    }
    have_read();
#pragma unroll
    for (int b = 0; b < 4; ++b)
#pragma unroll
      for (int i = 0; i < TILES; ++i) fetch_to_lds(values[b] + 16 * i * page_size, value_lane, blocks_address + (unsigned)(((4 + b) * BLOCK + i * 256) * 4));
  };
  // The queries, through LDS as well: a wait of the compiler's for a load of its own would wait for all keys behind it.
#pragma unroll
  for (int f = 0; f < FEW * D / 256; ++f) {
    const int at = f * 256 + 4 * lane, head = kv_head * heads + (at / D < heads ? at / D : 0);
    fetch_lanes_to_lds((uint64_t)(uintptr_t)(q + (int64_t)token * q_stride + head * D + at % D), (unsigned)(uintptr_t)(__attribute__((address_space(3))) float*)queries + (unsigned)(f * 1024));
  }
  load_keys(piece);
  load_values(piece);
  asm volatile("s_waitcnt vmcnt(%0)" :: "n"(8 * TILES < 60 ? 8 * TILES : 60) : "memory");
  float qf[TILES];                                                         // dim 16 j + lane / 4 of this lane's column
#pragma unroll
  for (int j = 0; j < TILES; ++j) qf[j] = queries[(lane & 3) * D + 16 * j + lane / 4];
  for (;;) {
    const int next = piece + divided;
    const bool more = next <= last_piece;
    // scores: this lane's key for every column
    floatx4 score_of = {0.f, 0.f, 0.f, 0.f};
    auto score_tile = [&](auto tile) {
      constexpr int j = decltype(tile)::value;
      asm volatile("s_waitcnt vmcnt(%0)" :: "n"(4 * TILES + 4 * (TILES - 1 - j)) : "memory");
      floatx4 key[4];
#pragma unroll
      for (int c = 0; c < 4; ++c) key[c] = *(const floatx4*)(blocks + g * BLOCK + j * 256 + r * 16 + (c ^ turn) * 4);
      each<16>([&](auto x) {                                               // dims 16 j + 4 c + t, t first to last and c within
        constexpr int t = x / 4, c = x % 4;
        add_few<4 * c + t>(score_of, qf[j], key[c][t]);
      });
    };
    each<TILES>(score_tile);
    if (more) load_keys(next);
#pragma unroll
    for (int i = 0; i < FEW; ++i) share[i * PITCH + lane] = score_of[i];
    __builtin_amdgcn_wave_barrier();
    // this lane: keys 16 b + 4 g + t of its column, as above
    floatx4 score[4];
#pragma unroll
    for (int b = 0; b < 4; ++b) score[b] = *(const floatx4*)(share + column * PITCH + 16 * b + 4 * g);
    float top = -INFINITY;
#pragma unroll
    for (int b = 0; b < 4; ++b)
#pragma unroll
      for (int t = 0; t < 4; ++t) {
        const int key = piece * PIECE + b * 16 + 4 * g + t;
        score[b][t] = key <= pos && key >= from ? score[b][t] * scale : -INFINITY;
        top = fmaxf(top, score[b][t]);
      }
    top = fmaxf(top, __shfl_xor(top, 16, WAVE));
    top = fmaxf(top, __shfl_xor(top, 32, WAVE));
    const float ref = top == -INFINITY ? 0.f : top;
    float sum = 0.f;
#pragma unroll
    for (int b = 0; b < 4; ++b)
#pragma unroll
      for (int t = 0; t < 4; ++t) {
        const int key = piece * PIECE + b * 16 + 4 * g + t;
        score[b][t] = key <= pos && key >= from ? expf(score[b][t] - ref) : 0.f;
        sum += score[b][t];
      }
    sum += __shfl_xor(sum, 16, WAVE);
    sum += __shfl_xor(sum, 32, WAVE);
    __builtin_amdgcn_wave_barrier();
    if (r < FEW)
#pragma unroll
      for (int b = 0; b < 4; ++b) *(floatx4*)(share + r * PITCH + 16 * b + 4 * g) = score[b];
    __builtin_amdgcn_wave_barrier();
    const floatx4 weights = *(const floatx4*)(share + (lane & 3) * PITCH + lane / 4 * 4);   // key 4 (lane / 4) + t of column lane % 4
    floatx4 acc[HALVES];
#pragma unroll
    for (int h = 0; h < HALVES; ++h) acc[h] = floatx4{0.f, 0.f, 0.f, 0.f};
    auto add_block = [&](auto block) {
      constexpr int b = decltype(block)::value;
      if (more) asm volatile("s_waitcnt vmcnt(%0)" :: "n"((3 - b) * TILES + 4 * TILES) : "memory");
      else asm volatile("s_waitcnt vmcnt(%0)" :: "n"((3 - b) * TILES) : "memory");
      const int key0 = piece * PIECE + b * 16;
      if (key0 > pos || key0 + 15 < from) return;
      floatx4 value[HALVES][4];
      float finite = 0.f;
#pragma unroll
      for (int h = 0; h < HALVES; ++h)
#pragma unroll
        for (int c = 0; c < 4; ++c) {
          value[h][c] = *(const floatx4*)(blocks + (4 + b) * BLOCK + (4 * h + g) * 256 + r * 16 + (c ^ turn) * 4);
#pragma unroll
          for (int t = 0; t < 4; ++t) finite = fmaf(value[h][c][t], 0.f, finite);
        }
      if (__any(finite != 0.f)) {
#pragma unroll
        for (int h = 0; h < HALVES; ++h) add_few_odd_values(value[h], weights, b, acc[h]);
      } else {
        each<16>([&](auto x) {                                             // keys 16 b + 4 c + t, t first to last and c within
          constexpr int t = x / 4, c = x % 4;
#pragma unroll
          for (int h = 0; h < HALVES; ++h) add_few<4 * b + c>(acc[h], weights[t], value[h][c][t]);
        });
      }
    };
    each<4>(add_block);
    const int place = piece - first_piece;
    if (place < slots) {
      const int64_t row = (int64_t)(token * nkv + kv_head) * heads;
#pragma unroll
      for (int h = 0; h < HALVES; ++h)
#pragma unroll
        for (int i = 0; i < FEW; ++i)
          if (i < heads) sums[((row + i) * slots + place) * D + 64 * h + lane] = acc[h][i];
      if (lane < heads) *(floatx2*)(maxima + ((row + lane) * slots + place) * 2) = floatx2{top, sum};
    }
    if (!more) return;
    load_values(next);
    piece = next;
  }
}

// A thread four dims of a (token, head): its pieces merged as above.  The first eight are asked for before the token's position is known (the
// buffer has `slots` of each).
constexpr int MERGE_AHEAD = 8;
template <int D>
__global__ __launch_bounds__(WAVE) void attention_f32_merge_kernel(const int* __restrict__ positions, const float* __restrict__ sums, const float* __restrict__ maxima,
                                                                  int items, int nq, int slots, int window, float* __restrict__ out, int out_stride) {
  const int item = blockIdx.x * WAVE + threadIdx.x;
  if (item >= items) return;
  const int row = item / (D / 4), dim = item % (D / 4) * 4, token = row / nq, head = row % nq;
  const float* from = sums + (int64_t)row * slots * D + dim;
  const float* tops = maxima + (int64_t)row * slots * 2;
  const int pos = positions[token];
  float run_max = -INFINITY, run_sum = 0.f;
  floatx4 run = {0.f, 0.f, 0.f, 0.f};
  int pieces = slots;
  for (int p0 = 0; p0 < pieces; p0 += MERGE_AHEAD) {
    floatx4 part[MERGE_AHEAD];
    floatx2 ml[MERGE_AHEAD];
#pragma unroll
    for (int e = 0; e < MERGE_AHEAD; ++e) {
      const int p = p0 + e < slots ? p0 + e : slots - 1;
      part[e] = *(const floatx4*)(from + (int64_t)p * D);
      ml[e] = *(const floatx2*)(tops + 2 * p);
    }
    if (p0 == 0) {
      const int seen = pos / PIECE - first_seen(pos, window) / PIECE + 1;
      pieces = seen < slots ? seen : slots;
    }
#pragma unroll
    for (int e = 0; e < MERGE_AHEAD; ++e)
      if (p0 + e < pieces) {
        const float now = fmaxf(run_max, ml[e][0]), keep = moved(run_max, now), take = moved(ml[e][0], now);
        run_sum = fmaf(run_sum, keep, ml[e][1] * take);
#pragma unroll
        for (int i = 0; i < 4; ++i) run[i] = fmaf(run[i], keep, part[e][i] * take);
        run_max = now;
      }
  }
  *(floatx4*)(out + (int64_t)token * out_stride + head * D + dim) = run * (1.f / run_sum);
}

template <int D, int WAVES, bool SHORT, bool DIRECT>
void launch(float* out, int out_stride, const float* q, int q_stride, const float* k_pages, const float* v_pages, const int* block_table, int table_stride,
            const int* token_request, const int* positions, int tokens, int heads, int nkv, int page_size, float scale, int window, int together,
            hipStream_t s) {
  const dim3 grid((tokens + together - 1) / together, nkv);
  attention_f32_mfma_kernel<D, WAVES, SHORT, DIRECT><<<grid, WAVES * WAVE, 0, s>>>(
      positions, token_request, block_table, q, table_stride, q_stride, tokens, together, heads, (int)grid.x, k_pages, v_pages, out, out_stride, nkv, page_size,
      scale, window);
}

}  // namespace

bool lrs_attention_f32_takes(const void* out, int out_stride, const void* q, int q_stride, const void* k_pages, const void* v_pages, int nq, int nkv,
                             int d, int dv, int page_size) {
  const uintptr_t places = (uintptr_t)out | (uintptr_t)q | (uintptr_t)k_pages | (uintptr_t)v_pages;
  return d == dv && (d == 32 || d == 64 || d == 96 || d == 128) && nq / nkv <= COLUMNS && page_size % 16 == 0 && places % 16 == 0 && out_stride % 4 == 0 && q_stride % 4 == 0;
}

// Whether keys and values go straight into registers (DIRECT): where a wave has one piece or two and waits for its first block, which comes a
// trip through LDS sooner, and where rows of a request each fill nearly one round of the chip over a few hundred keys.  us, direct / through LDS,
// 8 kv heads of 128: one row at 100 tokens 9.1 / 9.9, at 160 9.9 / 10.4, at 255 10.8 / 10.6; 32 rows at 255 14.5 / 15.1, at 509 27.7 / 28.1; 28 rows at
// 700 33.8 / 34.4; 32 at 2,000 97.8 / 95.3; 24 at 509 23.5 / 22.9; a prompt of 64 tokens 11.0 / 11.3, of 150 12.7 / 12.4, of 509 39.9 / 34.7.
LRS_API int lrs_attention_f32_direct(int64_t workgroups, int together, int longest) {
  const int units = lrs_compute_units() > 0 ? lrs_compute_units() : 256;
  if (longest <= 0) return 0;
  if (longest <= 2 * PIECE) return 1;
  if (together > 1) return 0;
  if (longest <= 4 * PIECE) return longest <= 3 * PIECE || 2 * workgroups >= units;
  return longest < 1024 && 4 * workgroups > 3 * units && workgroups <= units;
}

// together: the most consecutive tokens that may share a workgroup (1: a step in which every request brings one token).
// longest: no token's position + 1 is beyond it (0: not known).  Speed alone depends on either.
int lrs_attention_f32(float* out, int out_stride, const float* q, int q_stride, const float* k_pages, const float* v_pages, const int* block_table,
                      int table_stride, const int* token_request, const int* positions, int tokens, int nq, int nkv, int d, int page_size,
                      float scale, int window, int together, int longest, hipStream_t s) {
  const int heads = nq / nkv, fit = COLUMNS / heads;
  if (together > fit) together = fit;
  if (together < 1) together = 1;
  // Short contexts: blocks of keys that nobody sees are left out (SHORT; a branch a block, 0.7 us a launch where none are), up to 32
  // tokens, and more workgroups than units over a few pieces each have two waves, four times as many one: most of eight would wait
  // with nothing to do.  us of 64 tokens at 30 and at 100, eight waves before / now (the kernel for any shape): 32 heads of 128 on 32 58 / 17
  // (15) and 63 / 37 (36), 32 on 8 16 / 8 (12) and 18 / 16 (29), 16 heads of 64 on 16 21 / 7 (8) and 23 / 12 (17); one token at 10, 32 on 8 8.4 / 6.5 (5.3).
  const int64_t workgroups = (int64_t)((tokens + together - 1) / together) * nkv;
  const bool few_pieces = longest > 0 && longest <= 4 * PIECE, direct = lrs_attention_f32_direct(workgroups, together, longest) != 0;
  const int items = together * heads * (d / 4);                            // what the merge has to do, one a thread
#define CALL(D, WAVES, SHORT, DIRECT)                                                                                                          \
  launch<D, WAVES, SHORT, DIRECT>(out, out_stride, q, q_stride, k_pages, v_pages, block_table, table_stride, token_request, positions, tokens, heads, nkv, \
                          page_size, scale, window, together, s)
#define SIZE(D)                                                  \
  do {                                                           \
    if (few_pieces && workgroups > 4 * lrs_compute_units() && items <= WAVE) CALL(D, 1, true, true);     \
    else if (few_pieces && workgroups > lrs_compute_units() && items <= 2 * WAVE) CALL(D, 2, true, true); \
    else if (longest > 0 && longest <= 32) CALL(D, 8, true, true);                                      \
    else if (direct) CALL(D, 8, false, true);                                                           \
    else CALL(D, 8, false, false);                                                                      \
  } while (0)
  if (d == 32) SIZE(32);
  else if (d == 64) SIZE(64);
  else if (d == 96) SIZE(96);
  else SIZE(128);
#undef SIZE
#undef CALL
  return lrs_check_launch("attention");
}

// The same for a step in which every request brings one token, the pieces of a token divided between `splits` workgroups, with the bits of
// lrs_attention: heads of 64 and 128, at most four a kv head.  No token sees more than `slots` pieces of 64 positions (what lies beyond is
// left out); part_o holds tokens * nq * slots * d floats and part_ml two for every d.
LRS_API int lrs_attention_f32_divided(float* out, int out_stride, const float* q, int q_stride, const float* k_pages, const float* v_pages, const int* block_table,
                                      int table_stride, const int* token_request, const int* positions, int tokens, int nq, int nkv, int d, int page_size,
                                      float scale, int window, int splits, int slots, float* part_o, float* part_ml, void* stream) {
  LRS_REQUIRE(tokens > 0 && nq > 0 && nkv > 0 && nq % nkv == 0 && page_size > 0, "attention_f32_divided: bad sizes tokens=%d nq=%d nkv=%d page=%d", tokens, nq, nkv, page_size);
  LRS_REQUIRE(lrs_attention_f32_takes(out, out_stride, q, q_stride, k_pages, v_pages, nq, nkv, d, d, page_size) && d % 64 == 0 && nq / nkv <= FEW,
              "attention_f32_divided: takes heads of 64 or 128, at most 4 a kv head, pages of a multiple of 16, 16-byte aligned rows (nq=%d nkv=%d d=%d page=%d)", nq, nkv, d, page_size);
  LRS_REQUIRE(splits > 0 && splits <= 65535 && slots > 0 && part_o && part_ml && ((uintptr_t)part_o | (uintptr_t)part_ml) % 16 == 0,
              "attention_f32_divided: needs buffers for the parts' results (splits=%d slots=%d)", splits, slots);
  LRS_REQUIRE((int64_t)tokens * nq * (d / 4) < (1 << 30) && nkv <= 65535, "attention_f32_divided: too many rows (tokens=%d nq=%d nkv=%d)", tokens, nq, nkv);
  const hipStream_t s = (hipStream_t)stream;
  const int items = tokens * nq * (d / 4);
  const dim3 grid(tokens, nkv, splits);
#define SIZE(D)                                                                                                                                            \
  do {                                                                                                                                                     \
    attention_f32_few_kernel<D><<<grid, WAVE, 0, s>>>(positions, token_request, block_table, q, table_stride, q_stride, nq / nkv, splits, k_pages,        \
                                                      v_pages, part_o, part_ml, slots, nkv, page_size, scale, window);                                    \
    if (int rc = lrs_check_launch("attention_f32_divided")) return rc;                                                                                    \
    attention_f32_merge_kernel<D><<<(items + WAVE - 1) / WAVE, WAVE, 0, s>>>(positions, part_o, part_ml, items, nq, slots, window, out, out_stride);      \
  } while (0)
  if (d == 64) SIZE(64);
  else SIZE(128);
#undef SIZE
  return lrs_check_launch("attention_f32_divided");
}
