// Causal attention over the paged cache for a ragged batch: every query token attends to
// the cached keys of its own request at positions lo..p, p being the token's absolute
// position and lo = 0, max(0, p - window + 1) with a sliding window, or the start of p's chunk
// (first_seen in common.h: `window` 0, positive or negative).  Keys and values of this
// step's tokens are already in the cache when these kernels run.
//
// Key pages are [page, kv_head, slot, dim], value pages [page, kv_head, dim, slot] (transposed
// inside a page); block_table[r, i] is the page holding positions i*page_size ..
// (i+1)*page_size-1 of request r.  Scores, softmax and the weighted sum are
// float32.  Key tiles start at multiples of the tile size counted from position 0, so the
// rounding of a query's result depends on its position only, never on how the sequence
// was cut into steps.
#include <type_traits>

#include "common.h"

int lrs_attention_f32(float* out, int out_stride, const float* q, int q_stride, const float* k_pages, const float* v_pages, const int* block_table,
                      int table_stride, const int* token_request, const int* positions, int tokens, int nq, int nkv, int d, int page_size,
                      float scale, int window, int together, int longest, hipStream_t s);
bool lrs_attention_f32_takes(const void* out, int out_stride, const void* q, int q_stride, const void* k_pages, const void* v_pages, int nq, int nkv,
                             int d, int dv, int page_size);

// 2^x by the hardware instruction alone (arguments here are <= 0 or -inf; results below the
// smallest normal number may flush to zero, which a softmax weight can afford).
__device__ __forceinline__ float fast_exp2(float x) { return __builtin_amdgcn_exp2f(x); }

// How far (in powers of two) a new maximum must exceed the reference point of a running softmax
// before the reference point moves and the accumulators are rescaled.
constexpr float RESCALE_STEP = 8.0f;

// A cap on the scores: cap * tanh(x / cap), close to x for small |x| and within (-cap, cap) for all.  tanh by one
// exponential and one reciprocal (the hardware's, a unit in the last place each): the bfloat16 kernels' form; the kernel for
// any shape, which also serves float32 runs, calls tanhf.
__device__ __forceinline__ float capped(float x, float cap) {
  const float t = x * __builtin_amdgcn_rcpf(cap);
  const float e = fast_exp2(-2.f * 1.4426950408889634f * fabsf(t));       // e^(-2|t|), in (0, 1]
  const float r = (1.f - e) * __builtin_amdgcn_rcpf(1.f + e);
  return copysignf(cap * r, t);
}

// A sink: one more term exp(sink) in a softmax's denominator that has no key and no value.  Given sums that were taken
// against the reference point `top` (both in powers of two, as every kernel here keeps them), returns the factor for
// the weighted sums and changes `total` so that factor * sums / total is the softmax with the sink.
__device__ __forceinline__ float with_sink(float sink2, float top, float& total) {
  const float m = fmaxf(top, sink2);
  const float keep = top == -INFINITY ? 0.f : fast_exp2(top - m);
  total = total * keep + fast_exp2(sink2 - m);
  return keep;
}
constexpr float LOG2E = 1.4426950408889634f;

// A bias by distance, i the query's position, j the key's, in one of two forms:
//   DISTANCE_LOG     a score of query head h loses rate_h * ln(1 + reach_h * (i - j)); `distance` holds the rates of all nq heads,
//                    then their reaches;
//   DISTANCE_LINEAR  it loses rate_h * (i - j); `distance` holds the rates.
// (distance null: no bias.)  In the bfloat16 kernels the logarithm is the hardware's (base 2, a unit in the last place), and the
// distance from a query to the first key of a lane's four (or eight) is taken in whole positions before it meets the reach (or the
// rate), so that a near key's distance is exact however far on the sequence is.
enum { DISTANCE_LOG = 0, DISTANCE_LINEAR = 1 };
__device__ __forceinline__ float distance_loss(float rate2, float reach, float distance) {       // rate2: for base-2 logarithms
  return rate2 * __builtin_amdgcn_logf(fmaf(reach, distance, 1.f));
}
constexpr float LN2 = 0.6931471805599453f;
// Either form, in the base-2 units the scores have where it is taken off.
__device__ __forceinline__ float distance_loss_of(const float* __restrict__ distance, int form, int nq, int head, float behind) {
  return form == DISTANCE_LINEAR ? distance[head] * LOG2E * behind : distance_loss(distance[head], distance[nq + head], behind);
}

// A linear bias makes the scores of a walk towards the query rise by the rate at every position, so a reference point that fits a tile
// is soon far below the next ones'.  A walk whose weights have grown beyond GROWN raises its reference points by what brings the sums
// down to 2^-40 (never further: nothing that has been added up is lost) and goes on; `more` is what to add to the reference point, in
// powers of two, a whole number that the four lanes of a query agree on.
constexpr float GROWN = 0x1p24f;
__device__ __forceinline__ float growth_of(float run_sum) {
  float most = fmaxf(run_sum, __shfl_xor(run_sum, 16, WAVE));
  most = fmaxf(most, __shfl_xor(most, 32, WAVE));
  return most >= 1.f ? floorf(__builtin_amdgcn_logf(most)) + 40.f : 0.f;
}

// The linear form of the bias for four keys in a row, the first of them `behind` positions behind the query.
__device__ __forceinline__ floatx4 linear_of_four(float rate, float behind) {
  const float first = -rate * behind;
  return floatx4{first, first + rate, fmaf(rate, 2.f, first), fmaf(rate, 3.f, first)};
}

// A gate a head: the head's output times sigmoid(gates[token, head]), the gate values lying in rows of their own stride (the
// columns of the projection that made them).  Null: no gate.
template <typename T>
__device__ __forceinline__ float head_gate(const T* __restrict__ gates, int gate_stride, int64_t token, int head) {
  return gates ? 1.0f / (1.0f + __expf(-(float)gates[token * gate_stride + head])) : 1.f;
}

// ---------------------------------------------------------- generic kernel
// One workgroup per (query token, query head); any head_dim, values of any size dv up to 4 * threads.  keep_first: with a
// window, the keys at positions below keep_first stay visible however far back they lie (they keep their positions).
template <typename T, int THREADS>
__global__ __launch_bounds__(THREADS) void attention_generic_kernel(
    T* __restrict__ out, int out_stride, const T* __restrict__ q, int q_stride,
    const T* __restrict__ k_pages, const T* __restrict__ v_pages,
    const int* __restrict__ block_table, int table_stride, const int* __restrict__ token_request,
    const int* __restrict__ positions, int nq, int nkv, int d, int dv, int page_size, float scale,
    int window, int keep_first, const float* __restrict__ sinks, float softcap, const T* __restrict__ gates, int gate_stride,
    const float* __restrict__ distance, int distance_form) {
  extern __shared__ __attribute__((aligned(16))) float smem[];
  float* qs = smem;                           // [d]
  float* probs = qs + d + d % 2;              // [THREADS]
  int64_t* bases = (int64_t*)(probs + THREADS);  // [THREADS] index of each key's (page, kv head) block
  int* offsets = (int*)(bases + THREADS);        // [THREADS] slot of each key inside its page
  __shared__ float scratch[16];

  const int token = blockIdx.x, head = blockIdx.y, tid = threadIdx.x;
  const int request = token_request[token];
  const int pos = positions[token];
  const int kv_head = head / (nq / nkv);
  const int lo = first_seen(pos, window);
  const int kept = lo > 0 ? (keep_first < lo ? keep_first : lo) : 0;    // keys 0 .. kept-1 are seen besides lo .. pos
  const int* table = block_table + (int64_t)request * table_stride;

  for (int i = tid; i < d; i += THREADS) qs[i] = to_float(q[(int64_t)token * q_stride + (int64_t)head * d + i]);
  __syncthreads();

  float acc[4] = {0.f, 0.f, 0.f, 0.f};
  float running_max = -INFINITY, running_sum = 0.f;
  const int lo_tile = (lo / THREADS) * THREADS;
  for (int tile = kept > 0 ? 0 : lo_tile; tile <= pos; tile += THREADS) {
    if (tile >= kept && tile < lo_tile) {     // nothing to see between the kept keys and the window
      tile = lo_tile - THREADS;
      continue;
    }
    const int key = tile + tid;
    const bool valid = key <= pos && (key >= lo || key < kept);
    float score = -INFINITY;
    int64_t base = 0;
    const int off = key % page_size;
    if (valid) {
      const int64_t page = table[key / page_size];
      base = page * nkv + kv_head;
      const T* kr = k_pages + (base * page_size + off) * d;
      float dot = 0.f;
      if (sizeof(T) == 4 && d % 4 == 0 && ((uintptr_t)k_pages % 16) == 0) {
        // float32 rows, 16 bytes a load; the products are added up in the same order as one by one
        for (int i = 0; i < d; i += 4) {
          const floatx4 kv = *(const floatx4*)((const float*)kr + i);
          dot = fmaf(qs[i], kv[0], dot);
          dot = fmaf(qs[i + 1], kv[1], dot);
          dot = fmaf(qs[i + 2], kv[2], dot);
          dot = fmaf(qs[i + 3], kv[3], dot);
        }
      } else {
        for (int i = 0; i < d; ++i) dot = fmaf(qs[i], to_float(kr[i]), dot);
      }
      score = dot * scale;
      if (softcap > 0.f) score = softcap * tanhf(score / softcap);
      if (distance)
        score -= distance_form == DISTANCE_LINEAR ? distance[head] * (float)(pos - key)
                                                  : distance[head] * logf(1.f + distance[nq + head] * (float)(pos - key));
    }
    const float tile_max = block_max(score, scratch);
    const float new_max = fmaxf(running_max, tile_max);
    const float p = valid ? expf(score - new_max) : 0.f;
    const float tile_sum = block_sum(p, scratch);
    const float alpha = expf(running_max - new_max);  // exp(-inf) = 0 on the first tile
    running_sum = running_sum * alpha + tile_sum;
    running_max = new_max;
    probs[tid] = p;
    bases[tid] = base * page_size * dv;
    offsets[tid] = off;
    __syncthreads();
    const int count = (pos - tile + 1 < THREADS) ? pos - tile + 1 : THREADS;
    const bool whole = tile >= lo;             // every key of the tile up to pos is seen, so each has a page to read from
#pragma unroll
    for (int c = 0; c < 4; ++c) {
      const int dim = tid + c * THREADS;
      if (dim < dv) {
        float a = acc[c] * alpha;
        int j = 0;
        if (whole && sizeof(T) == 4 && page_size % 4 == 0 && THREADS % 4 == 0 && ((uintptr_t)v_pages % 16) == 0) {
          // four keys that lie side by side in a (transposed) page in one load of 16 bytes; added in key order as below
          for (; j + 4 <= count; j += 4) {
            const floatx4 vv = *(const floatx4*)((const float*)v_pages + bases[j] + (int64_t)dim * page_size + offsets[j]);
#pragma unroll
            for (int e = 0; e < 4; ++e) {
              const float pj = probs[j + e];
              if (pj != 0.f) a = fmaf(pj, vv[e], a);
            }
          }
        }
        for (; j < count; ++j) {
          const float pj = probs[j];
          if (pj != 0.f) a = fmaf(pj, to_float(v_pages[bases[j] + (int64_t)dim * page_size + offsets[j]]), a);
        }
        acc[c] = a;
      }
    }
    __syncthreads();
  }
  float keep = 1.f;
  if (sinks) {      // one more term in the denominator, with no key and no value
    const float sink = sinks[head], top = fmaxf(running_max, sink);
    keep = expf(running_max - top);
    running_sum = running_sum * keep + expf(sink - top);
  }
  const float inv = keep / running_sum * head_gate(gates, gate_stride, token, head);
#pragma unroll
  for (int c = 0; c < 4; ++c) {
    const int dim = tid + c * THREADS;
    if (dim < dv) out[(int64_t)token * out_stride + (int64_t)head * dv + dim] = from_float<T>(acc[c] * inv);
  }
}

// ------------------------------------------------- bf16 decode kernel
// What the decode kernel does to raw q, k and v rows when it also does the work of qk_prep: the
// per-head RMSNorm of q and k (weights null: none), the rotation of pairs (i, i + D/2) by the
// step's cos/sin tables (null: none) and the write of the new key and value into the pages.
struct DecodePrep {
  const void* q_weight;   // [D]
  const void* k_weight;   // [D]
  int weight_is_f32;
  float eps;
  const float* cosv;      // [tokens, D/2]
  const float* sinv;
  int kv_columns;         // kv heads held in the qkv rows after the q heads: k, then v; 0: keys and
                          // values are another layer's, already in the pages
};

// One head row, raw -> normalised and rotated, in the operand layout of the 16x16x32 products: the
// lane holds dims c*32 + g*8 .. +8 of every 32-dim chunk c, the four lanes g = 0..3 with equal
// lane % 16 hold one head between them.  All 64 lanes must call it together.
// What it needs besides the row is asked for on its own (HeadWeights, HeadTables), so that a kernel can do so before
// anything makes it wait; head_from_registers: from a row already in registers.
template <int D>
struct HeadWeights {      // the norm's weights of the lane's dims; left alone without a norm
  floatx4 raw[D / 32][2];
  __device__ __forceinline__ void fetch(const void* __restrict__ weight, int is_f32, int g) {
    if (!weight) return;
    // 16-byte loads (the host checks the alignment); bfloat16 weights need one for eight and load it twice: no branch around a load
    const int size = is_f32 ? 4 : 2;
#pragma unroll
    for (int c = 0; c < D / 32; ++c) {
      const char* from = (const char*)weight + (c * 32 + g * 8) * size;
      raw[c][0] = *(const floatx4*)from;
      raw[c][1] = *(const floatx4*)(from + (is_f32 ? 16 : 0));
    }
  }
  __device__ __forceinline__ float value(int c, int j, int is_f32) const {
    union { floatx4 f; bf16x8 b; } whole{raw[c][0]};
    return is_f32 ? raw[c][j / 4][j % 4] : (float)whole.b[j];
  }
};
template <int D>
struct HeadTables {       // the rotation's cosines and sines of the lane's dims; left alone without a rotation
  floatx4 cs[D < 64 ? 1 : D / 64][2], sn[D < 64 ? 1 : D / 64][2];
  __device__ __forceinline__ void fetch(const float* __restrict__ cosrow, const float* __restrict__ sinrow, int g) {
    if (!cosrow) return;
#pragma unroll
    for (int c = 0; c < D / 64; ++c)
#pragma unroll
      for (int n = 0; n < 2; ++n) {
        cs[c][n] = *(const floatx4*)(cosrow + c * 32 + g * 8 + 4 * n);
        sn[c][n] = *(const floatx4*)(sinrow + c * 32 + g * 8 + 4 * n);
      }
  }
};
// One head's norm and rotation: weights_of(c, w) and tables_of(c, cs, sn) give a chunk's eight weights, cosines and sines.
template <int D, typename Weights, typename Tables>
__device__ __forceinline__ void norm_and_rotate(bf16x8 (&r)[D / 32], float (&x)[D / 32][8], bool normed, float eps, bool rotated,
                                                const Weights& weights_of, const Tables& tables_of) {
  constexpr int DS = D / 32;
  if (normed) {
    float ss = 0.f;
#pragma unroll
    for (int c = 0; c < DS; ++c)
#pragma unroll
      for (int j = 0; j < 8; ++j) ss = fmaf(x[c][j], x[c][j], ss);
    ss += __shfl_xor(ss, 16, WAVE);
    ss += __shfl_xor(ss, 32, WAVE);
    const float inv = 1.0f / sqrtf(ss / (float)D + eps);
#pragma unroll
    for (int c = 0; c < DS; ++c) {
      float w[8];
      weights_of(c, w);
#pragma unroll
      for (int j = 0; j < 8; ++j) x[c][j] = x[c][j] * inv * w[j];
    }
  }
  if (rotated) {
#pragma unroll
    for (int c = 0; c < D / 64; ++c) {
      float cs[8], sn[8];
      tables_of(c, cs, sn);
#pragma unroll
      for (int j = 0; j < 8; ++j) {
        const float a = x[c][j], b = x[c + DS / 2][j];
        x[c][j] = a * cs[j] - b * sn[j];
        x[c + DS / 2][j] = b * cs[j] + a * sn[j];
      }
    }
  }
#pragma unroll
  for (int c = 0; c < DS; ++c)
#pragma unroll
    for (int j = 0; j < 8; ++j) r[c][j] = (bf16)x[c][j];
}
template <int D>
__device__ __forceinline__ void head_from_registers(bf16x8 (&r)[D / 32], float (&x)[D / 32][8], bool normed, const HeadWeights<D>& weights,
                                                    int weight_is_f32, float eps, bool rotated, const HeadTables<D>& tables) {
  norm_and_rotate<D>(
      r, x, normed, eps, rotated,
      [&](int c, float (&w)[8]) {
#pragma unroll
        for (int j = 0; j < 8; ++j) w[j] = weights.value(c, j, weight_is_f32);
      },
      [&](int c, float (&cs)[8], float (&sn)[8]) {
#pragma unroll
        for (int j = 0; j < 8; ++j) cs[j] = tables.cs[c][j / 4][j % 4], sn[j] = tables.sn[c][j / 4][j % 4];
      });
}

// The same for the prompt kernels, whose waves prepare their queries once a walk and have no registers to spare: weights and
// tables are loaded where they are used (asked for first they cost 30 to 90 spilled registers), in 16-byte loads (the host checks
// their alignment).
template <int D>
__device__ __forceinline__ void head_from_memory(bf16x8 (&r)[D / 32], float (&x)[D / 32][8], int g, const void* __restrict__ weight,
                                                 int weight_is_f32, float eps, const float* __restrict__ cosrow, const float* __restrict__ sinrow) {
  norm_and_rotate<D>(
      r, x, weight != nullptr, eps, cosrow != nullptr,
      [&](int c, float (&w)[8]) {
        if (weight_is_f32) {
          const floatx4 w0 = *(const floatx4*)((const float*)weight + c * 32 + g * 8), w1 = *(const floatx4*)((const float*)weight + c * 32 + g * 8 + 4);
#pragma unroll
          for (int j = 0; j < 4; ++j) w[j] = w0[j], w[4 + j] = w1[j];
        } else {
          const bf16x8 wb = *(const bf16x8*)((const bf16*)weight + c * 32 + g * 8);
#pragma unroll
          for (int j = 0; j < 8; ++j) w[j] = (float)wb[j];
        }
      },
      [&](int c, float (&cs)[8], float (&sn)[8]) {
#pragma unroll
        for (int n = 0; n < 2; ++n) {
          const floatx4 c4 = *(const floatx4*)(cosrow + c * 32 + g * 8 + 4 * n), s4 = *(const floatx4*)(sinrow + c * 32 + g * 8 + 4 * n);
#pragma unroll
          for (int j = 0; j < 4; ++j) cs[4 * n + j] = c4[j], sn[4 * n + j] = s4[j];
        }
      });
}

// One query token per request (a decode step).  A workgroup of four waves owns one
// (token, kv head, split): the query heads that share the kv head (at most 16) sit in the
// columns of the matrix-core tiles, so every key and value is loaded once for the whole
// group.  Keys are walked in tiles of 32; the tiles of a token are divided between `splits`
// workgroups (so that few long requests still fill the chip) and, inside a workgroup,
// dealt to the waves in turn.  Per tile:
//     S[key, head]   = K[key, :] . Q[head, :]          A = K rows (16 keys x 32 dims per MFMA)
//     P              = exp2(S * scale*log2(e) - max)   online softmax per head column
//     O^T[dim, head] += V^T[dim, key] . P[key, head]   A = V^T rows, read from the transposed page
// S comes out of the first product with a head per lane column and four keys per lane, which
// is exactly the operand layout the second product wants for P, so P never leaves registers.
// Waves are merged through LDS, splits by attention_merge_kernel.
// PREP: q holds the raw rows of the q/k/v product; the kernel prepares q and the new key itself; the wave that
// meets the token's own position takes that key and the new value in place of what the pages hold there, and
// its workgroup writes both into the pages (see DecodePrep).
// What bounds a walk of few keys is the chain of trips to memory (position, block table, keys) and what stands between them;
// so nothing that is asked for hides behind a branch, rows, weights and tables are asked for first, and only the wave that
// meets the new key waits for it.  A step of the 0.6B shape (28 layers, 16 heads on 8), one request at 509 tokens: 1,166 ->
// 1,076 us, 16 requests 1,276 -> 1,176; of the 8B shape (36 layers, 32 heads on 8) at 2,048 tokens, 8 requests 3,968 -> 3,879,
// 64 requests 7,040 -> 6,930: two and a half to three and a half microseconds a layer.  One wave prepares queries and key for the
// workgroup (all eight did, and the wave with the new key twice): 1,034 -> 1,000 us, 1,177 -> 1,161, 3,640 -> 3,606; of the 10.5 us that
// were inside the kernel 2 passed before the keys could be asked for behind that work's loads, 0.7 preparing, 1.3 with the new key alone.
// MORE: values narrower than keys and a bias by distance (dv and distance are looked at); instances of their own, so that the
// others are spared the checks.
template <int D, int WAVES>
struct DecodeLds {
  float sm_m[WAVES][16], sm_l[WAVES][16];
  __attribute__((aligned(16))) float sm_o[WAVES][16][D + 4];     // a head's dims side by side, heads four banks apart
  __attribute__((aligned(16))) bf16 queries[16][D + 8];           // prepared heads, four banks apart
  __attribute__((aligned(16))) bf16 own_k[D];
  bf16 own_v[D];
};
struct Inner { static constexpr bool value = false; };
struct End { static constexpr bool value = true; };
template <int D, bool PREP, int WAVES, bool AHEAD, bool MORE, bool ONCE>
__device__ __forceinline__ void attention_decode_part(
    DecodeLds<D, WAVES>& lds, int* page_ids, int split, int kvh, int token,
    bf16* __restrict__ out, int out_stride, float* __restrict__ part_o, float* __restrict__ part_ml,
    const bf16* __restrict__ q, int q_stride, bf16* __restrict__ k_pages,
    bf16* __restrict__ v_pages, const int* __restrict__ block_table, int table_stride,
    const int* __restrict__ token_request, const int* __restrict__ positions, int nq, int nkv,
    int page_size, float scale, int window, int splits, int slots, DecodePrep prep, const float* __restrict__ sinks,
    float softcap, const bf16* __restrict__ gates, int gate_stride, int dv_given, const float* __restrict__ distance_given,
    int distance_form) {
  constexpr int DS = D / 32, DB = D / 16, THREADS = WAVES * 64;
  const int dv = MORE ? dv_given : D;
  const float* __restrict__ distance = MORE ? distance_given : nullptr;
  auto &sm_m = lds.sm_m, &sm_l = lds.sm_l;
  auto& sm_o = lds.sm_o;
  const int tid = threadIdx.x, lane = tid % WAVE, wave = tid / WAVE;
  const int col = lane & 15, g = lane >> 4;
  const int pos = positions[token], request = token_request[token];
  asm volatile("" :: "s"(pos), "s"(request));                               // asked for together: the compiler would put the second off
  const int group = nq / nkv;
  const int* table = block_table + (int64_t)request * table_stride;
  const int lo = first_seen(pos, window);
  const int first_tile = lo / 32, last_tile = pos / 32;
  const int per_split = (last_tile - first_tile + splits) / splits;
  const int tile_begin = first_tile + split * per_split;
  const int tile_end = tile_begin + per_split <= last_tile + 1 ? tile_begin + per_split : last_tile + 1;
  // PREP: the raw rows, the norms' weights and the rotation's tables are asked for now, before anything here waits for
  // memory: they are there when the first keys are on their way.  (The new key and value too, since which workgroup walks the token's
  // position is not known yet; they are the token's own, whichever does.)
  // One wave, the last, does so for the workgroup: eight that all did would ask their compute unit for 160 loads of rows, weights and
  // tables before the first keys.  The new key is prepared where the queries are, in the column behind the group's heads (a group of 16
  // leaves none: there it follows them).
  const bf16* q_row = q + (int64_t)token * q_stride;
  const bool normed = PREP && prep.q_weight, rotated = PREP && prep.cosv, brings_key = PREP && prep.kv_columns > 0;
  const bool prepares = PREP && wave == WAVES - 1, key_column = brings_key && group < 16 && col == group;
  bf16x8 qf[DS];
  bf16 raw_v[(D + WAVE - 1) / WAVE];
  HeadWeights<D> weights;
  HeadTables<D> tables;
  if (!PREP || prepares) {
    const bf16* my_row = q_row + (int64_t)(key_column ? nq + kvh : kvh * group + (col < group ? col : 0)) * D + g * 8;
#pragma unroll
    for (int c = 0; c < DS; ++c) qf[c] = *(const bf16x8*)(my_row + c * 32);
    if (normed) weights.fetch(key_column ? prep.k_weight : prep.q_weight, prep.weight_is_f32, g);
    if (rotated) tables.fetch(prep.cosv + (int64_t)token * (D / 2), prep.sinv + (int64_t)token * (D / 2), g);
    if (brings_key) {
      const bf16* v_row = q_row + (int64_t)(nq + prep.kv_columns + kvh) * D;
#pragma unroll
      for (int n = 0; n < (D + WAVE - 1) / WAVE; ++n) raw_v[n] = v_row[min(lane + n * WAVE, D - 1)];
    }
  }

  // the block table entries of this workgroup's tiles, in LDS: the address of a key must not
  // wait for a trip to memory of its own.  (A split that has no tiles left looks the last one's up.)
  const int first_block = min(tile_begin, last_tile) * 32 / page_size;
  const int last_key = min(max(tile_end, min(tile_begin, last_tile) + 1) * 32 - 1, pos);
  for (int i = tid; i <= last_key / page_size - first_block; i += THREADS) page_ids[i] = table[first_block + i];
  __syncthreads();

  const bf16x8 zero8 = {0, 0, 0, 0, 0, 0, 0, 0};
  // Every key and value fragment of a tile is requested before any is used, so a tile costs one
  // trip to memory instead of two.  Which of the tile's 32 keys a row of the two key blocks stands
  // for is chosen so that a lane ends up with the weights of eight consecutive keys, g*8 .. g*8+7:
  // block h, row 4*r + i is key 8*r + 4*h + i.  The values of those eight keys lie side by side in
  // the (transposed) page, one 16-byte load a dim.  A key or eight keys that the token does not see
  // are read from the nearest it does see, not branched around (three branches were three trips to
  // memory one after the other): their scores are replaced, their values zeroed (work, below).
  // (A tile is two runs of 16 keys, each in one page; looked up once for the wave, with numbers that it shares, pages cost more than every lane's
  // own lookup: heads that come prepared, batch 128 at 64 tokens 11.7 us by lane / 13.1, 32 tokens 11.1 / 12.7, 300 27.2 / 27.7, one request at 40 4.5 / 4.9;
  // heads prepared here, 16 requests seeing 128 of 4,000 7.8 / 8.0, others the same.)
  const int key_of_row = (col >> 2) * 8 + (col & 3);           // + 4*h
  // (ONCE: with the hint that says that a key or value is read by this workgroup alone, see lrs_attention_decode)
  auto fetch = [&](int tile, bf16x8 (&kf)[2][DS], bf16x8 (&vf)[DB]) {
    const bf16* kp[2];
#pragma unroll
    for (int h = 0; h < 2; ++h) {
      const int key = max(lo, min(pos, tile * 32 + key_of_row + 4 * h));
      const int64_t page = page_ids[key / page_size - first_block];
      kp[h] = k_pages + ((page * nkv + kvh) * page_size + key % page_size) * D + g * 8;
    }
    const int key8 = max(lo & ~7, min(pos & ~7, tile * 32 + g * 8));         // this lane's eight keys; pages hold multiples of 16
    const int64_t page = page_ids[key8 / page_size - first_block];
    const bf16* vp = v_pages + (page * nkv + kvh) * (int64_t)dv * page_size + (int64_t)col * page_size + key8 % page_size;
#pragma unroll
    for (int h = 0; h < 2; ++h)
#pragma unroll
      for (int c = 0; c < DS; ++c) kf[h][c] = ONCE ? load_once((const bf16x8*)(kp[h] + c * 32)) : *(const bf16x8*)(kp[h] + c * 32);
    // (values narrower than keys: the blocks behind them repeat the last one, and nothing of them is written)
#pragma unroll
    for (int b = 0; b < DB; ++b) {
      const bf16x8* at = (const bf16x8*)(vp + (int64_t)(b * 16 < dv ? b * 16 : dv - 16) * page_size);
      vf[b] = ONCE ? load_once(at) : *at;
    }
  };
  // AHEAD: the wave's first tile is asked for as soon as the page ids are there, before the query (and
  // the new key) are prepared, so that the first trip to memory runs beside that work.  No branch around it, a wave
  // without a tile asks for the last one: where loads may or may not be on their way, the compiler waits for all.
  bf16x8 kf_a[AHEAD ? 2 : 1][AHEAD ? DS : 1], vf_a[AHEAD ? DB : 1];
  if constexpr (AHEAD) {
    fetch(min(tile_begin + wave, max(tile_end - 1, min(tile_begin, last_tile))), (bf16x8(&)[2][DS])kf_a, (bf16x8(&)[DB])vf_a);
  }
  auto prepare = [&](bf16x8 (&row)[DS]) {
    float x[DS][8];
#pragma unroll
    for (int c = 0; c < DS; ++c)
#pragma unroll
      for (int j = 0; j < 8; ++j) x[c][j] = (float)row[c][j];
    head_from_registers<D>(row, x, normed, weights, prep.weight_is_f32, prep.eps, rotated, tables);
  };
  // The queries, the new key and the new value meet the waves in LDS; the workgroup that walks the token's own position writes key and
  // value into the pages, and its wave that meets the position takes them in place of what the pages hold there.
  auto &own_k = lds.own_k, &own_v = lds.own_v;
  const bool own_here = brings_key && tile_begin <= last_tile && last_tile < tile_end;
  const bool holds_own = own_here && (last_tile - tile_begin) % WAVES == wave;
  if constexpr (PREP) {
    if (prepares) {
      prepare(qf);
      if (col < group)
#pragma unroll
        for (int c = 0; c < DS; ++c) *(bf16x8*)&lds.queries[col][c * 32 + g * 8] = qf[c];
      bool has_key = key_column;
      if (own_here && group == 16) {
#pragma unroll
        for (int c = 0; c < DS; ++c) qf[c] = *(const bf16x8*)(q_row + (int64_t)(nq + kvh) * D + c * 32 + g * 8);
        if (normed) weights.fetch(prep.k_weight, prep.weight_is_f32, g);
        prepare(qf);
        has_key = col == 0;
      }
      if (own_here) {
        if (has_key)
#pragma unroll
          for (int c = 0; c < DS; ++c) *(bf16x8*)&own_k[c * 32 + g * 8] = qf[c];
#pragma unroll
        for (int n = 0; n < (D + WAVE - 1) / WAVE; ++n)
          if (lane + n * WAVE < D) own_v[lane + n * WAVE] = raw_v[n];
      }
    }
    __syncthreads();
    if (prepares && own_here) {
      const int64_t page = page_ids[pos / page_size - first_block];
      const int off = pos % page_size;
      if (page >= 0) {
        bf16* kdst = k_pages + ((page * nkv + kvh) * page_size + off) * D;
        bf16* vdst = v_pages + (page * nkv + kvh) * (int64_t)D * page_size + off;
        if (lane < D / 8) *(bf16x8*)(kdst + lane * 8) = *(const bf16x8*)&own_k[lane * 8];
#pragma unroll
        for (int n = 0; n < (D + WAVE - 1) / WAVE; ++n)
          if (lane + n * WAVE < D) vdst[(int64_t)(lane + n * WAVE) * page_size] = raw_v[n];
      }
    }
#pragma unroll
    for (int c = 0; c < DS; ++c) qf[c] = *(const bf16x8*)&lds.queries[col < group ? col : 0][c * 32 + g * 8];
  }
#pragma unroll
  for (int c = 0; c < DS; ++c) qf[c] = col < group ? qf[c] : zero8;

  floatx4 o[DB];
#pragma unroll
  for (int b = 0; b < DB; ++b) o[b] = floatx4{0.f, 0.f, 0.f, 0.f};
  float run_max = -INFINITY, run_sum = 0.f;
  const float scale2 = scale * 1.4426950408889634f;
  // the column's head's bias by distance, in the base-2 units of the scores below
  const int biased = kvh * group + (col < group ? col : 0);
  const bool linear = MORE && distance_form == DISTANCE_LINEAR;
  const float rate2 = distance ? distance[biased] * (linear ? LOG2E : 1.f) : 0.f, reach = distance && !linear ? distance[nq + biased] : 0.f;

  // END: the wave's last tile, which may hold the token's own position or reach behind it (the others cannot: less code)
  auto work = [&](auto END, int tile, bf16x8 (&kf)[2][DS], bf16x8 (&vf)[DB]) {
    constexpr bool end = decltype(END)::value;
    const bool cut = tile * 32 < lo || (end && tile * 32 + 31 > pos);
    if (cut) {
      const int key8 = tile * 32 + g * 8;
      const bool seen = key8 <= pos && key8 + 7 >= lo;
#pragma unroll
      for (int b = 0; b < DB; ++b) vf[b] = seen ? vf[b] : zero8;
    }
    if (end && holds_own && tile == last_tile) {
      // the token's own key and value take the place of what the pages hold at its position
      const int own = pos % 32;
      const int own_h = (own % 8) / 4, own_col = (own / 8) * 4 + own % 4, own_g = own / 8, own_j = own % 8;
#pragma unroll
      for (int h = 0; h < 2; ++h)
#pragma unroll
        for (int c = 0; c < DS; ++c)
          if (h == own_h && col == own_col) kf[h][c] = *(const bf16x8*)&own_k[c * 32 + g * 8];
#pragma unroll
      for (int b = 0; b < DB; ++b) {
        const bf16 vn = own_v[b * 16 + col];
#pragma unroll
        for (int j = 0; j < 8; ++j)
          if (g == own_g && j == own_j) vf[b][j] = vn;
      }
    }
    floatx4 s[2];
#pragma unroll
    for (int h = 0; h < 2; ++h) {
      s[h] = floatx4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
      for (int c = 0; c < DS; ++c) s[h] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(kf[h][c], qf[c], s[h], 0, 0, 0);
    }
#pragma unroll
    for (int h = 0; h < 2; ++h)
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        const int key = tile * 32 + g * 8 + h * 4 + i;
        float scaled = softcap > 0.f ? capped(s[h][i] * scale, softcap) * LOG2E : s[h][i] * scale2;
        if (distance) scaled -= linear ? rate2 * (float)(pos - key) : distance_loss(rate2, reach, (float)(pos - key));
        s[h][i] = scaled;
      }
    if (cut) {
#pragma unroll
      for (int h = 0; h < 2; ++h)
#pragma unroll
        for (int i = 0; i < 4; ++i) {
          const int key = tile * 32 + g * 8 + h * 4 + i;
          s[h][i] = key <= pos && key >= lo ? s[h][i] : -INFINITY;
        }
    }
    float tile_max = -INFINITY;
#pragma unroll
    for (int h = 0; h < 2; ++h)
#pragma unroll
      for (int i = 0; i < 4; ++i) tile_max = fmaxf(tile_max, s[h][i]);
    tile_max = fmaxf(tile_max, __shfl_xor(tile_max, 16, WAVE));
    tile_max = fmaxf(tile_max, __shfl_xor(tile_max, 32, WAVE));
    const float new_max = tile_max > run_max + RESCALE_STEP ? tile_max : run_max;   // see RESCALE_STEP
    const float alpha = fast_exp2(run_max - new_max);
    run_max = new_max;
    bf16x8 pf;
    float tile_sum = 0.f;
#pragma unroll
    for (int h = 0; h < 2; ++h)
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        const float p = fast_exp2(s[h][i] - new_max);
        tile_sum += p;
        pf[h * 4 + i] = (bf16)p;
      }
    run_sum = run_sum * alpha + tile_sum;
    const bool rescale = __any(alpha != 1.f);
#pragma unroll
    for (int b = 0; b < DB; ++b) {
      if (rescale) o[b] *= alpha;
      o[b] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(vf[b], pf, o[b], 0, 0, 0);
    }
  };
  if constexpr (AHEAD) {
    // two register sets in turn: the next tile of this wave is on its way while this one is worked on
    bf16x8 (&kf_first)[2][DS] = (bf16x8(&)[2][DS])kf_a;
    bf16x8 (&vf_first)[DB] = (bf16x8(&)[DB])vf_a;
    bf16x8 kf_b[2][DS], vf_b[DB];
    // (no fetch that may or may not be made before a use, see above: the last two tiles stand by themselves)
    int tile = tile_begin + wave;
    for (; tile + 2 * WAVES < tile_end; tile += 2 * WAVES) {
      fetch(tile + WAVES, kf_b, vf_b);
      work(Inner{}, tile, kf_first, vf_first);
      fetch(tile + 2 * WAVES, kf_first, vf_first);
      work(Inner{}, tile + WAVES, kf_b, vf_b);
    }
    if (tile + WAVES < tile_end) {
      fetch(tile + WAVES, kf_b, vf_b);
      work(Inner{}, tile, kf_first, vf_first);
      work(End{}, tile + WAVES, kf_b, vf_b);
    } else if (tile < tile_end) {
      work(End{}, tile, kf_first, vf_first);
    }
  } else {
    for (int tile = tile_begin + wave; tile < tile_end; tile += WAVES) {
      bf16x8 kf[2][DS], vf[DB];
      fetch(tile, kf, vf);
      work(End{}, tile, kf, vf);
    }
  }
  run_sum += __shfl_xor(run_sum, 16, WAVE);
  run_sum += __shfl_xor(run_sum, 32, WAVE);
  if (g == 0) {
    sm_m[wave][col] = run_max;
    sm_l[wave][col] = run_sum;
  }
  if (col < group) {
#pragma unroll
    for (int b = 0; b < DB; ++b) *(floatx4*)&sm_o[wave][col][b * 16 + g * 4] = o[b];
  }
  __syncthreads();
  for (int e = tid; e < dv * group; e += THREADS) {
    const int h = e / dv, dim = e % dv;
    float top = sm_m[0][h];
#pragma unroll
    for (int w = 1; w < WAVES; ++w) top = fmaxf(top, sm_m[w][h]);
    float acc = 0.f, total = 0.f;
#pragma unroll
    for (int w = 0; w < WAVES; ++w) {
      const float weight = top == -INFINITY ? 0.f : fast_exp2(sm_m[w][h] - top);
      acc += sm_o[w][h][dim] * weight;
      total += sm_l[w][h] * weight;
    }
    const int head = kvh * group + h;
    if (slots <= 1) {
      if (sinks) acc *= with_sink(sinks[head] * LOG2E, top, total);
      out[(int64_t)token * out_stride + (int64_t)head * dv + dim] = (bf16)(acc / total * head_gate(gates, gate_stride, token, head));
    } else {
      const int64_t slot = ((int64_t)token * nq + head) * slots + split;
      part_o[slot * dv + dim] = acc;
      if (dim == 0) {
        part_ml[slot * 2] = top;
        part_ml[slot * 2 + 1] = total;
      }
    }
  }
}

template <int D, bool PREP, int WAVES, bool AHEAD, bool MORE, bool ONCE = false>
__global__ __launch_bounds__(WAVES * 64, WAVES == 4 && D == 128 ? 2 : 1) void attention_decode_bf16_kernel(
    const int* __restrict__ positions, const int* __restrict__ token_request, const int* __restrict__ block_table, const bf16* __restrict__ q,
    int table_stride, int q_stride, int nq, int nkv, int page_size, int splits, bf16* __restrict__ out, int out_stride,
    float* __restrict__ part_o, float* __restrict__ part_ml, bf16* __restrict__ k_pages, bf16* __restrict__ v_pages, float scale, int window,
    int slots, DecodePrep prep, const float* __restrict__ sinks, float softcap, const bf16* __restrict__ gates, int gate_stride, int dv_given,
    const float* __restrict__ distance_given, int distance_form) {
  // What leads to the first keys comes first: fourteen words of the arguments are in registers when a wave begins (the file is
  // compiled so), the others are a trip to memory away.
  __shared__ DecodeLds<D, WAVES> lds;
  extern __shared__ int page_ids[];
  attention_decode_part<D, PREP, WAVES, AHEAD, MORE, ONCE>(lds, page_ids, blockIdx.x, blockIdx.y, blockIdx.z, out, out_stride, part_o, part_ml, q, q_stride, k_pages, v_pages, block_table, table_stride, token_request, positions, nq, nkv, page_size, scale, window, splits, slots, prep, sinks, softcap, gates, gate_stride, dv_given, distance_given, distance_form);
}

// Merges the partial results of the splits of one (token, head): out = sum_s o_s 2^(m_s - m) / sum_s l_s 2^(m_s - m).
// A kernel of its own on purpose: letting the last workgroup to finish merge inside the decode
// kernel needs a device-wide fence in every workgroup, and on this chip (eight L2s) those fences
// write back and invalidate whole caches; measured, they cost many times what this kernel does.
__global__ void attention_merge_kernel(bf16* __restrict__ out, int out_stride, const float* __restrict__ part_o,
                                       const float* __restrict__ part_ml, int nq, int d, int splits,
                                       const float* __restrict__ sinks, const bf16* __restrict__ gates, int gate_stride) {
  const int token = blockIdx.x, head = blockIdx.y;
  const int64_t base = ((int64_t)token * nq + head) * splits;
  // Everything is asked for before anything is used: the partial sums of a split do not wait for its maximum
  // (a split that saw no key holds zeros and gets the weight zero), so the kernel is one trip to memory long.
  constexpr int AT_ONCE = 8;
  for (int dim = threadIdx.x; dim < d; dim += blockDim.x) {
    float top = -INFINITY, total = 0.f, acc = 0.f;
    for (int s0 = 0; s0 < splits; s0 += AT_ONCE) {
      float m[AT_ONCE], l[AT_ONCE], o[AT_ONCE];
#pragma unroll
      for (int i = 0; i < AT_ONCE; ++i) {
        const int s = s0 + i < splits ? s0 + i : splits - 1;
        m[i] = part_ml[(base + s) * 2];
        l[i] = part_ml[(base + s) * 2 + 1];
        o[i] = part_o[(base + s) * d + dim];
      }
      float chunk_top = top;
#pragma unroll
      for (int i = 0; i < AT_ONCE; ++i)
        if (s0 + i < splits) chunk_top = fmaxf(chunk_top, m[i]);
      const float keep = top == -INFINITY ? 0.f : fast_exp2(top - chunk_top);   // what was added up so far, against the new maximum
      total *= keep;
      acc *= keep;
      top = chunk_top;
#pragma unroll
      for (int i = 0; i < AT_ONCE; ++i) {
        const float weight = (s0 + i < splits && m[i] > -INFINITY) ? fast_exp2(m[i] - top) : 0.f;
        total += l[i] * weight;
        acc += o[i] * weight;
      }
    }
    if (sinks) acc *= with_sink(sinks[head] * LOG2E, top, total);
    out[(int64_t)token * out_stride + (int64_t)head * d + dim] = (bf16)(acc / total * head_gate(gates, gate_stride, token, head));
  }
}

// The same merge for steps of many tokens (prompt portions whose keys were divided): a thread owns four dims of one
// (token, head) and asks for everything it needs at once, 16 bytes a load; workgroups of four waves over all of them,
// where a workgroup a (token, head) would be tens of thousands of workgroups of two waves with a few loads each.  The
// sums are added in split order, as attention_merge_kernel adds them: the same bits.
template <int SPLITS>
__global__ __launch_bounds__(256) void attention_merge_wide_kernel(bf16* __restrict__ out, int out_stride, const float* __restrict__ part_o,
                                                                   const float* __restrict__ part_ml, int64_t quads, int nq, int d,
                                                                   const float* __restrict__ sinks, const bf16* __restrict__ gates, int gate_stride) {
  const int64_t e = (int64_t)blockIdx.x * 256 + threadIdx.x;
  if (e >= quads) return;
  const int per_head = d / 4;
  const int64_t pair = e / per_head;                 // token * nq + head
  const int dim = (int)(e % per_head) * 4;
  const int64_t base = pair * SPLITS;
  float m[SPLITS], l[SPLITS];
  floatx4 o[SPLITS];
#pragma unroll
  for (int s = 0; s < SPLITS; ++s) {
    const float2 ml = *(const float2*)(part_ml + (base + s) * 2);
    m[s] = ml.x;
    l[s] = ml.y;
    o[s] = *(const floatx4*)(part_o + (base + s) * d + dim);
  }
  float top = -INFINITY;
#pragma unroll
  for (int s = 0; s < SPLITS; ++s) top = fmaxf(top, m[s]);
  float total = 0.f;
  floatx4 acc = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
  for (int s = 0; s < SPLITS; ++s) {
    const float weight = m[s] > -INFINITY ? fast_exp2(m[s] - top) : 0.f;
    total += l[s] * weight;
#pragma unroll
    for (int i = 0; i < 4; ++i) acc[i] += o[s][i] * weight;
  }
  const int64_t token = pair / nq, head = pair % nq;
  if (sinks) {
    const float keep = with_sink(sinks[head] * LOG2E, top, total);
#pragma unroll
    for (int i = 0; i < 4; ++i) acc[i] *= keep;
  }
  bf16x4 r;
  const float gate = head_gate(gates, gate_stride, token, (int)head);
#pragma unroll
  for (int i = 0; i < 4; ++i) r[i] = (bf16)(acc[i] / total * gate);
  *(bf16x4*)(out + token * out_stride + head * d + dim) = r;
}

static void launch_attention_merge(bf16* out, int out_stride, const float* part_o, const float* part_ml, int tokens, int nq, int d,
                                   int splits, const float* sinks, const bf16* gates, int gate_stride, hipStream_t s) {
  const bool wide = tokens >= 64 && d % 4 == 0 && out_stride % 4 == 0 && (uintptr_t)out % 8 == 0 && (uintptr_t)part_o % 16 == 0 &&
                    (uintptr_t)part_ml % 8 == 0 && (splits == 2 || splits == 3 || splits == 4 || splits == 5 || splits == 8 || splits == 9);
  if (wide) {
    const int64_t quads = (int64_t)tokens * nq * (d / 4);
    const int blocks = (int)((quads + 255) / 256);
    if (splits == 2) attention_merge_wide_kernel<2><<<blocks, 256, 0, s>>>(out, out_stride, part_o, part_ml, quads, nq, d, sinks, gates, gate_stride);
    else if (splits == 3) attention_merge_wide_kernel<3><<<blocks, 256, 0, s>>>(out, out_stride, part_o, part_ml, quads, nq, d, sinks, gates, gate_stride);
    else if (splits == 4) attention_merge_wide_kernel<4><<<blocks, 256, 0, s>>>(out, out_stride, part_o, part_ml, quads, nq, d, sinks, gates, gate_stride);
    else if (splits == 5) attention_merge_wide_kernel<5><<<blocks, 256, 0, s>>>(out, out_stride, part_o, part_ml, quads, nq, d, sinks, gates, gate_stride);
    else if (splits == 9) attention_merge_wide_kernel<9><<<blocks, 256, 0, s>>>(out, out_stride, part_o, part_ml, quads, nq, d, sinks, gates, gate_stride);
    else attention_merge_wide_kernel<8><<<blocks, 256, 0, s>>>(out, out_stride, part_o, part_ml, quads, nq, d, sinks, gates, gate_stride);
  } else {
    attention_merge_kernel<<<dim3(tokens, nq), d < 64 ? 64 : d, 0, s>>>(out, out_stride, part_o, part_ml, nq, d, splits, sinks, gates, gate_stride);
  }
}

// The share of a sequence's kept first positions in a windowed attention: for every (token, head) the keys at positions
// below min(keep_first, lo), lo = pos - window + 1 being the window's first position (none while the window still reaches
// the start), as one more partial result beside those of the window's splits: unnormalised sums against a maximum, in the
// form attention_merge_kernel adds up (slot `slots - 1` of part_o [tokens, nq, slots, d] and part_ml [tokens, nq, slots, 2]).
// A wave per (token, head), a lane for every 64th dim; the kept keys are few, and every one is a row of d values.
__global__ __launch_bounds__(WAVE) void attention_kept_bf16_kernel(
    const bf16* __restrict__ q, int q_stride, const bf16* __restrict__ k_pages, const bf16* __restrict__ v_pages,
    const int* __restrict__ block_table, int table_stride, const int* __restrict__ token_request,
    const int* __restrict__ positions, int nq, int nkv, int d, int page_size, float scale, int window, int keep_first,
    int slots, float* __restrict__ part_o, float* __restrict__ part_ml, float softcap, int dv, const float* __restrict__ distance,
    int distance_form) {
  constexpr int PER_LANE = 4;                                     // heads of up to 256 dims
  const int token = blockIdx.x, head = blockIdx.y, lane = threadIdx.x;
  const int kvh = head / (nq / nkv);
  const int pos = positions[token];
  const int lo = pos - window + 1;
  const int kept = lo > 0 ? (keep_first < lo ? keep_first : lo) : 0;
  const int64_t slot = ((int64_t)token * nq + head) * slots + (slots - 1);
  const float scale2 = scale * 1.4426950408889634f;
  const int* table = block_table + (int64_t)token_request[token] * table_stride;
  float qv[PER_LANE], acc[PER_LANE];
#pragma unroll
  for (int n = 0; n < PER_LANE; ++n) {
    const int dim = lane + n * WAVE;
    qv[n] = dim < d ? (float)q[(int64_t)token * q_stride + (int64_t)head * d + dim] : 0.f;
    acc[n] = 0.f;
  }
  float top = -INFINITY, total = 0.f;
  for (int key = 0; key < kept; ++key) {
    const int64_t page = table[key / page_size];
    const int off = key % page_size;
    const bf16* kp = k_pages + ((page * nkv + kvh) * page_size + off) * (int64_t)d;
    const bf16* vp = v_pages + (page * nkv + kvh) * (int64_t)dv * page_size + off;
    float dot = 0.f, vv[PER_LANE];
#pragma unroll
    for (int n = 0; n < PER_LANE; ++n) {
      const int dim = lane + n * WAVE;
      dot += dim < d ? qv[n] * (float)kp[dim] : 0.f;
      vv[n] = dim < dv ? (float)vp[(int64_t)dim * page_size] : 0.f;
    }
#pragma unroll
    for (int step = 1; step < WAVE; step *= 2) dot += __shfl_xor(dot, step, WAVE);
    float score = softcap > 0.f ? capped(dot * scale, softcap) * LOG2E : dot * scale2;
    if (distance) score -= distance_loss_of(distance, distance_form, nq, head, (float)(pos - key));
    const float new_top = fmaxf(top, score);
    const float keep = top == -INFINITY ? 0.f : fast_exp2(top - new_top);
    const float weight = fast_exp2(score - new_top);
    total = total * keep + weight;
#pragma unroll
    for (int n = 0; n < PER_LANE; ++n) acc[n] = acc[n] * keep + weight * vv[n];
    top = new_top;
  }
#pragma unroll
  for (int n = 0; n < PER_LANE; ++n) {
    const int dim = lane + n * WAVE;
    if (dim < dv) part_o[slot * dv + dim] = acc[n];
  }
  if (lane == 0) {
    part_ml[slot * 2] = top;
    part_ml[slot * 2 + 1] = total;
  }
}

static void launch_attention_kept(const bf16* q, int q_stride, const bf16* k_pages, const bf16* v_pages, const int* block_table,
                                  int table_stride, const int* token_request, const int* positions, int tokens, int nq, int nkv, int d,
                                  int page_size, float scale, int window, int keep_first, int slots, float* part_o, float* part_ml,
                                  float softcap, int dv, const float* distance, int distance_form, hipStream_t s) {
  attention_kept_bf16_kernel<<<dim3(tokens, nq), WAVE, 0, s>>>(q, q_stride, k_pages, v_pages, block_table, table_stride, token_request,
                                                               positions, nq, nkv, d, page_size, scale, window, keep_first, slots, part_o,
                                                               part_ml, softcap, dv, distance, distance_form);
}

// Decode step in bf16: one query token per request.  part_o [tokens, nq, splits, d] and part_ml
// [tokens, nq, splits, 2] float32 are needed when splits > 1; with keep_first (a window's kept first positions, see
// attention_kept_bf16_kernel) they hold one partial result more and are always needed.  Returns an error for shapes the
// matrix-core kernel does not take (the caller then uses lrs_attention).
// prepare != 0: q points at the raw rows [q heads | kv_columns k heads | kv_columns v heads] of the
// q/k/v product and the kernel does the work of lrs_qk_prep as well (rotation over the whole head
// or none; kv_columns is nkv, or 0 for a layer that reads another layer's pages).
LRS_API int lrs_attention_decode(void* out, int out_stride, float* part_o, float* part_ml, const void* q,
                                 int q_stride, void* k_pages, void* v_pages,
                                 const int* block_table, int table_stride, const int* token_request,
                                 const int* positions, int tokens, int max_context, int nq, int nkv, int d,
                                 int page_size, float scale, int window, int keep_first, int splits, int form, int prepare,
                                 const void* q_weight, const void* k_weight, int w_dtype, float eps,
                                 const float* cosv, const float* sinv, int kv_columns, const float* sinks, float softcap,
                                 const void* gates, int gate_stride, int dv, const float* distance, int distance_form, void* stream) {
  LRS_REQUIRE(distance_form == DISTANCE_LOG || distance_form == DISTANCE_LINEAR, "attention_decode: unknown form %d of the bias by distance", distance_form);
  LRS_REQUIRE(dv > 0 && dv % 16 == 0 && dv <= d && (dv == d || !prepare),
              "attention_decode: values of %d dims beside keys of %d are not served (a multiple of 16, at most the keys', heads that come prepared)", dv, d);
  LRS_REQUIRE(tokens > 0 && nq > 0 && nkv > 0 && nq % nkv == 0, "attention_decode: bad sizes tokens=%d nq=%d nkv=%d", tokens, nq, nkv);
  LRS_REQUIRE(nq / nkv <= 16, "attention_decode: %d query heads per kv head, at most 16 fit a tile", nq / nkv);
  LRS_REQUIRE(page_size % 16 == 0, "attention_decode: page size %d is not a multiple of 16", page_size);
  LRS_REQUIRE(keep_first >= 0 && (keep_first == 0 || (window > 0 && !prepare)),
              "attention_decode: kept first positions (%d) need a window and prepared heads", keep_first);
  const int slots = splits + (keep_first > 0 ? 1 : 0);          // the kept keys' share is one more partial result
  LRS_REQUIRE(splits >= 1 && (slots == 1 || (part_o && part_ml)), "attention_decode: %d partial results need their buffers", slots);
  LRS_REQUIRE(form >= 0 && form <= 3, "attention_decode: form must be 0, 1, 2 or 3, got %d", form);
  LRS_REQUIRE(softcap >= 0.f, "attention_decode: the cap on the scores must be positive (0 = none), got %g", (double)softcap);
  LRS_REQUIRE(q_stride % 8 == 0 && ((uintptr_t)q % 16) == 0, "attention_decode: q rows must be 16-byte aligned");
  dim3 grid(splits, nkv, tokens);
  hipStream_t s = (hipStream_t)stream;
  // LDS copy of the block table entries one workgroup walks
  LRS_REQUIRE(max_context >= 1, "attention_decode: max_context must be the longest context length of the step");
  const int reach = window < 0 ? -window : window;
  const int span = reach > 0 && reach + 64 < max_context ? reach + 64 : max_context;
  const size_t table_lds = sizeof(int) * (size_t)((span / 32 + splits) / splits * 32 / page_size + 4);
  LRS_REQUIRE(table_lds <= 24 * 1024, "attention_decode: a context of %d tokens in %d splits needs more block table entries than fit LDS", max_context, splits);
  if (prepare) {
    LRS_REQUIRE((q_weight == nullptr) == (k_weight == nullptr), "attention_decode: q and k norm weights must come together");
    LRS_REQUIRE(q_weight == nullptr || eps > 0.f, "attention_decode: eps must be positive");
    LRS_REQUIRE((cosv == nullptr) == (sinv == nullptr), "attention_decode: cos and sin tables must come together");
    LRS_REQUIRE(cosv == nullptr || d % 64 == 0, "attention_decode: the kernel rotates heads of 64, 128 or 192 dims only, got %d", d);
    LRS_REQUIRE(kv_columns == 0 || kv_columns == nkv, "attention_decode: kv_columns must be 0 or the number of kv heads (%d), got %d", nkv, kv_columns);
    LRS_REQUIRE(q_stride >= (nq + 2 * kv_columns) * d, "attention_decode: q row stride %d too small for q, k and v heads", q_stride);
    LRS_REQUIRE((uintptr_t)q_weight % 16 == 0 && (uintptr_t)k_weight % 16 == 0 && (uintptr_t)cosv % 16 == 0 && (uintptr_t)sinv % 16 == 0,
                "attention_decode: norm weights and rotation tables must be 16-byte aligned");
  }
  const DecodePrep prep{q_weight, k_weight, w_dtype == LRS_F32, eps, cosv, sinv, kv_columns};
  // `form`: 0 = four waves, a tile at a time; 1 and 3 = four waves, 2 = eight waves, each wave with its next
  // tile on the way while it works (heads of 192 dims have no registers for that and stay with 0); 3 loads keys and values with the
  // streaming hint (load_once), which pays where a step's keys are many and a workgroup's as well: _keys_read_once in parts/attention.py
#define ARGS                                                                                                 \
  positions, token_request, block_table, (const bf16*)q, table_stride, q_stride, nq, nkv, page_size, splits, (bf16*)out, out_stride, part_o, \
      part_ml, (bf16*)k_pages, (bf16*)v_pages, scale, window, slots, prep, slots == 1 ? sinks : nullptr, softcap, \
      slots == 1 ? (const bf16*)gates : nullptr, gate_stride, dv, distance, distance_form
#define LAUNCH_PREP(D, PREP, MORE)                                                                           \
  do {                                                                                                       \
    if (form == 2 && D <= 128) attention_decode_bf16_kernel<D, PREP, 8, (D <= 128), MORE><<<grid, 512, table_lds, s>>>(ARGS); \
    else if (form == 3 && D <= 128) attention_decode_bf16_kernel<D, PREP, 4, (D <= 128), MORE, (D <= 128)><<<grid, 256, table_lds, s>>>(ARGS); \
    else if (form == 1 && D <= 128) attention_decode_bf16_kernel<D, PREP, 4, (D <= 128), MORE><<<grid, 256, table_lds, s>>>(ARGS); \
    else attention_decode_bf16_kernel<D, PREP, 4, false, MORE><<<grid, 256, table_lds, s>>>(ARGS);             \
  } while (0)
#define LAUNCH(D)                        \
  do {                                   \
    if (prepare && distance) LAUNCH_PREP(D, true, true);            \
    else if (prepare) LAUNCH_PREP(D, true, false);                  \
    else if (dv != d || distance) LAUNCH_PREP(D, false, true);      \
    else LAUNCH_PREP(D, false, false);                              \
  } while (0)
  switch (d) {
    case 32: LAUNCH(32); break;
    case 64: LAUNCH(64); break;
    case 96: LAUNCH(96); break;
    case 128: LAUNCH(128); break;
    case 192: LAUNCH(192); break;
    default: return lrs_fail("attention_decode: head_dim %d has no matrix-core kernel (32, 64, 96, 128, 192)", d);
  }
#undef LAUNCH
#undef LAUNCH_PREP
#undef ARGS
  if (lrs_check_launch("attention_decode")) return 1;
  if (keep_first > 0) {
    launch_attention_kept((const bf16*)q, q_stride, (const bf16*)k_pages, (const bf16*)v_pages, block_table, table_stride, token_request,
                          positions, tokens, nq, nkv, d, page_size, scale, window, keep_first, slots, part_o, part_ml, softcap, dv, distance, distance_form, s);
    if (lrs_check_launch("attention_kept")) return 1;
  }
  if (slots > 1) {
    launch_attention_merge((bf16*)out, out_stride, part_o, part_ml, tokens, nq, dv, slots, sinks, (const bf16*)gates, gate_stride, s);
    return lrs_check_launch("attention_merge");
  }
  return 0;
}

// ------------------------------------------------- bf16 kernel for any step
// Ragged batch of prompt portions and single tokens.  The step's tokens are cut on the host into
// groups of at most 16*QB consecutive tokens of one request; a workgroup owns one (group, kv head)
// and each of its (up to four) waves one query head of the kv group.  Keys are walked in tiles of
// 32: the workgroup brings a tile's keys and (transposed) values into LDS once, all waves take
// their matrix-core operands from there, and the next tile is on its way from memory while the
// current one is worked on (two LDS buffers, one barrier a tile).  A wave holds QB blocks of 16
// queries, so every fragment it reads serves QB products.  The arithmetic is that of the decode
// kernel with 16 queries in the tile columns instead of the heads: S[key, query] = K Q^T, online
// softmax per query column with the causal (and window) mask of that query's position,
// O^T[dim, query] += V^T P.  Every query is finished by one wave, so nothing is merged.
// Two workgroups share a compute unit (at most 256 registers a lane, which also keeps the
// accumulators out of the AGPRs, where rescaling them would cost moves at every tile), so one
// wave's exponentials run beside another's matrix products.  The grid is one-dimensional: groups
// come longest first, and in every second chunk of `chunk` workgroups (one per compute unit) the
// order is turned round, so that the two workgroups that meet on a compute unit are a long and a
// short one; the kv head changes fastest, which keeps one kv head's keys in one XCD's L2.
// splits > 1 (few queries over long contexts): the key tiles of every group are divided between
// `splits` workgroups, which leave unnormalised sums, maxima and weights in part_o / part_ml
// [tokens, heads, splits, ...] for attention_merge_kernel, as the decode kernel does.
// LINEAR: the linear bias by distance, as instances of their own so that the others keep their registers.
template <int D, int QB, bool LINEAR>
__global__ __launch_bounds__(256, D <= 128 ? 2 : 1) void attention_prefill_bf16_kernel(
    bf16* __restrict__ out, int out_stride, const bf16* __restrict__ q, int q_stride,
    const bf16* __restrict__ k_pages, const bf16* __restrict__ v_pages,
    const int* __restrict__ block_table, int table_stride, const int* __restrict__ token_request,
    const int* __restrict__ positions, const int* __restrict__ qblock_token0,
    const int* __restrict__ qblock_count, int n_blocks, int chunk, int nq, int nkv, int page_size, float scale,
    int window, int splits, int slots, float* __restrict__ part_o, float* __restrict__ part_ml,
    const float* __restrict__ sinks, float softcap, const bf16* __restrict__ gates, int gate_stride, int dv,
    const float* __restrict__ distance) {
  constexpr int DS = D / 32, DB = D / 16;
  // Padded LDS rows.  Every fragment is read 16 bytes a lane, 16 rows at a time (the lane's row is col, its
  // piece g), which the LDS serves at its full 256 bytes a cycle when rows lie 32 bytes more than a multiple
  // of 64 apart, and at half of that, or worse, otherwise (measured for every stride; 8-byte reads reach
  // half at best).  Key rows are D elements long; a row of the transposed value tile holds a dimension's 32
  // keys in the order the second product wants them, so that a lane's eight are one 16-byte piece: position
  // g * 8 + h * 4 + i for key h * 16 + g * 4 + i, which is where the first product leaves that key's weight.
  constexpr int KLD = D + 16, VLD = 32 + 16;
  __shared__ __attribute__((aligned(16))) bf16 ks[2][32 * KLD];
  __shared__ __attribute__((aligned(16))) bf16 vs[2][D * VLD];
  const int tid = threadIdx.x, threads = blockDim.x;
  const int lane = tid % WAVE, wave = tid / WAVE, waves = threads / WAVE;
  const int col = lane & 15, g = lane >> 4;
  const int group = nq / nkv;
  const int work = blockIdx.x % (n_blocks * nkv), split = blockIdx.x / (n_blocks * nkv);
  const int which_chunk = work / chunk, in_chunk = work % chunk;
  const int chunk_block0 = which_chunk * (chunk / nkv);
  const int chunk_blocks = n_blocks - chunk_block0 < chunk / nkv ? n_blocks - chunk_block0 : chunk / nkv;
  const int kvh = in_chunk % nkv;
  const int qblock = chunk_block0 + ((which_chunk & 1) ? chunk_blocks - 1 - in_chunk / nkv : in_chunk / nkv);
  const int token0 = qblock_token0[qblock], count = qblock_count[qblock];
  const int pos_first = positions[token0], pos_last = positions[token0 + count - 1];
  const int lo_first = first_seen(pos_first, window);
  const int lo_last = first_seen(pos_last, window);
  const int* table = block_table + (int64_t)token_request[token0] * table_stride;
  const bf16x8 zero8 = {0, 0, 0, 0, 0, 0, 0, 0};
  const float scale2 = scale * 1.4426950408889634f;
  const float rescale_step = RESCALE_STEP / scale2;              // in units of the unscaled scores
  int first_tile = lo_first / 32, last_tile = pos_last / 32;
  if (splits > 1) {                                              // this workgroup's share of the tiles (may be none)
    const int per_split = (last_tile - first_tile + splits) / splits;
    first_tile += split * per_split;
    if (first_tile + per_split - 1 < last_tile) last_tile = first_tile + per_split - 1;
  }
  // the part of the request's block table that the tiles need, in LDS: the address of a key must
  // not wait for a trip to memory of its own
  extern __shared__ int page_ids[];
  const int last_key = last_tile * 32 + 31 < pos_last ? last_tile * 32 + 31 : pos_last;
  {
    const int first = first_tile * 32 / page_size;
    if (first_tile <= last_tile)
      for (int i = tid; i <= last_key / page_size - first; i += threads) page_ids[i] = table[first + i];
  }
  __syncthreads();

  // Pieces of a tile this thread brings in: keys [32, D] and transposed values [D, 32].  A run of 16 keys
  // lies in one page, and a wave serves one run (waves 0 and 1 the tile's first, 2 and 3 its second), so
  // everything about the run's place in memory is the same for the whole wave and is worked out in
  // scalar registers: one block table entry, one base address; a lane adds a distance that never changes.
  constexpr int KPIECES = D / 8, RUN_CHUNKS = 16 * KPIECES, TPR = 128, KPT = (RUN_CHUNKS + TPR - 1) / TPR;
  constexpr int VRUN_CHUNKS = 2 * D, VPT = (VRUN_CHUNKS + TPR - 1) / TPR;
  bf16x8 kreg_a[KPT], vreg_a[VPT];
  const int wrun = __builtin_amdgcn_readfirstlane(tid / TPR), t1 = tid % TPR;
  const int pages16 = page_size / 16;                            // runs of 16 keys in a page
  const unsigned magic = pages16 > 1 ? 0xFFFFFFFFu / (unsigned)pages16 + 1u : 0u;   // run / pages16 = umulhi(run, magic)
  const int first_block = pages16 > 1 ? (int)__umulhi((unsigned)(first_tile * 2), magic) : first_tile * 2;
  unsigned koff[KPT], voff[VPT];
#pragma unroll
  for (int i = 0; i < KPT; ++i) koff[i] = (unsigned)(((t1 + i * TPR) / KPIECES) * D + ((t1 + i * TPR) % KPIECES) * 8);
#pragma unroll
  for (int i = 0; i < VPT; ++i) {                                 // (values narrower than keys: the dims behind them repeat the last one)
    const int dim = (t1 + i * TPR) / 2 < dv ? (t1 + i * TPR) / 2 : dv - 1;
    voff[i] = (unsigned)(dim * page_size + ((t1 + i * TPR) % 2) * 8);
  }
  auto fetch = [&](int tile, bf16x8 (&kreg)[KPT], bf16x8 (&vreg)[VPT]) {
    const int run = tile * 2 + wrun, key0 = run * 16;
    const bool present = key0 <= pos_last && key0 + 15 >= lo_first;
    if (present) {
      const int block = pages16 > 1 ? (int)__umulhi((unsigned)run, magic) : run;
      const int64_t page = __builtin_amdgcn_readfirstlane(page_ids[block - first_block]);
      const int off = (run - block * pages16) * 16;
      const bf16* kbase = k_pages + ((page * nkv + kvh) * page_size + off) * D;
      const bf16* vbase = v_pages + (page * nkv + kvh) * (int64_t)dv * page_size + off;
#pragma unroll
      for (int i = 0; i < KPT; ++i) kreg[i] = t1 + i * TPR < RUN_CHUNKS ? *(const bf16x8*)(kbase + koff[i]) : zero8;
#pragma unroll
      for (int i = 0; i < VPT; ++i) vreg[i] = t1 + i * TPR < VRUN_CHUNKS ? *(const bf16x8*)(vbase + voff[i]) : zero8;
    } else {
#pragma unroll
      for (int i = 0; i < KPT; ++i) kreg[i] = zero8;
#pragma unroll
      for (int i = 0; i < VPT; ++i) vreg[i] = zero8;
    }
  };
  auto stash = [&](int buffer, const bf16x8 (&kreg)[KPT], const bf16x8 (&vreg)[VPT]) {
#pragma unroll
    for (int i = 0; i < KPT; ++i) {
      const int c = t1 + i * TPR;
      if (c < RUN_CHUNKS) *(bf16x8*)(ks[buffer] + (wrun * 16 + c / KPIECES) * KLD + (c % KPIECES) * 8) = kreg[i];
    }
#pragma unroll
    for (int i = 0; i < VPT; ++i) {
      const int c = t1 + i * TPR;
      if (c < VRUN_CHUNKS) {
        // keys wrun * 16 + (c % 2) * 8 + 0..7 of dimension c / 2: h = wrun, g = (c % 2) * 2 and the next
        bf16* dst = vs[buffer] + (c / 2) * VLD + (c % 2) * 16 + wrun * 4;
        *(bf16x4*)dst = bf16x4{vreg[i][0], vreg[i][1], vreg[i][2], vreg[i][3]};
        *(bf16x4*)(dst + 8) = bf16x4{vreg[i][4], vreg[i][5], vreg[i][6], vreg[i][7]};
      }
    }
  };

  // kv groups of more than four heads take several passes over the keys
  for (int head0 = kvh * group; head0 < (kvh + 1) * group; head0 += waves) {
    const int head = head0 + wave;
    const bool active = head < (kvh + 1) * group;
    bf16x8 qf[QB][DS];
    floatx4 o[QB][DB];
    float run_max[QB], run_sum[QB];
    int pos[QB], lo[QB];
    bool live[QB];
#pragma unroll
    for (int b = 0; b < QB; ++b) {
      live[b] = active && b * 16 + col < count;
      const int token = token0 + (live[b] ? b * 16 + col : 0);
      pos[b] = live[b] ? positions[token] : -1;                // a dead column sees no key
      lo[b] = first_seen(pos[b], window);
      run_max[b] = -INFINITY;
      run_sum[b] = 0.f;
#pragma unroll
      for (int c = 0; c < DS; ++c)
        qf[b][c] = live[b] ? *(const bf16x8*)(q + (int64_t)token * q_stride + (int64_t)head * D + c * 32 + g * 8) : zero8;
#pragma unroll
      for (int e = 0; e < DB; ++e) o[b][e] = floatx4{0.f, 0.f, 0.f, 0.f};
    }

    // the head's bias by distance, in units of the unscaled scores
    const int biased = active ? head : head0;
    const float rate = distance ? distance[biased] * (LINEAR ? 1.f : LN2) / scale : 0.f, reach = !LINEAR && distance ? distance[nq + biased] : 0.f;
    // The linear form in two parts: what depends on a key's place in its tile is what the tile's products are added to (the same for
    // every tile), and what is the same for all of a query's keys in the tile joins the exponents' shift.  With a cap on the scores,
    // or two blocks of queries (whose registers are all in use), it is taken off whole.
    const bool in_parts = LINEAR && QB == 1 && !(softcap > 0.f);
    floatx4 in_tile[2] = {{0.f, 0.f, 0.f, 0.f}, {0.f, 0.f, 0.f, 0.f}};
    if constexpr (LINEAR && QB == 1) {
#pragma unroll
      for (int h = 0; h < 2; ++h)
#pragma unroll
        for (int i = 0; i < 4; ++i) in_tile[h][i] = in_parts ? rate * (float)(h * 16 + g * 4 + i) : 0.f;
    }
    auto of_tile = [&](int tile, int b) { return in_parts ? -rate * (float)((live[b] ? pos[b] : pos_last) - tile * 32) : 0.f; };
    bool grown = false;                                        // the weights have left the reference points behind
    auto raise_reference = [&]() {
#pragma unroll
      for (int b = 0; b < QB; ++b) {
        const float more = growth_of(run_sum[b]), shrink = fast_exp2(-more);
        run_max[b] += more / scale2;
        run_sum[b] *= shrink;
#pragma unroll
        for (int e = 0; e < DB; ++e) o[b][e] *= shrink;
      }
      grown = false;
    };
    // The three parts of a tile's work.
    // scores: S[key, query] = K Q^T, unscaled (the scale enters with the exponent).
    auto scores = [&](int tile, int buffer, floatx4 (&sc)[QB][2]) {
      const bf16* kt = ks[buffer];
#pragma unroll
      for (int b = 0; b < QB; ++b)
#pragma unroll
        for (int h = 0; h < 2; ++h) sc[b][h] = in_tile[h];
#pragma unroll
      for (int h = 0; h < 2; ++h)
#pragma unroll
        for (int c = 0; c < DS; ++c) {
          const bf16x8 kfrag = *(const bf16x8*)(kt + (h * 16 + col) * KLD + c * 32 + g * 8);
#pragma unroll
          for (int b = 0; b < QB; ++b) sc[b][h] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(kfrag, qf[b][c], sc[b][h], 0, 0, 0);
        }
      if (softcap > 0.f) {       // the cap, in units of the unscaled scores (the scale enters with the exponent)
        const float cap = softcap / scale;
#pragma unroll
        for (int b = 0; b < QB; ++b)
#pragma unroll
          for (int h = 0; h < 2; ++h)
#pragma unroll
            for (int i = 0; i < 4; ++i) sc[b][h][i] = capped(sc[b][h][i], cap);
      }
      if (LINEAR && !in_parts) {
#pragma unroll
        for (int b = 0; b < QB; ++b)
#pragma unroll
          for (int h = 0; h < 2; ++h) sc[b][h] += linear_of_four(rate, (float)((live[b] ? pos[b] : pos_last) - (tile * 32 + h * 16 + g * 4)));
      }
      if (!LINEAR && distance) { // (a key ahead of the query gives no number here; the mask takes it out)
#pragma unroll
        for (int b = 0; b < QB; ++b)
#pragma unroll
          for (int h = 0; h < 2; ++h) {
            const float behind = (float)((live[b] ? pos[b] : pos_last) - (tile * 32 + h * 16 + g * 4));
#pragma unroll
            for (int i = 0; i < 4; ++i) sc[b][h][i] -= distance_loss(rate, reach, behind - (float)i);
          }
      }
    };
    // weights: one step of the running softmax, p = 2^(s * scale2 - reference * scale2) as bfloat16 operands.
    // The reference point of a query's exponentials need not be its maximum: any value that keeps the
    // weights inside float32 and bfloat16 gives the same result up to rounding.  So a tile that needs no
    // mask first tries the reference it has, without looking for the tile's maximum at all (`weights`,
    // which changes nothing if it fails); only if a weight sum comes out above 2^60 (or the query has no
    // reference yet) is the tile done the long way (`weights_with_maximum`), which moves the reference to
    // the tile's maximum when that exceeds it by more than 2^8 and rescales the accumulators.  That
    // happens a few times per sequence.
    auto weights_with_maximum = [&](int tile, floatx4 (&sc)[QB][2], auto masked, bf16x8 (&pf)[QB]) {
      constexpr bool MASKED = decltype(masked)::value;
      float alpha[QB];
      bool rescale = false;
#pragma unroll
      for (int b = 0; b < QB; ++b) {
        float tile_max = -INFINITY;
        if (in_parts) {
          const float all = of_tile(tile, b);
          sc[b][0] += all;
          sc[b][1] += all;
        }
#pragma unroll
        for (int h = 0; h < 2; ++h)
#pragma unroll
          for (int i = 0; i < 4; ++i) {
            if (MASKED) {
              const int key = tile * 32 + h * 16 + g * 4 + i;
              sc[b][h][i] = (key <= pos[b] && key >= lo[b]) ? sc[b][h][i] : -INFINITY;
            }
            tile_max = fmaxf(tile_max, sc[b][h][i]);
          }
        tile_max = fmaxf(tile_max, __shfl_xor(tile_max, 16, WAVE));
        tile_max = fmaxf(tile_max, __shfl_xor(tile_max, 32, WAVE));
        const float new_max = tile_max > run_max[b] + rescale_step ? tile_max : run_max[b];
        // a query whose window or position leaves it no key so far keeps its state
        const bool empty = MASKED && new_max == -INFINITY;
        alpha[b] = empty ? 1.f : fast_exp2((run_max[b] - new_max) * scale2);
        const float shift = empty ? 0.f : -new_max * scale2;
        run_max[b] = new_max;
        float tile_sum = 0.f;
#pragma unroll
        for (int h = 0; h < 2; ++h)
#pragma unroll
          for (int i = 0; i < 4; ++i) {
            const float p = fast_exp2(fmaf(sc[b][h][i], scale2, shift));
            tile_sum += p;
            pf[b][h * 4 + i] = (bf16)p;
          }
        run_sum[b] = run_sum[b] * alpha[b] + tile_sum;
        rescale |= alpha[b] != 1.f;
      }
      // once the reference points have settled no column needs rescaling: skip the multiplies
      if (__any(rescale)) {
#pragma unroll
        for (int b = 0; b < QB; ++b)
#pragma unroll
          for (int e = 0; e < DB; ++e) o[b][e] *= alpha[b];
      }
    };
    auto weights = [&](int tile, floatx4 (&sc)[QB][2], bf16x8 (&pf)[QB]) -> bool {
      float sums[QB];
      bool again = false;
#pragma unroll
      for (int b = 0; b < QB; ++b) {
        const float shift = ((LINEAR && QB == 1 ? of_tile(tile, b) : 0.f) - run_max[b]) * scale2;      // +inf before the query's first tile: the sum then says "again"
        float tile_sum = 0.f;
#pragma unroll
        for (int h = 0; h < 2; ++h)
#pragma unroll
          for (int i = 0; i < 4; ++i) {
            const float p = fast_exp2(fmaf(sc[b][h][i], scale2, shift));
            tile_sum += p;
            pf[b][h * 4 + i] = (bf16)p;
          }
        sums[b] = tile_sum;
        again |= !(tile_sum <= 0x1p60f);                         // too large, infinite or not a number
      }
      if (__any(again)) return false;
      bool large = false;
#pragma unroll
      for (int b = 0; b < QB; ++b) {
        run_sum[b] += sums[b];
        if constexpr (LINEAR && QB == 1) large |= sums[b] > GROWN;
      }
      if constexpr (LINEAR && QB == 1) grown = __any(large);
      return true;
    };
    // values: O^T[dim, query] += V^T P
    auto values = [&](int buffer, const bf16x8 (&pf)[QB]) {
      const bf16* vt = vs[buffer];
#pragma unroll
      for (int e = 0; e < DB; ++e) {
        const bf16x8 vv = *(const bf16x8*)(vt + (e * 16 + col) * VLD + g * 8);
#pragma unroll
        for (int b = 0; b < QB; ++b) o[b][e] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(vv, pf[b], o[b][e], 0, 0, 0);
      }
    };

    // Tiles [whole_begin, whole_end) need no mask: every query of the group sees every key of theirs.
    int whole_begin = (lo_last + 31) / 32, whole_end = (pos_first + 1) / 32;
    if (whole_begin < first_tile) whole_begin = first_tile;
    if (whole_begin > last_tile + 1) whole_begin = last_tile + 1;
    if (whole_end > last_tile + 1) whole_end = last_tile + 1;
    if (whole_end < whole_begin) whole_end = whole_begin;

    // The walk over the tiles.  At the top of a turn `tile` is in LDS buffer (tile - first_tile) % 2; the
    // next tile is asked for before the work on this one and put into the other buffer after it.  Most
    // turns take the short way through the weights; the inner loop holds only those, so that nothing in it
    // touches the accumulators but the matrix products.  A tile that needs the mask, or whose weights
    // came out too large for the reference point it was tried with, leaves the inner loop, is finished
    // the long way and the inner loop begins again behind it.
    __syncthreads();                                           // the buffers of an earlier pass are done with
    if (first_tile <= last_tile) {
      fetch(first_tile, kreg_a, vreg_a);
      stash(0, kreg_a, vreg_a);
    }
    __syncthreads();
    floatx4 sc[QB][2];
    bf16x8 pf[QB];
    int tile = first_tile;
    for (;;) {
      bool unfinished = false;
      for (; tile <= last_tile && !(LINEAR && QB == 1 && grown); ++tile) {
        const int buffer = (tile - first_tile) & 1;
        if (tile < last_tile) fetch(tile + 1, kreg_a, vreg_a);
        scores(tile, buffer, sc);
        if (tile < whole_begin || tile >= whole_end || !weights(tile, sc, pf)) {
          unfinished = true;
          break;
        }
        values(buffer, pf);
        if (tile < last_tile) stash(buffer ^ 1, kreg_a, vreg_a);
        __syncthreads();
      }
      if constexpr (LINEAR && QB == 1) {
        if (grown) {
          raise_reference();
          continue;
        }
      }
      if (!unfinished) break;
      const int buffer = (tile - first_tile) & 1;
      if (tile < whole_begin || tile >= whole_end) weights_with_maximum(tile, sc, std::true_type{}, pf);
      else weights_with_maximum(tile, sc, std::false_type{}, pf);
      values(buffer, pf);
      if (tile < last_tile) stash(buffer ^ 1, kreg_a, vreg_a);
      __syncthreads();
      ++tile;
    }
#pragma unroll
    for (int b = 0; b < QB; ++b) {
      float total = run_sum[b];
      total += __shfl_xor(total, 16, WAVE);
      total += __shfl_xor(total, 32, WAVE);
      if (live[b] && slots > 1) {
        const int64_t slot = ((int64_t)(token0 + b * 16 + col) * nq + head) * slots + split;
#pragma unroll
        for (int e = 0; e < DB; ++e)
          if (e * 16 < dv) *(floatx4*)(part_o + slot * dv + e * 16 + g * 4) = o[b][e];
        if (g == 0) {
          part_ml[slot * 2] = run_max[b] * scale2;               // -inf stays -inf: no key seen
          part_ml[slot * 2 + 1] = total;
        }
      } else if (live[b]) {
        const float keep = sinks ? with_sink(sinks[head] * LOG2E, run_max[b] * scale2, total) : 1.f;
        const float inv = keep / total * head_gate(gates, gate_stride, token0 + b * 16 + col, head);
        bf16* dst = out + (int64_t)(token0 + b * 16 + col) * out_stride + (int64_t)head * dv + g * 4;
#pragma unroll
        for (int e = 0; e < DB; ++e) {
          if (e * 16 >= dv) break;
          const bf16x4 packed = {(bf16)(o[b][e][0] * inv), (bf16)(o[b][e][1] * inv), (bf16)(o[b][e][2] * inv), (bf16)(o[b][e][3] * inv)};
          *(bf16x4*)(dst + e * 16) = packed;
        }
      }
    }
  }
}

// ------------------------------------- bf16 kernel for any step, head size 128
// The same walk as attention_prefill_bf16_kernel with the tiles brought in differently: memory
// writes them straight into LDS (global_load_lds_dwordx4: a wave's 64 lanes fetch 16 bytes each,
// from addresses of their own choice, and the 1,024 bytes land in lane order at the address in m0),
// so a tile passes through no registers, three tiles are in flight instead of one, nothing is written
// to LDS by the waves, and where a piece lies in LDS is decided by which lane fetches it.
//
// LDS serves 16-byte reads at its full 256 bytes a cycle when the lanes it takes together (eight
// consecutive rows of the fragment, pieces g and g + 1) fall on 64 different banks; measured, and
// that is what the layout is made for:
//   keys    eight blocks of 1,024 bytes (four rows of 256), block j at j * 1,056; row (h, col) of
//           the first product's fragments lies in block col % 8 as its row 2 h + col / 8, so eight
//           consecutive columns meet eight blocks, each 8 banks further on than the one before.
//   values  transposed, a half for each run of 16 keys: [half][dim][16 keys], the second half 16
//           bytes out of step; lanes g = 0, 2 read the first half's two pieces, g = 1, 3 the second's.
// A block is one fetch of one wave and comes from one page.  Which key a fragment row holds is free
// as long as the second product meets the weights where the first left them: lanes of group g hold
// the scores of keys 8 m + 4 h + i (m = 0, 2, 1, 3 for g = 0..3; h the fragment, i the register), and
// read the values of keys 8 m .. 8 m + 7 as one piece.
// The wave that fetched a tile waits for its own fetches (vmcnt) before the barrier that opens the
// tile to the others; the fetches of the tile after it stay in flight.  The fetches are written in
// assembly because the compiler would wait for all of them before any LDS read it cannot tell apart.
// What bounds a walk is the instructions a wave issues beside its products (one every four cycles at most): 32 products of a turn
// of 32 queries come with 80 vector, 33 scalar and 18 LDS instructions, and the chip's clock is at 2.1 GHz meanwhile.  Turns of
// 215 instructions that also waited for the fetches they had just made, for scalar loads of the block table and for every value
// fragment in turn took 1.40 us with two workgroups a unit behind contexts in memory, these 1.11 (16 heads on 8, 2,048 tokens after
// 14,336: 360 -> 284 us a layer; 32 on 8 691 -> 486; 32,768 tokens 8.95 -> 7.64 ms, 1.15 PFLOP/s; 2,048 after 2,048 152 -> 115).
// A walk of a few tiles (short prompts, windows) is bound by what stands before its first turn.  us with the longer turns of that
// time / with these and a chain of waits before them / with all asked for at once and nothing spilled: 16 heads on 8, 2,048 tokens,
// window of 128 21.4 / 29.1 / 21.9, linear bias 26.1 / 42.9 / 26.7; 100 tokens 8.5 / 9.3 / 8.6; 32 on 8, linear bias, 32 tokens 7.1 /
// 8.9 / 7.3, 2,048 in a window of 512 51 / 61 / 47; plain, 2,048 tokens 63.7 / 62.2 / 57.6, 2,048 after 2,048 165 / 124 / 116.
// SCORES: what happens to the scores before the softmax, by instances of their own so that the others keep their registers:
// nothing, a cap (softcap * tanh(score / softcap) of the scaled scores), a bias by distance (in the form with a logarithm, or the
// linear one, which without a cap is what the products are added to and costs nothing), or the cap and then the bias.
enum { SCORES_PLAIN = 0, SCORES_CAPPED = 1, SCORES_DISTANCE = 2, SCORES_BOTH = 3, SCORES_LINEAR = 4, SCORES_CAPPED_LINEAR = 5 };
// SPREAD: how a kv group's heads meet the waves: a wave a head (in several passes if there are more heads than waves); the same with
// waves that have no head in some pass; and for two heads, which left half of the waves idle, a wave a (head, block of 16 queries) or,
// where neighbouring groups are one request's, a wave a (head, group of 32).  A turn of the walk costs its tile's way from the
// L2s (16 KB a turn and workgroup) and its barrier whatever is done with them, so a pair walking together does twice as much with it
// (before turns were made shorter: 16 heads on 8, 2,048 tokens after 14,336: 569 us with idle waves, 444 with halves, 322 in pairs with
// the keys divided by two; 8,192 tokens 584 / 385 / 390; 2,048 after 2,048 142 / 136 / 100).
enum { SPREAD_HEADS = 0, SPREAD_SOME_IDLE = 1, SPREAD_HALVES = 2, SPREAD_PAIRS = 3 };
struct PrefillLds {
  static constexpr int D = 128, STAGES = 3, KBLOCK = 1024 + 32, KBYTES = 8 * KBLOCK, VHALF = 16 * D * 2 + 16;
  static constexpr int VSTAGE = (2 * VHALF + 63) / 64 * 64;
  __attribute__((aligned(64))) unsigned char key_tiles[STAGES * KBYTES];
  __attribute__((aligned(64))) unsigned char value_tiles[STAGES * VSTAGE];
  // where runs of 16 keys lie in memory, and their values: rings of two blocks of 64 runs (the values' a tile further on, so that
  // one place in both holds what a turn asks for: the keys of one tile and the values of the tile before it)
  static constexpr int BLOCK_RUNS = 64, RUNS = 2 * BLOCK_RUNS;
  __attribute__((aligned(16))) uint64_t key_runs[RUNS];
  __attribute__((aligned(16))) uint64_t value_runs[RUNS];
};
template <int QB, bool MANY_WAVES, int SPREAD, int SCORES>
__device__ __forceinline__ void attention_prefill_d128_part(
    PrefillLds& lds, int block, bf16* __restrict__ out, int out_stride, const bf16* __restrict__ q, int q_stride,
    const bf16* __restrict__ k_pages, const bf16* __restrict__ v_pages,
    const int* __restrict__ block_table, int table_stride, const int* __restrict__ token_request,
    const int* __restrict__ positions, const int* __restrict__ qblock_token0,
    const int* __restrict__ qblock_count, int n_blocks, int chunk, int nq, int nkv, int page_size, float scale,
    int window, int splits, int slots, float* __restrict__ part_o, float* __restrict__ part_ml, int prepare_q, DecodePrep prep,
    const float* __restrict__ sinks, float softcap, const bf16* __restrict__ gates, int gate_stride, int dv,
    const float* __restrict__ distance) {
  constexpr bool CAPPED = (SCORES & SCORES_CAPPED) != 0, DISTANCE = (SCORES & SCORES_DISTANCE) != 0, LINEAR = (SCORES & SCORES_LINEAR) != 0;
  constexpr bool IDLE_WAVES = SPREAD == SPREAD_SOME_IDLE, HALVES = SPREAD == SPREAD_HALVES, PAIRS = SPREAD == SPREAD_PAIRS;
  static_assert(!HALVES || (QB == 1 && !MANY_WAVES), "two heads and two blocks of 16 queries are four waves' work");
  static_assert(!PAIRS || (QB == 2 && !MANY_WAVES), "two heads and two groups of 32 queries are four waves' work");
  constexpr int D = 128, DS = D / 32, DB = D / 16, STAGES = 3;
  constexpr int KBLOCK = PrefillLds::KBLOCK, KBYTES = PrefillLds::KBYTES, VHALF = PrefillLds::VHALF, VSTAGE = PrefillLds::VSTAGE;
  static_assert(D == PrefillLds::D && STAGES == PrefillLds::STAGES, "what the tiles' place is made for");
  auto& key_tiles = lds.key_tiles;
  auto& value_tiles = lds.value_tiles;
  const int tid = threadIdx.x;
  const int wave = __builtin_amdgcn_readfirstlane(tid / WAVE);
  int lane = tid % WAVE;                                           // (set anew in every pass over the keys: see there)
  const int group = nq / nkv;
  const int n_walks = PAIRS ? (n_blocks + 1) / 2 : n_blocks;       // PAIRS: two neighbouring groups of one request walk together
  const int work = block % (n_walks * nkv), split = block / (n_walks * nkv);
  const int which_chunk = work / chunk, in_chunk = work % chunk;
  const int chunk_block0 = which_chunk * (chunk / nkv);
  const int chunk_blocks = n_walks - chunk_block0 < chunk / nkv ? n_walks - chunk_block0 : chunk / nkv;
  const int kvh = in_chunk % nkv;
  const int walk = chunk_block0 + ((which_chunk & 1) ? chunk_blocks - 1 - in_chunk / nkv : in_chunk / nkv);
  // groups stand from a request's last tokens to its first
  const int later = PAIRS ? 2 * walk : walk, earlier = PAIRS && later + 1 < n_blocks ? later + 1 : later;
  const int qblock = PAIRS && wave >= 2 ? earlier : later;
  const int token0 = qblock_token0[qblock], count = PAIRS && wave >= 2 && earlier == later ? 0 : qblock_count[qblock];
  const int pos_first = positions[qblock_token0[earlier]], pos_last = positions[qblock_token0[later] + qblock_count[later] - 1];
  const int lo_first = first_seen(pos_first, window);
  const int lo_last = first_seen(pos_last, window);
  const int* table = block_table + (int64_t)token_request[token0] * table_stride;
  const bf16x8 zero8 = {0, 0, 0, 0, 0, 0, 0, 0};
  const float scale2 = scale * 1.4426950408889634f;
  const float rescale_step = RESCALE_STEP / scale2;              // in units of the unscaled scores
  int first_tile = lo_first / 32, last_tile = pos_last / 32;
  if (splits > 1) {                                              // this workgroup's share of the tiles (may be none)
    const int per_split = (last_tile - first_tile + splits) / splits;
    first_tile += split * per_split;
    if (first_tile + per_split - 1 < last_tile) last_tile = first_tile + per_split - 1;
  }
  const int first_run = lo_first / 16, last_run = pos_last / 16;   // runs of 16 keys that hold a key some query sees

  // What this wave fetches of a tile: key blocks `wave` (first run) and `wave + 4` (second run), and the
  // dimensions 32 wave .. 32 wave + 31 of both value halves.  A lane's distance from the run's first key
  // (or first slot) never changes; the run's page is looked up once a wave.
  const int pages16 = page_size / 16;                            // runs of 16 keys in a page
  const unsigned magic = pages16 > 1 ? 0xFFFFFFFFu / (unsigned)pages16 + 1u : 0u;   // run / pages16 = umulhi(run, magic)
  const unsigned keys_address = (unsigned)(uintptr_t)(__attribute__((address_space(3))) unsigned char*)key_tiles;
  const unsigned values_address = (unsigned)(uintptr_t)(__attribute__((address_space(3))) unsigned char*)value_tiles;
  // Where a run of 16 keys lies in memory: a page from the block table and a place in it.  A run no query sees is masked: any page
  // with numbers in it will do, so runs are clamped to those the queries do see.
  const uint64_t page_bytes = (uint64_t)nkv * page_size * D * 2;            // from page to page of keys ...
  const uint64_t value_page_bytes = (uint64_t)nkv * page_size * dv * 2;     // ... and of values
  const char* const k_head = (const char*)(k_pages + (int64_t)kvh * page_size * D);
  const char* const v_head = (const char*)(v_pages + (int64_t)kvh * page_size * dv);
  struct Run {
    int number, entry;
  };
  auto run_in_reach = [&](int run) {
    run = run < first_run ? first_run : run > last_run ? last_run : run;
    return Run{run, pages16 > 1 ? (int)__umulhi((unsigned)run, magic) : run};
  };
  auto locate = [&](const Run& run, int page, uint64_t& keys, uint64_t& values) {
    const unsigned in_page = (unsigned)(run.number - run.entry * pages16) * 16u;
    keys = (uint64_t)(uintptr_t)k_head + (uint64_t)(unsigned)page * page_bytes + in_page * (unsigned)(D * 2);
    values = (uint64_t)(uintptr_t)v_head + (uint64_t)(unsigned)page * value_page_bytes + in_page * 2u;
  };
  constexpr int BLOCK_RUNS = PrefillLds::BLOCK_RUNS, RUNS = PrefillLds::RUNS;

  // kv groups of more than four heads take several passes over the keys
  const int waves = MANY_WAVES ? blockDim.x / WAVE : 4;
  // two heads: a wave has one of them and one of the group's two blocks of 16 queries (beginning at query0), or one of two groups
  const int query0 = HALVES ? (wave >> 1) * 16 : 0;
  // waves without a head sit on other SIMDs in the workgroup that shares the compute unit (the 256th from here)
  const int my_wave = HALVES || PAIRS ? wave & 1 : IDLE_WAVES && !MANY_WAVES ? (wave + (block >> 8 & 1) * 2) & 3 : wave;
  for (int head0 = kvh * group; head0 < (kvh + 1) * group; head0 += waves) {
    const int head = head0 + my_wave;
    const bool active = head < (kvh + 1) * group;
    // What follows from the lane is worked out in every pass.  Left alone the compiler takes all of it, addresses of loads before and
    // behind the walk too, for values to keep through all passes, and has no registers for them: 14 to 63 were spilled, and each one's
    // way back waits for every fetch asked for before it.
    int begin = first_tile;
    asm volatile("" : "+v"(lane), "+s"(begin));
    const int col = lane & 15, g = lane >> 4;
    const int key_chunk = ((g & 1) << 1) | (g >> 1);           // m: the eight keys this lane group holds weights of
    // lane l of a key block brings row l / 16 (h = row / 2, k = row % 2), piece l % 16: key 8 k + 4 h + wave of its run
    const unsigned key_offset = (unsigned)(((((lane >> 4) & 1) * 8 + (lane >> 5) * 4 + wave) * D + (lane & 15) * 8) * 2);
    // lane l of a value block brings dimension 32 wave + l / 2, keys 8 (l % 2) .. + 7 of the run
    // (values narrower than keys: the dims behind them repeat the last one)
    const int value_dim = wave * 32 + (lane >> 1) < dv ? wave * 32 + (lane >> 1) : dv - 1;
    const unsigned value_offset = (unsigned)(((value_dim * page_size) + (lane & 1) * 8) * 2);
    // where this lane's fragments lie in a stage
    const int key_fragment = (col & 7) * KBLOCK + (col >> 3) * 256 + g * 16;              // + h * 512 + c * 64
    const int value_fragment = (g & 1) * VHALF + col * 32 + (g >> 1) * 16;                // + e * 512

    // A wave's lanes look up a block of 64 runs at a time and leave the addresses in LDS, from where every turn takes its four: the
    // same work done by every wave in every turn with scalar instructions (loads of the block table among them, which LDS reads cannot
    // be waited for apart from) was 60 of a turn's 215 instructions.
    auto leave_block = [&](int which, const Run& run, int page) {
      uint64_t keys, values;
      locate(run, page, keys, values);
      const int at = (which & 1) * BLOCK_RUNS + lane;
      lds.key_runs[at] = keys;
      lds.value_runs[(at + 2) & (RUNS - 1)] = values;
      asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");             // there before this wave comes to the next barrier
    };
    struct Pair {
      uint64_t run[2];
    };
    auto runs_at = [&](const uint64_t (&ring)[RUNS], int place) {
      typedef uint64_t pair __attribute__((ext_vector_type(2)));
      const pair at = *(const pair*)&ring[place];
      return Pair{{at[0], at[1]}};
    };
    // (a kv group of five to eight heads brings as many waves, so that one walk over the keys serves them all;
    // the first four waves bring the tiles in)
    auto fetch_keys = [&](const Pair& from, int stage) {      // two fetches a wave
      if (MANY_WAVES && wave >= 4) return;
#pragma unroll
      for (int half = 0; half < 2; ++half)
        fetch_lanes_to_lds(from.run[half] + key_offset, keys_address + (unsigned)(stage * KBYTES + (wave + 4 * half) * KBLOCK));
    };
    auto fetch_values = [&](const Pair& from, int stage) {    // two fetches a wave
      if (MANY_WAVES && wave >= 4) return;
#pragma unroll
      for (int half = 0; half < 2; ++half)
        fetch_lanes_to_lds(from.run[half] + value_offset, values_address + (unsigned)(stage * VSTAGE + half * VHALF + wave * 1024));
    };
    // What a walk begins with is asked for before anything is waited for: the pages of the first two blocks of runs, positions and
    // raw rows, and behind them the first tiles, whose addresses come by scalar loads.  A wait in between is a trip to memory of its
    // own, since a wave's loads come back in the order they were asked for, and short walks are little else.
    __syncthreads();                                           // the stages of an earlier pass are done with
    bf16x8 qf[QB][DS];
    int pos[QB], lo[QB];
    bool live[QB];
    const Run my_run = run_in_reach(begin * 2 + (wave & 1) * BLOCK_RUNS + lane);
    const int my_page = table[my_run.entry];
#pragma unroll
    for (int b = 0; b < QB; ++b) {
      live[b] = active && query0 + b * 16 + col < count;
      const int token = token0 + (live[b] ? query0 + b * 16 + col : 0);      // (a dead column takes its group's first token and drops the result)
      pos[b] = positions[token];
      const bf16* row = q + (int64_t)token * q_stride + (int64_t)(active ? head : head0) * D + g * 8;
#pragma unroll
      for (int c = 0; c < DS; ++c) qf[b][c] = *(const bf16x8*)(row + c * 32);
    }
    int pending = 0;
    if (first_tile <= last_tile) {
      const char *keys[3][2], *values[3][2];
#pragma unroll
      for (int n = 0; n < 3; ++n)
#pragma unroll
        for (int half = 0; half < 2; ++half) {
          const Run run = run_in_reach((begin + n) * 2 + half);
          uint64_t key_at, value_at;
          locate(run, table[run.entry], key_at, value_at);
          keys[n][half] = (const char*)(uintptr_t)key_at, values[n][half] = (const char*)(uintptr_t)value_at;
        }
      auto first_keys = [&](int n) {
        if (MANY_WAVES && wave >= 4) return;
#pragma unroll
        for (int half = 0; half < 2; ++half) fetch_to_lds(keys[n][half], key_offset, keys_address + (unsigned)(n * KBYTES + (wave + 4 * half) * KBLOCK));
      };
      auto first_values = [&](int n) {
        if (MANY_WAVES && wave >= 4) return;
#pragma unroll
        for (int half = 0; half < 2; ++half) fetch_to_lds(values[n][half], value_offset, values_address + (unsigned)(n * VSTAGE + half * VHALF + wave * 1024));
      };
      first_keys(0);
      first_values(0);
      if (first_tile + 1 <= last_tile) first_keys(1);
      if (first_tile + 2 <= last_tile) first_keys(2), pending += 2;
      if (first_tile + 1 <= last_tile) first_values(1), pending += 2;
      if (wave < 2 && first_tile + 2 <= last_tile) leave_block(wave, my_run, my_page);
    }
    floatx4 o[QB][DB];
    float run_max[QB], run_sum[QB];
#pragma unroll
    for (int b = 0; b < QB; ++b) {
      pos[b] = live[b] ? pos[b] : -1;                          // a dead column sees no key
      lo[b] = first_seen(pos[b], window);
      run_max[b] = -INFINITY;
      run_sum[b] = 0.f;
      // q holds the raw rows of the q/k/v product: the head is normalised and rotated here, in the registers it stays in
      if (prepare_q) {
        float x[DS][8];
#pragma unroll
        for (int c = 0; c < DS; ++c)
#pragma unroll
          for (int j = 0; j < 8; ++j) x[c][j] = (float)qf[b][c][j];
        const int token = token0 + (live[b] ? query0 + b * 16 + col : 0);
        head_from_memory<D>(qf[b], x, g, prep.q_weight, prep.weight_is_f32, prep.eps, prep.cosv ? prep.cosv + (int64_t)token * (D / 2) : nullptr,
                            prep.sinv ? prep.sinv + (int64_t)token * (D / 2) : nullptr);
      }
#pragma unroll
      for (int c = 0; c < DS; ++c) qf[b][c] = live[b] ? qf[b][c] : zero8;
#pragma unroll
      for (int e = 0; e < DB; ++e) o[b][e] = floatx4{0.f, 0.f, 0.f, 0.f};
    }
    // The queries and positions are waited for here.  Left to the compiler the wait stands before their first use, in the walk's
    // inner loop, where it waits for every fetch just asked for as well, in every turn.
#pragma unroll
    for (int b = 0; b < QB; ++b) {
      asm volatile("" : "+v"(pos[b]));
#pragma unroll
      for (int c = 0; c < DS; ++c) asm volatile("" : "+v"(qf[b][c]));
    }

    // the cap, in units of the unscaled scores (the scale enters with the exponent)
    auto cap_scores = [&](floatx4 (&sc)[QB][2]) {
      const float cap = softcap / scale;
#pragma unroll
      for (int b = 0; b < QB; ++b)
#pragma unroll
        for (int h = 0; h < 2; ++h)
#pragma unroll
          for (int i = 0; i < 4; ++i) sc[b][h][i] = capped(sc[b][h][i], cap);
    };
    // the bias by distance, likewise; sc[b][h][i] belongs to key tile * 32 + 8 m + 4 h + i (a key ahead of the query gives no
    // number here; the mask takes it out)
    float rate = 0.f, reach = 0.f;
    if constexpr (DISTANCE) {
      const int biased = active ? head : head0;
      rate = distance[biased] * LN2 / scale;
      reach = distance[nq + biased];
    }
    if constexpr (LINEAR) rate = distance[active ? head : head0] / scale;
    // The linear form in two parts, as in attention_prefill_bf16_kernel: the lane's eight keys' places in their tile, and the tile's
    // distance from the query, which joins the exponents' shift; or taken off whole.
    constexpr bool IN_PARTS = LINEAR && !CAPPED && QB == 1, RAISES = LINEAR && QB == 1;
    floatx4 in_tile[2] = {{0.f, 0.f, 0.f, 0.f}, {0.f, 0.f, 0.f, 0.f}};
    if constexpr (IN_PARTS) {
#pragma unroll
      for (int h = 0; h < 2; ++h)
#pragma unroll
        for (int i = 0; i < 4; ++i) in_tile[h][i] = rate * (float)(key_chunk * 8 + h * 4 + i);
    }
    auto of_tile = [&](int tile, int b) { return -rate * (float)((live[b] ? pos[b] : pos_last) - tile * 32); };
    auto linear_bias = [&](int tile, int b, int h) {
      return linear_of_four(rate, (float)((live[b] ? pos[b] : pos_last) - (tile * 32 + key_chunk * 8 + h * 4)));
    };
    // what a tile's products are added to
    auto begin_scores = [&](int tile, floatx4 (&sc)[QB][2]) {
#pragma unroll
      for (int b = 0; b < QB; ++b)
#pragma unroll
        for (int h = 0; h < 2; ++h) {
          if constexpr (LINEAR && !CAPPED && !IN_PARTS) sc[b][h] = linear_bias(tile, b, h);
          else sc[b][h] = in_tile[h];
        }
    };
    auto take_off_linear = [&](int tile, floatx4 (&sc)[QB][2]) {
#pragma unroll
      for (int b = 0; b < QB; ++b)
#pragma unroll
        for (int h = 0; h < 2; ++h) sc[b][h] += linear_bias(tile, b, h);
    };
    bool grown = false;                                        // a linear bias's weights have left the reference points behind
    auto raise_reference = [&]() {
#pragma unroll
      for (int b = 0; b < QB; ++b) {
        const float more = growth_of(run_sum[b]), shrink = fast_exp2(-more);
        run_max[b] += more / scale2;
        run_sum[b] *= shrink;
#pragma unroll
        for (int e = 0; e < DB; ++e) o[b][e] *= shrink;
      }
      grown = false;
    };
    auto take_off_distance = [&](int tile, floatx4 (&sc)[QB][2]) {
#pragma unroll
      for (int b = 0; b < QB; ++b) {
        const float behind = (float)((live[b] ? pos[b] : pos_last) - (tile * 32 + key_chunk * 8));
        const float first = fmaf(reach, behind, 1.f);
#pragma unroll
        for (int h = 0; h < 2; ++h)
#pragma unroll
          for (int i = 0; i < 4; ++i) sc[b][h][i] = fmaf(-rate, __builtin_amdgcn_logf(fmaf(-reach, (float)(4 * h + i), first)), sc[b][h][i]);
      }
    };
    // scores: S[key, query] = K Q^T, unscaled (the scale enters with the exponent)
    auto scores = [&](int tile, int stage, floatx4 (&sc)[QB][2]) {
      const unsigned char* kt = key_tiles + stage * KBYTES + key_fragment;
      begin_scores(tile, sc);
#pragma unroll
      for (int h = 0; h < 2; ++h)
#pragma unroll
        for (int c = 0; c < DS; ++c) {
          const bf16x8 kfrag = *(const bf16x8*)(kt + h * 512 + c * 64);
#pragma unroll
          for (int b = 0; b < QB; ++b) sc[b][h] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(kfrag, qf[b][c], sc[b][h], 0, 0, 0);
        }
      if constexpr (CAPPED) cap_scores(sc);
      if constexpr (DISTANCE) take_off_distance(tile, sc);
      if constexpr (LINEAR && CAPPED) take_off_linear(tile, sc);
    };
    // weights: as in attention_prefill_bf16_kernel; sc[b][h][i] belongs to key tile * 32 + 8 m + 4 h + i
    auto weights_with_maximum = [&](int tile, floatx4 (&sc)[QB][2], auto masked, bf16x8 (&pf)[QB]) {
      constexpr bool MASKED = decltype(masked)::value;
      float alpha[QB];
      bool rescale = false;
#pragma unroll
      for (int b = 0; b < QB; ++b) {
        float tile_max = -INFINITY;
        if constexpr (IN_PARTS) {
          const float all = of_tile(tile, b);
          sc[b][0] += all;
          sc[b][1] += all;
        }
#pragma unroll
        for (int h = 0; h < 2; ++h)
#pragma unroll
          for (int i = 0; i < 4; ++i) {
            if (MASKED) {
              const int key = tile * 32 + key_chunk * 8 + h * 4 + i;
              sc[b][h][i] = (key <= pos[b] && key >= lo[b]) ? sc[b][h][i] : -INFINITY;
            }
            tile_max = fmaxf(tile_max, sc[b][h][i]);
          }
        tile_max = fmaxf(tile_max, __shfl_xor(tile_max, 16, WAVE));
        tile_max = fmaxf(tile_max, __shfl_xor(tile_max, 32, WAVE));
        const float new_max = tile_max > run_max[b] + rescale_step ? tile_max : run_max[b];
        // a query whose window or position leaves it no key so far keeps its state
        const bool empty = MASKED && new_max == -INFINITY;
        alpha[b] = empty ? 1.f : fast_exp2((run_max[b] - new_max) * scale2);
        const float shift = empty ? 0.f : -new_max * scale2;
        run_max[b] = new_max;
        float tile_sum = 0.f;
#pragma unroll
        for (int h = 0; h < 2; ++h)
#pragma unroll
          for (int i = 0; i < 4; ++i) {
            const float p = fast_exp2(fmaf(sc[b][h][i], scale2, shift));
            tile_sum += p;
            pf[b][h * 4 + i] = (bf16)p;
          }
        run_sum[b] = run_sum[b] * alpha[b] + tile_sum;
        rescale |= alpha[b] != 1.f;
      }
      if (__any(rescale)) {
#pragma unroll
        for (int b = 0; b < QB; ++b)
#pragma unroll
          for (int e = 0; e < DB; ++e) o[b][e] *= alpha[b];
      }
    };
    // The short way through the weights of the tile whose scores are in `sc`, and beside it the scores of the
    // tile after it (keys in `stage`) into `next`: the matrix cores work on the next tile's products while the
    // vector units turn this tile's scores into weights.  The two are independent and are written here one
    // product, one weight at a time, with a fence for the instruction scheduler after each pair, so that this
    // is the order the wave issues them in: a product keeps the matrix core busy for 16 cycles, in which the
    // three or four vector instructions of a weight cost nothing.  A head of 128 has as many products a tile
    // (8 for every 16 queries) as a lane has weights.  Returns false, and has changed nothing but pf and
    // next, if a weight sum says the reference point will not do.
    // The fragments of keys, and those of the tile's own values for the products that follow (values_read_ahead), are asked for
    // READ_AHEAD ahead of their products.
    constexpr int READ_AHEAD = 3;
    auto weights_beside_scores = [&](int next_tile, int key_stage, int value_stage, floatx4 (&sc)[QB][2], floatx4 (&next)[QB][2],
                                     bf16x8 (&pf)[QB], bf16x8 (&vf)[DB]) -> bool {
      const unsigned char* kt = key_tiles + key_stage * KBYTES + key_fragment;
      const unsigned char* vt = value_tiles + value_stage * VSTAGE + value_fragment;
      constexpr int FRAGMENTS = 2 * DS;
      static_assert(FRAGMENTS * QB == QB * 8, "one weight for every product");
      bf16x8 kf[FRAGMENTS];
#pragma unroll
      for (int f = 0; f < READ_AHEAD; ++f) kf[f] = *(const bf16x8*)(kt + (f / DS) * 512 + (f % DS) * 64);
      float shift[QB], tile_sum[QB], weight[QB * 8];
      begin_scores(next_tile, next);
#pragma unroll
      for (int b = 0; b < QB; ++b) {
        shift[b] = ((IN_PARTS ? of_tile(next_tile - 1, b) : 0.f) - run_max[b]) * scale2;      // +inf before the query's first tile: the sum then says "again"
        tile_sum[b] = 0.f;
      }
      __builtin_amdgcn_sched_barrier(0);
#pragma unroll
      for (int n = 0; n < FRAGMENTS * QB; ++n) {
        const int f = n / QB, b = n % QB;
        if (b == 0 && f + READ_AHEAD < FRAGMENTS)
          kf[f + READ_AHEAD] = *(const bf16x8*)(kt + ((f + READ_AHEAD) / DS) * 512 + ((f + READ_AHEAD) % DS) * 64);
        else if (b == 0) vf[f + READ_AHEAD - FRAGMENTS] = *(const bf16x8*)(vt + (f + READ_AHEAD - FRAGMENTS) * 512);
        next[b][f / DS] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(kf[f], qf[b][f % DS], next[b][f / DS], 0, 0, 0);
        const int wb = n / 8, wh = (n / 4) % 2, wi = n % 4;      // the n-th weight of the lane
        weight[n] = fast_exp2(fmaf(sc[wb][wh][wi], scale2, shift[wb]));
        tile_sum[wb] += weight[n];
        if (n % 2 == 1) {
          pf[wb][wh * 4 + wi - 1] = (bf16)weight[n - 1];
          pf[wb][wh * 4 + wi] = (bf16)weight[n];
        }
        __builtin_amdgcn_sched_barrier(0);
      }
#pragma unroll
      for (int b = 0; b < QB; ++b) asm volatile("" : "+v"(pf[b]));       // packed before the way parts: half the registers
      bool again = false;
#pragma unroll
      for (int b = 0; b < QB; ++b) again |= !(tile_sum[b] <= 0x1p60f);   // too large, infinite or not a number
      if (__builtin_amdgcn_ballot_w64(again) != 0) return false;
#pragma unroll
      for (int b = 0; b < QB; ++b) run_sum[b] += tile_sum[b];
      if constexpr (RAISES) {
        bool large = false;
#pragma unroll
        for (int b = 0; b < QB; ++b) large |= tile_sum[b] > GROWN;
        grown = __any(large);
      }
      if constexpr (CAPPED) cap_scores(next);
      if constexpr (DISTANCE) take_off_distance(next_tile, next);
      if constexpr (LINEAR && CAPPED) take_off_linear(next_tile, next);
      return true;
    };
    // values: O^T[dim, query] += V^T P
    auto values = [&](int stage, const bf16x8 (&pf)[QB]) {
      const unsigned char* vt = value_tiles + stage * VSTAGE + value_fragment;
#pragma unroll
      for (int e = 0; e < DB; ++e) {
        const bf16x8 vv = *(const bf16x8*)(vt + e * 512);
#pragma unroll
        for (int b = 0; b < QB; ++b) o[b][e] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(vv, pf[b], o[b][e], 0, 0, 0);
      }
    };

    // ... whose first fragments are on their way
    auto values_read_ahead = [&](int stage, const bf16x8 (&pf)[QB], bf16x8 (&vf)[DB]) {
      const unsigned char* vt = value_tiles + stage * VSTAGE + value_fragment;
#pragma unroll
      for (int e = 0; e < DB; ++e) {
        if (e + READ_AHEAD < DB) vf[e + READ_AHEAD] = *(const bf16x8*)(vt + (e + READ_AHEAD) * 512);
#pragma unroll
        for (int b = 0; b < QB; ++b) o[b][e] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(vf[e], pf[b], o[b][e], 0, 0, 0);
        __builtin_amdgcn_sched_barrier(0);
      }
    };

    // Tiles [whole_begin, whole_end) need no mask: every query of the group sees every key of theirs.
    int whole_begin = (lo_last + 31) / 32, whole_end = (pos_first + 1) / 32;
    if (whole_begin < first_tile) whole_begin = first_tile;
    if (whole_begin > last_tile + 1) whole_begin = last_tile + 1;
    if (whole_end > last_tile + 1) whole_end = last_tile + 1;
    if (whole_end < whole_begin) whole_end = whole_begin;

    // The walk.  Keys and values of tile t lie in stage (t - first_tile) % 3 of their rings.  A turn works on
    // tile t, whose scores the turn before has left in registers: it asks memory for the keys of t + 3 (their
    // stage was last read a turn ago, for the scores of t) and the values of t + 2 (likewise), computes the
    // scores of t + 1 beside the weights of t, adds the values of t, and before the barrier waits until only
    // what it asked for itself is still on its way: the keys of t + 2 and the values of t + 1 are then in LDS.
    floatx4 sa[QB][2], sb[QB][2];
    bf16x8 pf[QB];
    Pair keys_ahead, values_ahead;                             // where the keys of tile + 3 and the values of tile + 2 lie: known at the top of a turn
    if (first_tile <= last_tile) {
      if (pending == 4) fetched_and_read_then_barrier<4>();
      else if (pending == 2) fetched_and_read_then_barrier<2>();
      else fetched_and_read_then_barrier<0>();
      keys_ahead = runs_at(lds.key_runs, 6);
      values_ahead = runs_at(lds.value_runs, 6);
      if (!IDLE_WAVES || active) scores(first_tile, 0, sa);
      asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory");   // everyone has read the first keys: their stage may be filled again
    }
    int tile = first_tile, stage = 0;                          // stage = (tile - first_tile) % 3
    int place = 6;                                             // where the addresses of the tiles ahead stand in their rings
    // the third block and those after it are looked up two turns into the block before them, the last one that holds a tile too
    const int last_locate = last_tile - (BLOCK_RUNS / 2 - 2);
    int locate_at = first_tile + BLOCK_RUNS / 2 + 2 <= last_locate ? first_tile + BLOCK_RUNS / 2 + 2 : -1;
    // the turn's fetches, and how many they are; EVERY: tile + 3 is not past the last, so all of them happen
    auto ask_ahead = [&](auto every) -> int {
      constexpr bool EVERY = decltype(every)::value;
      int pending = 0;
      if (tile == locate_at) {
        // the block of runs behind the one that the walk is in takes the place of the one before it, which the walk left two turns ago
        if (wave == 0) {
          const int which = (tile - first_tile) / (BLOCK_RUNS / 2) + 1;
          const Run run = run_in_reach(first_tile * 2 + which * BLOCK_RUNS + lane);
          leave_block(which, run, table[run.entry]);
        }
        locate_at += BLOCK_RUNS / 2;
        if (locate_at > last_locate) locate_at = -1;
      }
      if (EVERY || tile + 3 <= last_tile) fetch_keys(keys_ahead, stage), pending += 2;
      if (EVERY || tile + 2 <= last_tile) fetch_values(values_ahead, stage == 0 ? STAGES - 1 : stage - 1), pending += 2;
      return pending;
    };
    // the addresses for the next turn's fetches, read late in a turn, where registers are free
    auto look_ahead = [&]() {
      place = (place + 2) & (RUNS - 1);
      keys_ahead = runs_at(lds.key_runs, place);
      values_ahead = runs_at(lds.value_runs, place);
    };
    auto turn_over = [&](int pending) {
      if (pending == 4) fetched_and_read_then_barrier<4>();
      else if (pending == 2) fetched_and_read_then_barrier<2>();
      else fetched_and_read_then_barrier<0>();
      stage = stage == STAGES - 1 ? 0 : stage + 1;
      ++tile;
    };
    // Most turns take the short way and have three tiles behind them: the inner loop holds only those, with
    // every count fixed, so that nothing in it touches the accumulators but the matrix products.  A tile
    // that needs the mask, or whose weights came out too large, or one of the last three, leaves it and takes
    // the long way.  The scores of the tile at hand are in sa at the top of every turn.
    const int fast_begin = whole_begin, fast_end = whole_end < last_tile - 2 ? whole_end : last_tile - 2;
    // A wave without a head (a kv group whose heads are no multiple of the waves: IDLE_WAVES, a kernel of its own
    // so that the others keep their registers) only brings its share of the tiles in and keeps the workgroup's
    // barriers: one a tile, as the others.
    if (IDLE_WAVES && !active) {
      while (tile <= last_tile) {
        const int on_their_way = ask_ahead(std::false_type{});
        look_ahead();
        turn_over(on_their_way);
      }
      continue;
    }
    for (;;) {
      bool asked = false;                                      // the turn's fetches have been asked for already
      const int fast_until = tile >= fast_begin ? fast_end : tile;
      // one way out of the inner loop only, at its top, before anything of the turn has happened to the accumulators
      for (;;) {
        if (asked || tile >= fast_until || (RAISES && grown)) break;
        ask_ahead(std::true_type{});
        bf16x8 vf[DB];
        if (!weights_beside_scores(tile + 1, stage == STAGES - 1 ? 0 : stage + 1, stage, sa, sb, pf, vf)) {
          asked = true;
          continue;
        }
        look_ahead();
        values_read_ahead(stage, pf, vf);
        turn_over(4);
#pragma unroll
        for (int b = 0; b < QB; ++b) sa[b][0] = sb[b][0], sa[b][1] = sb[b][1];
      }
      if constexpr (RAISES) {
        if (grown && !asked) {
          raise_reference();
          continue;
        }
      }
      const bool unfinished = tile <= last_tile;
      if (!unfinished) break;
      const int on_their_way = asked ? 4 : ask_ahead(std::false_type{});
      if (tile < last_tile) scores(tile + 1, stage == STAGES - 1 ? 0 : stage + 1, sb);
      if (tile >= whole_begin && tile < whole_end) weights_with_maximum(tile, sa, std::false_type{}, pf);
      else weights_with_maximum(tile, sa, std::true_type{}, pf);
      look_ahead();
      values(stage, pf);
      turn_over(on_their_way);
#pragma unroll
      for (int b = 0; b < QB; ++b) sa[b][0] = sb[b][0], sa[b][1] = sb[b][1];
    }
#pragma unroll
    for (int b = 0; b < QB; ++b) {
      float total = run_sum[b];
      total += __shfl_xor(total, 16, WAVE);
      total += __shfl_xor(total, 32, WAVE);
      if (live[b] && slots > 1) {
        const int64_t slot = ((int64_t)(token0 + query0 + b * 16 + col) * nq + head) * slots + split;
#pragma unroll
        for (int e = 0; e < DB; ++e)
          if (e * 16 < dv) *(floatx4*)(part_o + slot * dv + e * 16 + g * 4) = o[b][e];
        if (g == 0) {
          part_ml[slot * 2] = run_max[b] * scale2;               // -inf stays -inf: no key seen
          part_ml[slot * 2 + 1] = total;
        }
      } else if (live[b]) {
        const float keep = sinks ? with_sink(sinks[head] * LOG2E, run_max[b] * scale2, total) : 1.f;
        const float inv = keep / total * head_gate(gates, gate_stride, token0 + query0 + b * 16 + col, head);
        bf16* dst = out + (int64_t)(token0 + query0 + b * 16 + col) * out_stride + (int64_t)head * dv + g * 4;
#pragma unroll
        for (int e = 0; e < DB; ++e) {
          if (e * 16 >= dv) break;
          const bf16x4 packed = {(bf16)(o[b][e][0] * inv), (bf16)(o[b][e][1] * inv), (bf16)(o[b][e][2] * inv), (bf16)(o[b][e][3] * inv)};
          *(bf16x4*)(dst + e * 16) = packed;
        }
      }
    }
  }
}

template <int QB, bool MANY_WAVES, int SPREAD, int SCORES>
__global__ __launch_bounds__(MANY_WAVES ? 512 : 256, MANY_WAVES ? 1 : QB == 1 && (SCORES & SCORES_LINEAR) ? 3 : 2) void attention_prefill_d128_bf16_kernel(
    bf16* __restrict__ out, int out_stride, const bf16* __restrict__ q, int q_stride,
    const bf16* __restrict__ k_pages, const bf16* __restrict__ v_pages,
    const int* __restrict__ block_table, int table_stride, const int* __restrict__ token_request,
    const int* __restrict__ positions, const int* __restrict__ qblock_token0,
    const int* __restrict__ qblock_count, int n_blocks, int chunk, int nq, int nkv, int page_size, float scale,
    int window, int splits, int slots, float* __restrict__ part_o, float* __restrict__ part_ml, int prepare_q, DecodePrep prep,
    const float* __restrict__ sinks, float softcap, const bf16* __restrict__ gates, int gate_stride, int dv,
    const float* __restrict__ distance) {
  __shared__ PrefillLds lds;
  attention_prefill_d128_part<QB, MANY_WAVES, SPREAD, SCORES>(lds, blockIdx.x, out, out_stride, q, q_stride, k_pages, v_pages, block_table, table_stride, token_request, positions, qblock_token0, qblock_count, n_blocks, chunk, nq, nkv, page_size, scale, window, splits, slots, part_o, part_ml, prepare_q, prep, sinks, softcap, gates, gate_stride, dv, distance);
}

// --------------------------------- a mixed step's two kinds of rows in one launch
// The single tokens at the head of a mixed step (decoding requests) and the prompt portion behind them are independent, but
// as two launches one waits for the other: 24 tokens at 1,500 are bound by their keys' way from memory, 488 tokens behind as
// many by the length of a walk in fewer workgroups than the chip has room for.  Here the first single_blocks workgroups
// (token by token, the kv heads in turn) do what attention_decode_bf16_kernel does with four waves, the others what the
// kernel above does with four waves: 77 us a layer in two launches (32 heads on 8), 43 in one; which steps come here: _one_launch in
// parts/attention.py.  Heads of 128, plain scores, undivided keys.
template <int QB, int SPREAD, bool PREP>
__global__ __launch_bounds__(256, 2) void attention_mixed_d128_kernel(
    bf16* __restrict__ out, int out_stride, const bf16* __restrict__ q, int q_stride, bf16* __restrict__ k_pages, bf16* __restrict__ v_pages,
    const int* __restrict__ block_table, int table_stride, const int* __restrict__ token_request, const int* __restrict__ positions,
    const int* __restrict__ qblock_token0, const int* __restrict__ qblock_count, int n_blocks, int chunk, int nq, int nkv, int page_size,
    float scale, int window, DecodePrep prep, int singles) {
  __shared__ union Place {
    DecodeLds<128, 4> single;
    PrefillLds portion;
  } lds;
  extern __shared__ int page_ids[];
  const int single_blocks = singles * nkv;
  if ((int)blockIdx.x < single_blocks) {
    // The hint (load_once) for pages whose lines a wave reads alone, see _keys_read_once in parts/attention.py; whole steps with it / without, 24 requests at
    // 1,500 beside 488 tokens after 488 7,516 / 7,545 us (36 layers of the 4B sizes) and 4,241 / 4,177 (28 of the 1.7B), 40 at 800 beside 1,900 19,702 / 19,809
    // and 8,662 / 8,787, 8 at 4,000 beside 1,000 12,345 / 12,335 and 5,954 / 5,924.  Larger pages have the kernel alone take 49.0 / 44.7 for the first.
    auto one = [&](auto once) {
      attention_decode_part<128, PREP, 4, true, false, decltype(once)::value>(
          lds.single, page_ids, 0, blockIdx.x % nkv, blockIdx.x / nkv, out, out_stride, nullptr, nullptr, q, q_stride, k_pages, v_pages, block_table, table_stride,
          token_request, positions, nq, nkv, page_size, scale, window, 1, 1, prep, nullptr, 0.f, nullptr, 0, 128, nullptr, 0);
    };
    if (page_size <= 32) one(std::true_type{});
    else one(std::false_type{});
    return;
  }
  DecodePrep rest = prep;                                                  // the tables' rows of the tokens behind
  if (prep.cosv) rest.cosv += (int64_t)singles * 64, rest.sinv += (int64_t)singles * 64;
  attention_prefill_d128_part<QB, false, SPREAD, SCORES_PLAIN>(lds.portion, blockIdx.x - single_blocks, out + (int64_t)singles * out_stride, out_stride,
                                                               q + (int64_t)singles * q_stride, q_stride, k_pages, v_pages, block_table, table_stride,
                                                               token_request + singles, positions + singles, qblock_token0, qblock_count, n_blocks,
                                                               chunk, nq, nkv, page_size, scale, window, 1, 1, nullptr, nullptr, PREP, rest, nullptr,
                                                               0.f, nullptr, 0, 128, nullptr);
}

// Compute units of the current device (asked once).
static int compute_units() {
  static int units = 0;
  if (!units) {
    int device = 0;
    hipDeviceProp_t prop;
    if (hipGetDevice(&device) == hipSuccess && hipGetDeviceProperties(&prop, device) == hipSuccess) units = prop.multiProcessorCount;
    if (units <= 0) units = 256;
  }
  return units;
}

// Largest number of tokens in one query group of lrs_attention_prefill.
LRS_API int lrs_attention_prefill_group() { return 32; }

// The group size that serves a step of `tokens` tokens best, the longest context among them being `longest`
// (0: not known): groups of 16 while those of 32 would not give every compute unit its two workgroups several
// times over (measured on MI355X: a fresh prompt of up to 2,048 tokens is faster with 16, longer ones with 32);
// but groups of 32 already for 2,048 tokens behind as many or more, and for 1,024 behind three times as many: the
// walks are long then, and a wave with 32 queries does half as much beside its products for every key (2,048
// tokens after 2,048 / 6,144 / 30,720: 173 / 366 / 1,412 us with groups of 16, 142 / 272 / 1,071 with 32; 1,024
// after 7,168: 204 against 181 us; 512 after 7,680 stay with 16: 117 against 140 us).
LRS_API int lrs_attention_prefill_group_for(int tokens, int longest) {
  const int units = compute_units();
  if (tokens > 8 * units) return 32;
  if (tokens >= 8 * units && longest >= 2 * tokens) return 32;
  if (tokens >= 4 * units && longest >= 4 * tokens) return 32;
  return 16;
}

// Whether lrs_attention_prefill can be given the raw q rows of the q/k/v product (prepare != 0) for this head size.
LRS_API int lrs_attention_prefill_prepares(int d) { return d == 128; }

// Any step in bf16.  qblock_token0 / qblock_count [n_blocks]: first token and number of tokens
// (1..lrs_attention_prefill_group()) of each group of consecutive tokens of one request.
// splits > 1: every group's keys are divided between that many workgroups; needs part_o
// [tokens, nq, splits, d] and part_ml [tokens, nq, splits, 2] float32 and `tokens`, the step's size.
// prepare != 0 (heads of 128 only): q holds raw rows; every query head gets its RMSNorm (q_weight [d], or null for none)
// and the rotation of pairs (i, i + d/2) by the step's tables cosv / sinv [tokens, d/2] (null: none) on its way into the
// kernel's registers, as lrs_qk_prep would have left it in memory; the keys and values are in the pages already.
LRS_API int lrs_attention_prefill(void* out, int out_stride, const void* q, int q_stride, const void* k_pages,
                                  const void* v_pages, const int* block_table, int table_stride,
                                  const int* token_request, const int* positions, const int* qblock_token0,
                                  const int* qblock_count, int n_blocks, int max_count, int max_context, int nq,
                                  int nkv, int d, int page_size, float scale, int window, int keep_first, int tokens, int splits,
                                  float* part_o, float* part_ml, int prepare, const void* q_weight, int w_dtype, float eps,
                                  const float* cosv, const float* sinv, const float* sinks, float softcap, const void* gates,
                                  int gate_stride, int dv, const float* distance, int distance_form, int one_request, void* stream) {
  LRS_REQUIRE(distance_form == DISTANCE_LOG || distance_form == DISTANCE_LINEAR, "attention_prefill: unknown form %d of the bias by distance", distance_form);
  LRS_REQUIRE(dv > 0 && dv % 16 == 0 && dv <= d, "attention_prefill: values of %d dims beside keys of %d are not served (a multiple of 16, at most the keys')", dv, d);
  LRS_REQUIRE(n_blocks > 0 && nq > 0 && nkv > 0 && nq % nkv == 0, "attention_prefill: bad sizes blocks=%d nq=%d nkv=%d", n_blocks, nq, nkv);
  if (prepare) {
    LRS_REQUIRE(lrs_attention_prefill_prepares(d), "attention_prefill: only the kernel for heads of 128 prepares the queries itself, got head_dim %d", d);
    LRS_REQUIRE(q_weight == nullptr || eps > 0.f, "attention_prefill: eps must be positive");
    LRS_REQUIRE((cosv == nullptr) == (sinv == nullptr), "attention_prefill: cos and sin tables must come together");
    LRS_REQUIRE((uintptr_t)q_weight % 16 == 0 && (uintptr_t)cosv % 16 == 0 && (uintptr_t)sinv % 16 == 0,
                "attention_prefill: norm weight and rotation tables must be 16-byte aligned");
  }
  const DecodePrep prep{q_weight, nullptr, w_dtype == LRS_F32, eps, cosv, sinv, 0};
  LRS_REQUIRE(max_count >= 1 && max_count <= 32, "attention_prefill: query groups hold 1..32 tokens, got %d", max_count);
  LRS_REQUIRE(softcap >= 0.f, "attention_prefill: the cap on the scores must be positive (0 = none), got %g", (double)softcap);
  LRS_REQUIRE(page_size % 16 == 0, "attention_prefill: page size %d is not a multiple of 16", page_size);
  LRS_REQUIRE(keep_first >= 0 && (keep_first == 0 || (window > 0 && !prepare)),
              "attention_prefill: kept first positions (%d) need a window and prepared heads", keep_first);
  const int slots = splits + (keep_first > 0 ? 1 : 0);          // the kept keys' share is one more partial result
  const float* own_sinks = slots == 1 ? sinks : nullptr;          // with partial results the merge adds the sink
  const bf16* own_gates = slots == 1 ? (const bf16*)gates : nullptr;   // ... and applies the gate
  LRS_REQUIRE(q_stride % 8 == 0 && ((uintptr_t)q % 16) == 0 && out_stride % 4 == 0 && ((uintptr_t)out % 8) == 0,
              "attention_prefill: q rows must be 16-byte and out rows 8-byte aligned");
  // four waves (with fewer heads in a kv group the spare waves still help to bring tiles in), more only below
  LRS_REQUIRE(splits >= 1 && splits <= 64 && (slots == 1 || (part_o && part_ml && tokens > 0)),
              "attention_prefill: splits=%d (1..64) need partial buffers and the number of tokens", splits);
  LRS_REQUIRE(slots == 1 || ((uintptr_t)part_o % 16) == 0, "attention_prefill: part_o must be 16-byte aligned");
  dim3 grid(n_blocks * nkv * splits), block(4 * WAVE);
  // workgroups that share a compute unit: see the kernel
  const int chunk = nkv >= compute_units() ? nkv : compute_units() / nkv * nkv;
  // LDS copy of the block table entries a workgroup walks: at most those of the longest context
  LRS_REQUIRE(max_context >= 1, "attention_prefill: max_context must be the longest context length of the step");
  const int reach = window < 0 ? -window : window;
  const int span = reach > 0 && reach + 32 + 64 < max_context ? reach + 32 + 64 : max_context;
  const size_t table_lds = sizeof(int) * (size_t)(span / page_size + 2);
  // (the kernel for heads of 128 reads the block table with scalar loads and keeps no copy)
  LRS_REQUIRE(d == 128 || table_lds <= 24 * 1024, "attention_prefill: a context of %d tokens needs more block table entries than fit LDS", max_context);
  hipStream_t s = (hipStream_t)stream;
#define LAUNCH2(D, QB)                                                                                               \
  do {                                                                                                               \
    if (distance && distance_form == DISTANCE_LINEAR) LAUNCH3(D, QB, true);                                          \
    else LAUNCH3(D, QB, false);                                                                                      \
  } while (0)
#define LAUNCH3(D, QB, LINEAR)                                                                                       \
  attention_prefill_bf16_kernel<D, QB, LINEAR><<<grid, block, table_lds, s>>>((bf16*)out, out_stride, (const bf16*)q, q_stride, \
                                                              (const bf16*)k_pages, (const bf16*)v_pages, block_table, \
                                                              table_stride, token_request, positions, qblock_token0, \
                                                              qblock_count, n_blocks, chunk, nq, nkv, page_size, scale, window, \
                                                              splits, slots, part_o, part_ml, own_sinks, softcap, own_gates, gate_stride, dv, distance)
#define LAUNCH(D)                                \
  if (max_count <= 16) LAUNCH2(D, 1);            \
  else LAUNCH2(D, 2)
  switch (d) {
    case 32: LAUNCH(32); break;
    case 64: LAUNCH(64); break;
    case 96: LAUNCH(96); break;
    case 128:
      // head size 128 has a kernel of its own, whose tiles go from memory straight into LDS
      // A kv group of five to eight heads: a wave for every head and one walk over the keys instead of two, while
      // the launch is small (measured, 40 heads on 8: 512 tokens 28.9 -> 19.6 us, 512 tokens after 1,536 88 -> 54 us;
      // but 2,048 tokens 113 -> 129 us: a full chip does better with the smaller workgroups, three to a unit)
      {
        const bool many = nq / nkv > 4 && (int64_t)n_blocks * nkv * splits <= 2 * compute_units();
        if (many) block = dim3((nq / nkv < 8 ? nq / nkv : 8) * WAVE);
#define D128(QB, MANY, SPREAD)                                                                                                      \
        const bool linear = distance && distance_form == DISTANCE_LINEAR;                                                             \
        if (softcap > 0.f && linear) D128C(QB, MANY, SPREAD, SCORES_CAPPED_LINEAR);                                                     \
        else if (linear) D128C(QB, MANY, SPREAD, SCORES_LINEAR);                                                                        \
        else if (softcap > 0.f && distance) D128C(QB, MANY, SPREAD, SCORES_BOTH);                                                       \
        else if (softcap > 0.f) D128C(QB, MANY, SPREAD, SCORES_CAPPED);                                                                 \
        else if (distance) D128C(QB, MANY, SPREAD, SCORES_DISTANCE);                                                                    \
        else D128C(QB, MANY, SPREAD, SCORES_PLAIN)
#define D128C(QB, MANY, SPREAD, SCORES)                                                                                             \
        attention_prefill_d128_bf16_kernel<QB, MANY, SPREAD, SCORES><<<grid, block, 0, s>>>(                                            \
            (bf16*)out, out_stride, (const bf16*)q, q_stride, (const bf16*)k_pages, (const bf16*)v_pages, block_table, table_stride, \
            token_request, positions, qblock_token0, qblock_count, n_blocks, chunk, nq, nkv, page_size, scale, window, splits, slots, part_o, part_ml, \
            prepare, prep, own_sinks, softcap, own_gates, gate_stride, dv, distance)
#define D128_OF(QB)                                        \
        if (many && idle) { D128(QB, true, SPREAD_SOME_IDLE); }  \
        else if (many) { D128(QB, true, SPREAD_HEADS); }         \
        else if (idle) { D128(QB, false, SPREAD_SOME_IDLE); }    \
        else { D128(QB, false, SPREAD_HEADS); }
        const bool idle = (nq / nkv) % (int)(block.x / WAVE) != 0;   // some wave of some pass has no head
        if (max_count <= 16) { D128_OF(1); }
        else if (nq / nkv == 2 && one_request) {
          grid = dim3((n_blocks + 1) / 2 * nkv * splits);
          D128(2, false, SPREAD_PAIRS);
        } else if (nq / nkv == 2) { D128(1, false, SPREAD_HALVES); }
        else { D128_OF(2); }
#undef D128_OF
#undef D128
#undef D128C
      }
      break;
    case 192: LAUNCH(192); break;
    default: return lrs_fail("attention_prefill: head_dim %d has no matrix-core kernel (32, 64, 96, 128, 192)", d);
  }
#undef LAUNCH
#undef LAUNCH2
#undef LAUNCH3
  if (lrs_check_launch("attention_prefill")) return 1;
  if (keep_first > 0) {
    launch_attention_kept((const bf16*)q, q_stride, (const bf16*)k_pages, (const bf16*)v_pages, block_table, table_stride, token_request,
                          positions, tokens, nq, nkv, d, page_size, scale, window, keep_first, slots, part_o, part_ml, softcap, dv, distance, distance_form, s);
    if (lrs_check_launch("attention_kept")) return 1;
  }
  if (slots > 1) {
    launch_attention_merge((bf16*)out, out_stride, part_o, part_ml, tokens, nq, dv, slots, sinks, (const bf16*)gates, gate_stride, s);
    return lrs_check_launch("attention_merge");
  }
  return 0;
}

// lrs_attention_decode for the first `singles` tokens and lrs_attention_prefill for those behind them (qblock_token0 counts from
// there) in one launch: heads of 128, plain scores, undivided keys; prepare as there (the keys are in the pages already).
LRS_API int lrs_attention_mixed(void* out, int out_stride, const void* q, int q_stride, void* k_pages, void* v_pages, const int* block_table,
                                int table_stride, const int* token_request, const int* positions, const int* qblock_token0, const int* qblock_count,
                                int n_blocks, int max_count, int max_context, int nq, int nkv, int page_size, float scale, int window, int singles,
                                int prepare, const void* q_weight, int w_dtype, float eps, const float* cosv, const float* sinv, int one_request,
                                void* stream) {
  LRS_REQUIRE(singles > 0 && n_blocks > 0 && nq > 0 && nkv > 0 && nq % nkv == 0 && nq / nkv <= 16, "attention_mixed: bad sizes singles=%d blocks=%d nq=%d nkv=%d",
              singles, n_blocks, nq, nkv);
  LRS_REQUIRE(max_count >= 1 && max_count <= 32, "attention_mixed: query groups hold 1..32 tokens, got %d", max_count);
  LRS_REQUIRE(page_size > 0 && page_size % 16 == 0, "attention_mixed: page size %d is not a multiple of 16", page_size);
  LRS_REQUIRE(q_stride % 8 == 0 && ((uintptr_t)q % 16) == 0 && out_stride % 4 == 0 && ((uintptr_t)out % 8) == 0, "attention_mixed: q rows must be 16-byte and out rows 8-byte aligned");
  LRS_REQUIRE(max_context >= 1, "attention_mixed: max_context must be the longest context length of the step");
  if (prepare) {
    LRS_REQUIRE(q_weight == nullptr || eps > 0.f, "attention_mixed: eps must be positive");
    LRS_REQUIRE((cosv == nullptr) == (sinv == nullptr), "attention_mixed: cos and sin tables must come together");
    LRS_REQUIRE((uintptr_t)q_weight % 16 == 0 && (uintptr_t)cosv % 16 == 0 && (uintptr_t)sinv % 16 == 0, "attention_mixed: norm weight and rotation tables must be 16-byte aligned");
  }
  const int reach = window < 0 ? -window : window;
  const int span = reach > 0 && reach + 64 < max_context ? reach + 64 : max_context;
  const size_t table_lds = sizeof(int) * (size_t)((span / 32 + 1) * 32 / page_size + 4);
  LRS_REQUIRE(table_lds <= 24 * 1024, "attention_mixed: a context of %d tokens needs more block table entries than fit LDS", max_context);
  const DecodePrep prep{q_weight, nullptr, w_dtype == LRS_F32, eps, cosv, sinv, 0};
  const int chunk = nkv >= compute_units() ? nkv : compute_units() / nkv * nkv;
  const int heads = nq / nkv;
  hipStream_t s = (hipStream_t)stream;
#define MIXED(QB, SPREAD, WALKS)                                                                                                          \
  do {                                                                                                                                    \
    const dim3 grid(singles * nkv + (WALKS) * nkv);                                                                                       \
    if (prepare) attention_mixed_d128_kernel<QB, SPREAD, true><<<grid, 256, table_lds, s>>>(MIXED_ARGS);                                  \
    else attention_mixed_d128_kernel<QB, SPREAD, false><<<grid, 256, table_lds, s>>>(MIXED_ARGS);                                         \
  } while (0)
#define MIXED_ARGS                                                                                                                        \
  (bf16*)out, out_stride, (const bf16*)q, q_stride, (bf16*)k_pages, (bf16*)v_pages, block_table, table_stride, token_request, positions,  \
      qblock_token0, qblock_count, n_blocks, chunk, nq, nkv, page_size, scale, window, prep, singles
  const bool idle = heads % 4 != 0;
  if (max_count <= 16) { if (idle) MIXED(1, SPREAD_SOME_IDLE, n_blocks); else MIXED(1, SPREAD_HEADS, n_blocks); }
  else if (heads == 2 && one_request) MIXED(2, SPREAD_PAIRS, (n_blocks + 1) / 2);
  else if (heads == 2) MIXED(1, SPREAD_HALVES, n_blocks);
  else if (idle) MIXED(2, SPREAD_SOME_IDLE, n_blocks);
  else MIXED(2, SPREAD_HEADS, n_blocks);
#undef MIXED
#undef MIXED_ARGS
  return lrs_check_launch("attention_mixed");
}

// Compute units of the device, for callers that size their launches by it.
LRS_API int lrs_compute_units() { return compute_units(); }

// out [tokens, nq*d] (row stride out_stride); q rows are [nq*d] with row stride q_stride.
LRS_API int lrs_attention(void* out, int out_stride, const void* q, int q_stride, const void* k_pages,
                          const void* v_pages, const int* block_table, int table_stride,
                          const int* token_request, const int* positions, int dtype, int tokens,
                          int nq, int nkv, int d, int dv, int page_size, float scale, int window, int keep_first,
                          const float* sinks, float softcap, const void* gates, int gate_stride, const float* distance, int distance_form,
                          int together, int longest, void* stream) {
  // value pages [P, nkv, dv, page]; out rows hold nq heads of dv values; together, longest: attention_f32.hip
  LRS_REQUIRE(tokens > 0 && nq > 0 && nkv > 0 && d > 0 && dv > 0 && page_size > 0, "attention: bad sizes tokens=%d nq=%d nkv=%d d=%d dv=%d page=%d", tokens, nq, nkv, d, dv, page_size);
  LRS_REQUIRE(nq % nkv == 0, "attention: %d query heads do not divide into %d kv heads", nq, nkv);
  LRS_REQUIRE(d <= 512 && dv <= 512, "attention: head sizes %d and %d above the supported 512", d, dv);
  LRS_REQUIRE(keep_first >= 0 && (keep_first == 0 || window >= 0), "attention: keep_first must be >= 0 (0 = none) and comes with a window, not with chunks");
  LRS_REQUIRE(distance_form == DISTANCE_LOG || distance_form == DISTANCE_LINEAR, "attention: unknown form %d of the bias by distance", distance_form);
  LRS_REQUIRE(softcap >= 0.f, "attention: the cap on the scores must be positive (0 = none), got %g", (double)softcap);
  constexpr int THREADS = 128;
  dim3 grid(tokens, nq);
  const size_t lds = sizeof(float) * (d + d % 2 + THREADS) + (sizeof(int64_t) + sizeof(int)) * THREADS + 16;
  hipStream_t s = (hipStream_t)stream;
  // The plain form in float32 goes to the matrix cores (the choice never depends on the step, so a model's rows round alike in
  // every step); 16 heads on 8 of 128 dims, this kernel against that: a prompt of 509 tokens 230 / 41 us, of 2,048 3,174 / 305,
  // eight tokens at 509 35 / 18 (52 / 24 in a decode step), at 4,000 298 / 122, 16 tokens at 100 13.0 / 12.6
  if (dtype == LRS_F32 && !sinks && softcap == 0.f && !gates && !distance && keep_first == 0 &&
      lrs_attention_f32_takes(out, out_stride, q, q_stride, k_pages, v_pages, nq, nkv, d, dv, page_size))
    return lrs_attention_f32((float*)out, out_stride, (const float*)q, q_stride, (const float*)k_pages, (const float*)v_pages, block_table, table_stride,
                             token_request, positions, tokens, nq, nkv, d, page_size, scale, window, together, longest, s);
  if (dtype == LRS_F32)
    attention_generic_kernel<float, THREADS><<<grid, THREADS, lds, s>>>(
        (float*)out, out_stride, (const float*)q, q_stride, (const float*)k_pages, (const float*)v_pages,
        block_table, table_stride, token_request, positions, nq, nkv, d, dv, page_size, scale, window, keep_first, sinks, softcap, (const float*)gates, gate_stride, distance, distance_form);
  else if (dtype == LRS_BF16)
    attention_generic_kernel<bf16, THREADS><<<grid, THREADS, lds, s>>>(
        (bf16*)out, out_stride, (const bf16*)q, q_stride, (const bf16*)k_pages, (const bf16*)v_pages,
        block_table, table_stride, token_request, positions, nq, nkv, d, dv, page_size, scale, window, keep_first, sinks, softcap, (const bf16*)gates, gate_stride, distance, distance_form);
  else
    return lrs_fail("attention: unknown dtype %d", dtype);
  return lrs_check_launch("attention");
}
