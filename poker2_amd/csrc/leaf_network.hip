// A ReLU network behind single-card chance nodes, in float32, on the matrix cores.
//
// The value of such a node is the mean of the network's answers over the cards that can come
// (ChanceNodeHelper.single_card_chance_values, src/p2/search/chance_node_helper.py:360-479).  For a network of
// linear layers with ReLU between them whose input is [ranges of both players | one-hot of the board], three things
// follow from the algebra alone:
//   * the last layer is linear, so the mean over the cards is taken in front of it: 1/48 of its work;
//   * a sample's range is the state's without the 51 hands that hold the dealt card c, over the mass left:
//         W1 x_c = sum_p inv[p][c] * (T[p] - sum of the hands of p that hold c) + board columns,   T[p] = W1[p] t[p],
//     so the first layer is one product per state (1326 wide per player) and one of 102 columns per sample
//     instead of 2704 per sample;
//   * what is left is the hidden layers: samples x width x width multiply-adds each.
//
// Products in float32 accuracy at the rate of the 16-bit matrix instructions: a row is scaled by a power of two and
// every value kept as hi + lo, two float16 numbers that hold 22 bits of it together; a product of two rows is
// hi hi + hi lo + lo hi, added up in float32.  What is dropped (lo lo and the bits below lo) is 2^-22 of a product, below
// what adding 1536 of them in float32 rounds away: against 64 bits such a layer is 1.6e-7 off (norm over norm, 1536
// wide), the library's float32 product 5.0e-7.  The whole call, 3 x 1536, against 64 bits, before (library, mean of the
// answers) and now: 1.72e-7 / 1.61e-7 over Gamma(1/2) ranges, 1.91e-7 / 1.67e-7 over their eighth powers, 1.79e-7 /
// 1.65e-7 over single hands; with torch's own initial weights 1.12e-7 / 0.57e-7.  An answer's error is bounded against
// what its unit's weights can reach, not against the answer itself: hence a scale per unit (below), since units that
// share one lose their bits to the largest.
// 2240 states x 48 cards, 3 x 1536: 20.4 -> 3.7 ms (the hidden layers 1.36 + 1.59, the first 0.5).  Every call prepares
// all weights, which is what few samples pay for: 35 states 0.56 -> 0.27 ms, 1 state 0.19 -> 0.23 (the caller's rule,
// chance_node_helper.py, sends those through the layers).
//
// Numbers that are not finite stay so on the way through, but an infinity may turn into NaN (its low part does).
#pragma once
#include "common.h"
#include "unblocked.hip"
#include "chance.hip"

namespace p2 {

typedef _Float16 ln_half8 __attribute__((ext_vector_type(8)));
typedef _Float16 ln_half4 __attribute__((ext_vector_type(4)));
typedef float ln_float4 __attribute__((ext_vector_type(4)));

// Split rows: ceil(columns / 32) blocks of 128 bytes, 32 high parts then 32 low parts, so that one line holds both
// operands of a step of the product; columns past the end are zero.  A row r carries 1 / scale in its own array.
constexpr int LN_BLOCK_BYTES = 128;
constexpr int LN_RANGE_BLOCKS = (P2_H + 31) / 32;       // 42: a player's range
constexpr int LN_CARD_SLOTS = 2 * 51 + 1;               // hands of both players that hold a card, and the card itself
constexpr int LN_CARD_BLOCKS = 4;                       // 103 slots in 128
constexpr int LN_INPUT = CH_INPUT_WIDTH;                // 2704
constexpr int LN_MAX_LAYERS = 16;                       // equals P2HIP_NETWORK_MAX_LAYERS of include/p2hip.h
constexpr int64_t LN_MAX_SAMPLES = (1 << 23) - 1;       // P2HIP_NETWORK_MAX_SAMPLES: x 512 bytes stays below 2^32
constexpr float LN_SAMPLE_SCALE = 16384.0f;             // entries of a sample's input are at most 1

struct LnScale { float up, down; };
// Power of two that takes values of at most `bound` to at most 2^15 (float16 reaches 65504), and its inverse.
__device__ __forceinline__ LnScale ln_scale(float bound) {
  int e = 14 - ((int)((__builtin_bit_cast(uint32_t, bound) >> 23) & 255u) - 127);
  e = e > 100 ? 100 : (e < -100 ? -100 : e);
  return {__builtin_bit_cast(float, (uint32_t)(127 + e) << 23), __builtin_bit_cast(float, (uint32_t)(127 - e) << 23)};
}
__device__ __forceinline__ void ln_split(float y, _Float16& hi, _Float16& lo) {
  hi = (_Float16)y;
  lo = (_Float16)(y - (float)hi);
}
// Eight consecutive columns of a split row (`first` a multiple of 8).
__device__ __forceinline__ void ln_store8(char* row, int first, const float (&y)[8]) {
  ln_half8 hi, lo;
#pragma unroll
  for (int q = 0; q < 8; ++q) {
    _Float16 h, l;
    ln_split(y[q], h, l);
    hi[q] = h;
    lo[q] = l;
  }
  char* at = row + (first >> 5) * LN_BLOCK_BYTES + (first & 31) * 2;
  *reinterpret_cast<ln_half8*>(at) = hi;
  *reinterpret_cast<ln_half8*>(at + 64) = lo;
}
// Maximum over float bit patterns; `v` is not negative (and no -0).
__device__ __forceinline__ void ln_atomic_max(float* at, float v) {
  atomicMax(reinterpret_cast<unsigned*>(at), __builtin_bit_cast(unsigned, v));
}
// NaN stays NaN, like torch's relu.
__device__ __forceinline__ float ln_relu(float v) { return v < 0.f ? 0.f : v; }

// Largest float over a workgroup's threads; `red` holds one per wave.  Two barriers.
constexpr int LN_THREADS = 256;
__device__ __forceinline__ float ln_block_max(float v, float* red) {
  for (int off = 32; off; off >>= 1) v = fmaxf(v, __shfl_xor(v, off, 64));
  p2_sync_lds();
  if ((threadIdx.x & 63) == 0) red[threadIdx.x >> 6] = v;
  p2_sync_lds();
  return fmaxf(fmaxf(red[0], red[1]), fmaxf(red[2], red[3]));
}

// ---- weights ------------------------------------------------------------------------------------
// Two networks are the same function if a hidden unit's weights and bias are divided by a power of two u and the column
// that reads it is multiplied by u.  The network is computed as the one whose units all answer with about 1: a row of
// answers has ONE scale, and a unit far below the largest would lose its low bits to float16's smallest number (with
// units 2^N(0, 4) apart, 3 x 768: 8e-2 off, like this 4.4e-8 as with units of one size).  u is the power of two below
// sqrt(sum of absolute weights x largest) + bias, which lies between the weights' 2-norm and their sum: in the first layer
// the largest weight + bias.  A negative bias makes no answer larger and does not count, here or in a row's bound: a unit
// may be switched off by one of any size, -infinity too.  A unit that is always 0 gets the smallest u, so that what reads
// it sets no row's scale.
// A layer's weights are therefore prepared behind those of the layer in front of it.
__device__ __forceinline__ float ln_unit(float size) {
  int e = (int)((__builtin_bit_cast(uint32_t, size) >> 23) & 255u) - 127;
  e = e > 96 ? 96 : (e < -96 ? -96 : e);
  return __builtin_bit_cast(float, (uint32_t)(127 + e) << 23);
}
__device__ __forceinline__ float ln_inverse(float power_of_two) {
  return __builtin_bit_cast(float, 0x7F000000u - __builtin_bit_cast(uint32_t, power_of_two));
}

// A layer as its product needs it, a workgroup per row.  `inv`, `bias` and `bound` are those of the answers in units of u;
// `bound` is what an answer can reach for inputs of at most 1, without the bias (the sum of absolute weights).
struct LnLayerWeights {
  const float *w, *b;          // as given; b: none if the layer has no bias
  const float* column_unit;    // u of the units that the layer reads
  char* out;                   // split rows
  float *inv, *bound, *bias, *unit;
  int columns, hidden;         // the last layer's answers are not `hidden`: u = 1
};
__global__ __launch_bounds__(LN_THREADS) void ln_weights_kernel(LnLayerWeights a) {
  __shared__ float red[LN_THREADS / 64];
  __shared__ float red_sum[LN_THREADS / 64];
  const int64_t r = blockIdx.x;
  const int units = a.columns / 8;                        // columns are a multiple of 32
  const float4* src = reinterpret_cast<const float4*>(a.w + r * a.columns);
  const float4* of = reinterpret_cast<const float4*>(a.column_unit);
  auto load = [&](int u) {
    const float4 v = src[u], c = of[u];
    return make_float4(v.x * c.x, v.y * c.y, v.z * c.z, v.w * c.w);
  };
  float mx = 0.f, l1 = 0.f;
  for (int u = threadIdx.x; u < units; u += LN_THREADS)
#pragma unroll
    for (int q = 0; q < 2; ++q) {
      const float4 v = load(2 * u + q);
      mx = fmaxf(fmaxf(mx, fmaxf(fabsf(v.x), fabsf(v.y))), fmaxf(fabsf(v.z), fabsf(v.w)));
      l1 += (fabsf(v.x) + fabsf(v.y)) + (fabsf(v.z) + fabsf(v.w));
    }
  l1 = p2_wave_sum(l1);
  if ((threadIdx.x & 63) == 0) red_sum[threadIdx.x >> 6] = l1;
  mx = ln_block_max(mx, red);
  const LnScale s = ln_scale(mx);
  if (threadIdx.x == 0) {
    const float sum = (red_sum[0] + red_sum[1]) + (red_sum[2] + red_sum[3]), b = a.b ? a.b[r] : 0.f;
    const float unit = a.hidden ? ln_unit(sqrtf(sum) * sqrtf(mx) + fmaxf(b, 0.f)) : 1.0f, down = ln_inverse(unit);
    a.inv[r] = s.down * down;
    a.bound[r] = sum * down;
    a.bias[r] = b * down;
    a.unit[r] = unit;
  }
  char* out = a.out + r * (units / 4) * (int64_t)LN_BLOCK_BYTES;
  for (int u = threadIdx.x; u < units; u += LN_THREADS) {
    const float4 v = load(2 * u), w = load(2 * u + 1);
    const float y[8] = {v.x * s.up, v.y * s.up, v.z * s.up, v.w * s.up, w.x * s.up, w.y * s.up, w.z * s.up, w.w * s.up};
    ln_store8(out, 8 * u, y);
  }
}

// The first layer [width, 2704], a row cut up the way its products need it, all of it under one scale:
//   ranges  [2][width] split rows of 1326 columns, a player each;
//   cards   [52][width] split rows of 103 columns: the hands of player 0, then of player 1, that hold the card (in the
//           order of the partner card), then the card's own board column;
//   board   [52][width] float: the board columns, in units of u.
// `bound`: a sample's ranges add up to 1 each and its board holds at most five cards, seven times the largest weight.
// A few more workgroups clear the maxima that are kept below.
struct LnFirstWeights {
  LnLayerWeights layer;        // without `out`, `column_unit`
  char *ranges, *cards;
  float* board;
  uint4* clear;
  int64_t clear_units;
  int width, clear_blocks;
};
__global__ __launch_bounds__(LN_THREADS) void ln_first_weights_kernel(LnFirstWeights a) {
  __shared__ __align__(16) float row[LN_INPUT];
  __shared__ float red[LN_THREADS / 64];
  if ((int)blockIdx.x >= a.width) {
    for (int64_t k = (int64_t)((int)blockIdx.x - a.width) * LN_THREADS + threadIdx.x; k < a.clear_units;
         k += (int64_t)a.clear_blocks * LN_THREADS)
      a.clear[k] = make_uint4(0u, 0u, 0u, 0u);
    return;
  }
  const int64_t n = blockIdx.x, width = a.width;
  const float4* src = reinterpret_cast<const float4*>(a.layer.w + n * LN_INPUT);
  float mx = 0.f;
  for (int k = threadIdx.x; k < LN_INPUT / 4; k += LN_THREADS) {
    const float4 v = src[k];
    reinterpret_cast<float4*>(row)[k] = v;
    mx = fmaxf(fmaxf(mx, fmaxf(fabsf(v.x), fabsf(v.y))), fmaxf(fabsf(v.z), fabsf(v.w)));
  }
  mx = ln_block_max(mx, red);                             // its barriers cover `row` too
  const LnScale s = ln_scale(mx);
  const float b = a.layer.b ? a.layer.b[n] : 0.f, unit = ln_unit(mx + fmaxf(b, 0.f)), down = ln_inverse(unit);
  if (threadIdx.x == 0) {
    a.layer.inv[n] = s.down * down;
    a.layer.bound[n] = 7.f * (mx * down);
    a.layer.bias[n] = b * down;
    a.layer.unit[n] = unit;
  }
  for (int u = threadIdx.x; u < 2 * LN_RANGE_BLOCKS * 4; u += LN_THREADS) {
    const int p = u / (LN_RANGE_BLOCKS * 4), f = 8 * (u - p * (LN_RANGE_BLOCKS * 4));
    float y[8];
#pragma unroll
    for (int q = 0; q < 8; ++q) y[q] = f + q < P2_H ? row[p * P2_H + f + q] * s.up : 0.f;
    ln_store8(a.ranges + (p * width + n) * (LN_RANGE_BLOCKS * LN_BLOCK_BYTES), f, y);
  }
  for (int u = threadIdx.x; u < P2_CARDS * LN_CARD_BLOCKS * 4; u += LN_THREADS) {
    const int c = u / (LN_CARD_BLOCKS * 4), f = 8 * (u - c * (LN_CARD_BLOCKS * 4));
    float y[8];
#pragma unroll
    for (int q = 0; q < 8; ++q) {
      const int slot = f + q, p = slot >= 51, j = slot - 51 * p, other = j + (j >= c);
      float v = 0.f;
      if (slot < 102) v = row[p * P2_H + (other < c ? p2_combo_index(other, c) : p2_combo_index(c, other))];
      else if (slot == 102) v = row[2 * P2_H + c];
      y[q] = v * s.up;
    }
    ln_store8(a.cards + (c * width + n) * (LN_CARD_BLOCKS * LN_BLOCK_BYTES), f, y);
  }
  if (threadIdx.x < P2_CARDS) a.board[threadIdx.x * width + n] = row[2 * P2_H + threadIdx.x] * down;
}

// What is known of a sample.  `inv`: 1 / the mass left to a player, -1 where the uniform range takes its place.
struct LnSample {
  float inv0, inv1;
  int32_t state;   // among the call's states
  int32_t card;    // the dealt card, -1: no card is left to deal (input all zero)
};

// A player's hands with the dealt card may hold nearly all of his mass.  T minus their share would then cancel: above
// this share the sample is taken whole (`ln_whole_kernel`), at most seven cards per player.
constexpr double LN_HEAVY_SHARE = 0.25;

// One workgroup per state: the ranges without the board's hands as split rows [2][states], and for each of its samples
// the first layer's inputs that leave with the card, its weights and its place.  A range without any mass (at most
// 1e-12) is the uniform one in every sample; it is written as such.
__global__ __launch_bounds__(LN_THREADS) void ln_states_kernel(
    const float* __restrict__ pre_beliefs, const int64_t* __restrict__ root_indices, const int64_t* __restrict__ board,
    const int64_t* __restrict__ sample_offsets, int64_t source_rows, int64_t total_samples, char* __restrict__ ranges,
    float* __restrict__ ranges_inv, char* __restrict__ gone, float2* __restrict__ weight, LnSample* __restrict__ samples,
    int32_t* __restrict__ row_of, int32_t* __restrict__ whole, int32_t* __restrict__ whole_count) {
  __shared__ __align__(16) float t[2 * P2_H + CH_LDS_PAD];
  __shared__ double cs[2 * P2_CARDS];
  __shared__ float red[LN_THREADS / 64];
  __shared__ float2 w_of[P2_CARDS];
  const int64_t i = blockIdx.x, n = gridDim.x;
  const int64_t root = root_indices ? root_indices[i] : i;
  const bool in_table = root >= 0 && root < source_rows;
  int bcards[5];
  uint64_t bits = 0;
  const int ncards = in_table ? chance_board(board + root * 5, bcards, bits) : 5;
  const int have = ncards < 5 ? P2_CARDS - ncards : 0;
  int64_t s0 = sample_offsets[i], s1 = sample_offsets[i + 1];
  if (s0 < 0) s0 = 0;
  if (s1 > total_samples) s1 = total_samples;
  for (int k = threadIdx.x; k < 2 * P2_H; k += LN_THREADS) {
    const int h = k >= P2_H ? k - P2_H : k;
    const bool off = ((bits >> p2_combo.a[h]) | (bits >> p2_combo.b[h])) & 1ull;
    t[k] = off || have == 0 ? 0.f : pre_beliefs[root * (2 * P2_H) + k];
  }
  p2_sync_lds();
  card_sums_multi(t, P2_H, 2, cs);
  const double total[2] = {card_total(cs), card_total(cs + P2_CARDS)};
  const int left = P2_CARDS - ncards - 1;               // cards left for the hands of a sample
  const float uniform = 1.0f / fmaxf((float)(left * (left - 1) / 2), 1.0f);
  const bool empty[2] = {!((float)total[0] > 1e-12f), !((float)total[1] > 1e-12f)};
  p2_sync_lds();                                        // card_sums_multi reads t
  float mx[2] = {0.f, 0.f};
  for (int k = threadIdx.x; k < 2 * P2_H; k += LN_THREADS) {
    const int p = k >= P2_H, h = k - p * P2_H;
    if (empty[p]) t[k] = (((bits >> p2_combo.a[h]) | (bits >> p2_combo.b[h])) & 1ull) || have == 0 ? 0.f : 1.f;
    mx[p] = fmaxf(mx[p], fabsf(t[k]));
  }
  // the samples: cards off the board in ascending order, then what is left of the state's share
  if (threadIdx.x < P2_CARDS) {
    const int c = threadIdx.x;
    const bool dealt = (bits >> c) & 1ull;
    const int64_t s = s0 + c - __popcll(bits & ((1ull << c) - 1ull));
    const bool there = have > 0 && !dealt && s < s1;
    row_of[c * n + i] = there ? (int32_t)s : -1;
    if (there) {
      float inv[2];
      bool heavy = false;
      float2 wt;
#pragma unroll
      for (int p = 0; p < 2; ++p) {
        const float sum = (float)(total[p] - cs[p * P2_CARDS + c]);
        const bool ok = sum > 1e-12f;
        inv[p] = ok ? 1.0f / fmaxf(sum, 1e-12f) : -1.0f;
        // (negated, so that a NaN makes the sample a whole one)
        heavy = heavy || (!empty[p] && !(ok && cs[p * P2_CARDS + c] <= LN_HEAVY_SHARE * total[p]));
        (p ? wt.y : wt.x) = empty[p] ? uniform : inv[p];
      }
      if (heavy) {
        wt = make_float2(0.f, 0.f);
        whole[atomicAdd(whole_count, 1)] = (int32_t)s;
      }
      w_of[c] = wt;
      weight[s] = wt;
      samples[s] = LnSample{inv[0], inv[1], (int32_t)i, c};
    }
  }
  for (int64_t s = s0 + have + threadIdx.x; s < s1; s += LN_THREADS) {
    weight[s] = make_float2(0.f, 0.f);
    samples[s] = LnSample{0.f, 0.f, (int32_t)i, -1};
    whole[atomicAdd(whole_count, 1)] = (int32_t)s;
  }
#pragma unroll
  for (int p = 0; p < 2; ++p) {
    const LnScale s = ln_scale(ln_block_max(mx[p], red));   // (its barriers cover t and w_of too)
    if (threadIdx.x == 0) ranges_inv[p * n + i] = s.down;
    for (int u = threadIdx.x; u < LN_RANGE_BLOCKS * 4; u += LN_THREADS) {
      float y[8];
#pragma unroll
      for (int q = 0; q < 8; ++q) y[q] = 8 * u + q < P2_H ? t[p * P2_H + 8 * u + q] * s.up : 0.f;
      ln_store8(ranges + (p * n + i) * (LN_RANGE_BLOCKS * LN_BLOCK_BYTES), 8 * u, y);
    }
  }
  // what leaves with card c: the weighted hands that hold it; the card's own board column comes in, so it counts -1
  for (int u = threadIdx.x; u < P2_CARDS * LN_CARD_BLOCKS * 4; u += LN_THREADS) {
    const int c = u / (LN_CARD_BLOCKS * 4), f = 8 * (u - c * (LN_CARD_BLOCKS * 4));
    const int64_t s = s0 + c - __popcll(bits & ((1ull << c) - 1ull));
    if (have == 0 || ((bits >> c) & 1ull) || s >= s1) continue;
    const float2 wt = w_of[c];
    float y[8];
#pragma unroll
    for (int q = 0; q < 8; ++q) {
      const int slot = f + q, p = slot >= 51, j = slot - 51 * p, other = j + (j >= c);
      float v = 0.f;
      if (slot < 102)
        v = t[p * P2_H + (other < c ? p2_combo_index(other, c) : p2_combo_index(c, other))] * (p ? wt.y : wt.x);
      else if (slot == 102)
        v = -1.f;
      y[q] = v * LN_SAMPLE_SCALE;
    }
    ln_store8(gone + s * (LN_CARD_BLOCKS * LN_BLOCK_BYTES), f, y);
  }
}

// Workgroup l of the first `layers`: stats[2 l], stats[2 l + 1] = the largest bound and bias (0 at least) of layer l.  The
// others, a state each: base[i][n] = the first layer's bias + the columns of the cards on the state's board.
struct LnBounds {
  const float *bound[LN_MAX_LAYERS], *bias[LN_MAX_LAYERS];   // in units of u
  int rows[LN_MAX_LAYERS];
};
__global__ __launch_bounds__(LN_THREADS) void ln_base_kernel(LnBounds bounds, int layers, float* __restrict__ stats,
                                                              const int64_t* __restrict__ root_indices,
                                                              const int64_t* __restrict__ board, int64_t source_rows,
                                                              const float* __restrict__ columns, int width,
                                                              float* __restrict__ base) {
  __shared__ float red[LN_THREADS / 64];
  if ((int)blockIdx.x < layers) {
    const int l = blockIdx.x;
    const float *bound = bounds.bound[l], *bias = bounds.bias[l];
    float m = 0.f, b = 0.f;
    for (int k = threadIdx.x; k < bounds.rows[l]; k += LN_THREADS) {
      m = fmaxf(m, bound[k]);
      b = fmaxf(b, bias[k]);
    }
    m = ln_block_max(m, red);
    b = ln_block_max(b, red);
    if (threadIdx.x == 0) { stats[2 * l] = m; stats[2 * l + 1] = b; }
    return;
  }
  const int64_t i = blockIdx.x - layers;
  const int64_t root = root_indices ? root_indices[i] : i;
  int bcards[5];
  uint64_t bits = 0;
  if (root >= 0 && root < source_rows) chance_board(board + root * 5, bcards, bits);
  for (int k = threadIdx.x; k < width; k += LN_THREADS) {
    float v = bounds.bias[0][k];
    for (uint64_t b = bits; b; b &= b - 1) v += columns[(__ffsll((unsigned long long)b) - 1) * width + k];
    base[i * width + k] = v;
  }
}

// ---- the product --------------------------------------------------------------------------------
enum { LN_PLAIN = 0, LN_HIDDEN = 1, LN_MEAN = 2 };

struct LnGemm {
  const char* a;            // split rows [m] (LN_PLAIN: [batch][m]): the layer's input
  const char* b;            // split rows [n] (LN_PLAIN: [batch][n]): its weights
  const float* a_inv;       // [m] (LN_PLAIN: [batch][m])
  const float* b_inv;       // [n]
  const float* bias;        // [n] or none
  int64_t m;
  int n, blocks, batches;
  float* out;               // LN_PLAIN: [batch][m][n]
  // LN_HIDDEN: the next layer's input.  An answer is at most stats[0] * (largest entry of the input) + stats[1], the
  // input at most a_max[row] or, without that, first_stats[0] + first_stats[1].
  const float *stats, *first_stats, *a_max;
  char* out_split;
  float* out_inv;
  float* out_max;           // [m], largest entry of a row, starts at zero; none if no hidden layer but the last follows
  // LN_MEAN: sums over the samples of each state
  const int64_t* offsets;
  int64_t states;
  double *sums, *parts;
};

__device__ __forceinline__ void ln_to_lds(const char* from, char* to) {   // 16 bytes per lane, to `to` + 16 * lane
  __builtin_amdgcn_global_load_lds((const __attribute__((address_space(1))) uint32_t*)from,
                                   (__attribute__((address_space(3))) uint32_t*)to, 16, 0, 0);
}

// C = A B^T over split rows; a workgroup of WM x WN waves makes a tile of (WM TM 16) x (WN TN 16), a wave TM x TN
// squares of 16 x 16 (`v_mfma_f32_16x16x32_f16`).  The weights are the instruction's first operand, so a lane holds
// one row of the layer's input and four neighbouring columns of its answer.
// A step is one 128-byte block of every row, fetched straight into LDS one step ahead of its use; 16-byte chunk q of
// row r lies in place q ^ (r / 2 & 7), so that sixteen rows read at once meet in no bank (with r & 7 half of the LDS
// cycles were conflicts: 1.51 -> 1.37 ms).  The loads are pinned in front of the step's 96 products per wave, or the
// compiler puts them behind, next to the barrier that waits for them.
// The three products of a step start from zero and are added to the sum by the vector ALU, a row of squares behind the
// matrix instructions: added up inside them the result is 4.4e-7 off, like this 1.6e-7, for 8 % of the time.  LN_PLAIN
// (few rows, and the layer whose error nothing averages) also keeps sums of 256 columns apart and takes lo lo along.
// 107 520 x 1536 x 1536, 6 x as many float16 operations: 1.36-1.41 ms = 1075-1121 TFLOP/s (32 x 32 squares, one sum 1.37;
// 16 x 16, one sum 1.27; the library's float32 product 3.6-3.7 ms, its plain bfloat16 products reach 1144 on this card).
// Bound: the card's power; it runs them at 1.8-2.0 GHz, the matrix cores busy 53-57 % of the cycles, no bank conflicts.
// 256 x 256 tiles need 128 KiB of LDS (one workgroup per CU); 128 x 128 tiles make it 1.93 ms at that size, but 2240 x
// 2652 x 1536 goes from 0.109 to 0.067 and 8192 x 1536 x 1536 from 0.118 to 0.112 (first version): the smaller tile below
// four large ones per CU, and 64 x 64 where even those leave CUs idle.
template <int EPI, int WM, int WN, int TM, int TN>
__global__ __launch_bounds__(WM * WN * 64, 2) void ln_gemm_kernel(LnGemm g) {
  constexpr int BM = WM * TM * 16, BN = WN * TN * 16, NW = WM * WN;
  constexpr int LA = BM / 8 / NW, LB = BN / 8 / NW;      // 1 KiB pieces (8 rows) a wave fetches per step
  static_assert(LA >= 1 && LB >= 1 && TM % 2 == 0 && BM * TN * 16 * 4 <= (BM + BN) * LN_BLOCK_BYTES, "tile");
  __shared__ __align__(128) char buf0[(BM + BN) * LN_BLOCK_BYTES];
  __shared__ __align__(128) char buf1[(BM + BN) * LN_BLOCK_BYTES];
  const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int wm = wave / WN, wn = wave % WN;
  // Workgroup b runs on XCD b mod 8: each XCD gets a run of neighbouring tiles, the columns of one stripe of rows
  // first, so they share operands in its L2.
  const unsigned tiles = gridDim.x, xcd = blockIdx.x & 7, per = tiles >> 3, more = tiles & 7;
  unsigned tile = xcd * per + (xcd < more ? xcd : more) + (blockIdx.x >> 3);
  const unsigned tiles_n = (unsigned)((g.n + BN - 1) / BN);
  const unsigned tiles_m = (unsigned)((g.m + BM - 1) / BM);
  const unsigned tn = tile % tiles_n, tm = tile / tiles_n % tiles_m, batch = tile / tiles_n / tiles_m;
  const int64_t m0 = (int64_t)tm * BM;
  const int n0 = (int)tn * BN;
  const int row_bytes = g.blocks * LN_BLOCK_BYTES;
  const int rows_left = (int)(g.m - m0 < BM ? g.m - m0 : BM), cols_left = g.n - n0 < BN ? g.n - n0 : BN;

  // rows past the end are read as the last one and never stored
  uint32_t off_a[LA], off_b[LB];
#pragma unroll
  for (int i = 0; i < LA; ++i) {
    int r = wave * (BM / NW) + i * 8 + (lane >> 3);
    const uint32_t chunk = (uint32_t)(((lane & 7) ^ ((r >> 1) & 7)) * 16);
    r = r < rows_left ? r : rows_left - 1;
    off_a[i] = (uint32_t)r * (uint32_t)row_bytes + chunk;
  }
#pragma unroll
  for (int i = 0; i < LB; ++i) {
    int r = wave * (BN / NW) + i * 8 + (lane >> 3);
    const uint32_t chunk = (uint32_t)(((lane & 7) ^ ((r >> 1) & 7)) * 16);
    r = r < cols_left ? r : cols_left - 1;
    off_b[i] = (uint32_t)r * (uint32_t)row_bytes + chunk;
  }
  const char* pa = g.a + ((int64_t)(EPI == LN_PLAIN ? batch : 0) * g.m + m0) * row_bytes;
  const char* pb = g.b + ((int64_t)(EPI == LN_PLAIN ? batch : 0) * g.n + n0) * row_bytes;

  auto fetch = [&](char* buf, int block) {
    const int64_t at = (int64_t)block * LN_BLOCK_BYTES;
#pragma unroll
    for (int i = 0; i < LA; ++i) ln_to_lds(pa + at + off_a[i], buf + (wave * (BM / NW) + i * 8) * LN_BLOCK_BYTES);
#pragma unroll
    for (int i = 0; i < LB; ++i)
      ln_to_lds(pb + at + off_b[i], buf + (BM + wave * (BN / NW) + i * 8) * LN_BLOCK_BYTES);
    __builtin_amdgcn_sched_barrier(0);
  };
  ln_float4 acc[TM][TN] = {};
  const int fr = lane & 15, fq = lane >> 4, turn = (fr >> 1) & 7;
  auto multiply = [&](const char* buf) {
    const int ch = (fq ^ turn) * 16, cl = ((4 + fq) ^ turn) * 16;
    const char* la = buf + (wm * TM * 16 + fr) * LN_BLOCK_BYTES;
    const char* lb = buf + (BM + wn * TN * 16 + fr) * LN_BLOCK_BYTES;
    ln_half8 wh[TN], wl[TN], xh[TM], xl[TM];
    auto take = [&](int i) {
      xh[i] = *reinterpret_cast<const ln_half8*>(la + i * 16 * LN_BLOCK_BYTES + ch);
      xl[i] = *reinterpret_cast<const ln_half8*>(la + i * 16 * LN_BLOCK_BYTES + cl);
    };
#pragma unroll
    for (int j = 0; j < TN; ++j) {
      wl[j] = *reinterpret_cast<const ln_half8*>(lb + j * 16 * LN_BLOCK_BYTES + cl);
      wh[j] = *reinterpret_cast<const ln_half8*>(lb + j * 16 * LN_BLOCK_BYTES + ch);
    }
    take(0);
#pragma unroll
    for (int i = 0; i < TM; ++i) {
      if (i + 1 < TM) take(i + 1);
      ln_float4 t[TN];
#pragma unroll
      for (int j = 0; j < TN; ++j)
        t[j] = EPI == LN_PLAIN ? __builtin_amdgcn_mfma_f32_16x16x32_f16(wl[j], xl[i], ln_float4{}, 0, 0, 0) : ln_float4{};
#pragma unroll
      for (int j = 0; j < TN; ++j) t[j] = __builtin_amdgcn_mfma_f32_16x16x32_f16(wl[j], xh[i], t[j], 0, 0, 0);
#pragma unroll
      for (int j = 0; j < TN; ++j) t[j] = __builtin_amdgcn_mfma_f32_16x16x32_f16(wh[j], xl[i], t[j], 0, 0, 0);
#pragma unroll
      for (int j = 0; j < TN; ++j) t[j] = __builtin_amdgcn_mfma_f32_16x16x32_f16(wh[j], xh[i], t[j], 0, 0, 0);
#pragma unroll
      for (int j = 0; j < TN; ++j) acc[i][j] += t[j];
    }
  };
  ln_float4 whole[EPI == LN_PLAIN ? TM : 1][EPI == LN_PLAIN ? TN : 1] = {};
  auto carry = [&]() {
    if constexpr (EPI == LN_PLAIN) {
#pragma unroll
      for (int i = 0; i < TM; ++i)
#pragma unroll
        for (int j = 0; j < TN; ++j) {
          whole[i][j] += acc[i][j];
          acc[i][j] = ln_float4{};
        }
    }
  };
  fetch(buf0, 0);
  int kb = 0;
  for (; kb + 2 <= g.blocks; kb += 2) {
    p2_sync_loads();                                       // block kb is there, and everyone is done with buf1
    fetch(buf1, kb + 1);
    multiply(buf0);
    p2_sync_loads();
    fetch(buf0, kb + 2 < g.blocks ? kb + 2 : kb + 1);      // past the end: a block nobody uses
    multiply(buf1);
    if ((kb & 6) == 6) carry();
  }
  p2_sync_loads();
  if (kb < g.blocks) multiply(buf0);
  carry();

  // ---- what becomes of the tile: acc[i][j][e] is row (wm TM + i) 16 + fr, column (wn TN + j) 16 + 4 fq + e
  if constexpr (EPI != LN_MEAN) {
    // 32 rows at a time go through the wave's own 32 x (16 TN) floats of LDS, so that its lanes then hold whole runs of
    // a row and their stores cover whole lines.
    constexpr int COLS = TN * 16, CHUNKS = COLS / 4, ROWS = 64 / CHUNKS;
    static_assert(NW * 32 * COLS * 4 <= (int)sizeof(buf0), "a stage per wave");
    char* stage = buf0 + wave * 32 * COLS * 4;
    const int chunk = lane & (CHUNKS - 1), n = n0 + wn * COLS + chunk * 4;
    const bool in = n < g.n;                               // g.n is a multiple of 4 (of 32 if the answer is split rows)
    const float4 bi = in ? *reinterpret_cast<const float4*>(g.b_inv + n) : make_float4(0.f, 0.f, 0.f, 0.f);
    const float4 c4 = in && g.bias ? *reinterpret_cast<const float4*>(g.bias + n) : make_float4(0.f, 0.f, 0.f, 0.f);
    float s0 = 0.f, s1 = 0.f, bound0 = 0.f;
    if constexpr (EPI == LN_HIDDEN) {
      s0 = g.stats[0];
      s1 = g.stats[1];
      if (!g.a_max) bound0 = g.first_stats[0] + g.first_stats[1];
    }
    __syncthreads();                                       // everyone is done with the last block
#pragma unroll
    for (int half = 0; half < TM / 2; ++half) {
#pragma unroll
      for (int i = 2 * half; i < 2 * half + 2; ++i)
#pragma unroll
        for (int j = 0; j < TN; ++j) {
          const int rr = (i & 1) * 16 + fr;
          const ln_float4 v = EPI == LN_PLAIN ? whole[EPI == LN_PLAIN ? i : 0][EPI == LN_PLAIN ? j : 0] : acc[i][j];
          *reinterpret_cast<ln_float4*>(stage + rr * COLS * 4 + (((j * 4 + fq) ^ (rr & (CHUNKS - 1))) << 4)) = v;
        }
      __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
      __builtin_amdgcn_wave_barrier();
#pragma unroll
      for (int it = 0; it < 32 / ROWS; ++it) {
        const int rr = it * ROWS + lane / CHUNKS, r = wm * TM * 16 + half * 32 + rr;
        const float4 a4 = *reinterpret_cast<const float4*>(stage + rr * COLS * 4 + ((chunk ^ (rr & (CHUNKS - 1))) << 4));
        if (r >= rows_left) continue;
        if constexpr (EPI == LN_PLAIN) {
          if (!in) continue;
          const int64_t row = (int64_t)batch * g.m + m0 + r;
          const float ai = g.a_inv[row];
          *reinterpret_cast<float4*>(g.out + row * g.n + n) = make_float4(
              a4.x * ai * bi.x + c4.x, a4.y * ai * bi.y + c4.y, a4.z * ai * bi.z + c4.z, a4.w * ai * bi.w + c4.w);
        } else {
          const int64_t row = m0 + r;
          const float ai = g.a_inv[row];
          const LnScale s = ln_scale((g.a_max ? g.a_max[row] : bound0) * s0 + s1);
          float v[4] = {a4.x * ai * bi.x + c4.x, a4.y * ai * bi.y + c4.y, a4.z * ai * bi.z + c4.z, a4.w * ai * bi.w + c4.w};
          ln_half4 hi, lo;
          float mx = 0.f;
#pragma unroll
          for (int e = 0; e < 4; ++e) {
            v[e] = ln_relu(v[e]);
            mx = v[e] > mx ? v[e] : mx;                    // (never -0)
            _Float16 h, l;
            ln_split(v[e] * s.up, h, l);
            hi[e] = h;
            lo[e] = l;
          }
          // neighbouring lanes hold eight columns: the even one stores their high parts, the odd one the low parts
          const uint2 uh = __builtin_bit_cast(uint2, hi), ul = __builtin_bit_cast(uint2, lo);
          const bool odd = lane & 1;
          const uint2 mine = odd ? uh : ul;
          const uint2 other = make_uint2((uint32_t)__builtin_amdgcn_update_dpp(0, (int)mine.x, 0xB1, 0xF, 0xF, false),
                                         (uint32_t)__builtin_amdgcn_update_dpp(0, (int)mine.y, 0xB1, 0xF, 0xF, false));
          char* at = g.out_split + row * ((int64_t)(g.n / 32) * LN_BLOCK_BYTES) + (n >> 5) * LN_BLOCK_BYTES;
          if (in)
            *reinterpret_cast<uint4*>(at + (odd ? 64 + (n & 31) * 2 - 8 : (n & 31) * 2)) =
                odd ? make_uint4(other.x, other.y, ul.x, ul.y) : make_uint4(uh.x, uh.y, other.x, other.y);
          if (n == 0) g.out_inv[row] = s.down;
          if (g.out_max) {
            // largest of the row's columns: pairs, quads, halves of a row of 16 lanes, the row
            mx = in ? mx : 0.f;
            mx = fmaxf(mx, p2_dpp0<0xB1>(mx));
            mx = fmaxf(mx, p2_dpp0<0x4E>(mx));
            mx = fmaxf(mx, p2_dpp0<0x141>(mx));
            if (CHUNKS == 16) mx = fmaxf(mx, p2_dpp0<0x140>(mx));
            if (chunk == 0) ln_atomic_max(g.out_max + row, mx);
          }
        }
      }
      __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
      __builtin_amdgcn_wave_barrier();
    }
  }
  if constexpr (EPI == LN_MEAN) {
    // A column of waves at a time puts its part of the tile into LDS; then every wave adds up rows of whole states, in
    // row order.  What is complete inside the tile goes to sums[state], the piece of a state that began in an earlier
    // tile to parts[tile][0], the piece of one that goes on in the next to parts[tile][1].
    const int64_t m_end = m0 + rows_left;
    int64_t lo = 0, hi = g.states;                         // the state that row m0 belongs to
    while (hi - lo > 1) {
      const int64_t mid = (lo + hi) >> 1;
      if (g.offsets[mid] <= m0) lo = mid; else hi = mid;
    }
    constexpr int COLS = TN * 16, CHUNKS = COLS / 4;
#pragma unroll
    for (int pass = 0; pass < WN; ++pass) {
      char* stage = pass & 1 ? buf1 : buf0;
      __syncthreads();                                     // (the products above read both)
      if (wn == pass) {
#pragma unroll
        for (int j = 0; j < TN; ++j) {
          const int n = n0 + (wn * TN + j) * 16 + fq * 4;
          const bool in = n < g.n;
          const float4 bi = in ? *reinterpret_cast<const float4*>(g.b_inv + n) : make_float4(0.f, 0.f, 0.f, 0.f);
          const float4 c = in && g.bias ? *reinterpret_cast<const float4*>(g.bias + n) : make_float4(0.f, 0.f, 0.f, 0.f);
#pragma unroll
          for (int i = 0; i < TM; ++i) {
            const int r = (wm * TM + i) * 16 + fr;
            const float ai = r < rows_left ? g.a_inv[m0 + r] : 0.f;
            *reinterpret_cast<float4*>(stage + r * COLS * 4 + (((j * 4 + fq) ^ (r & (CHUNKS - 1))) << 4)) =
                make_float4(ln_relu(acc[i][j][0] * ai * bi.x + c.x), ln_relu(acc[i][j][1] * ai * bi.y + c.y),
                            ln_relu(acc[i][j][2] * ai * bi.z + c.z), ln_relu(acc[i][j][3] * ai * bi.w + c.w));
          }
        }
      }
      __syncthreads();
      const int col = lane & (COLS - 1), n = n0 + pass * COLS + col;
      auto staged = [&](int r) {
        return *reinterpret_cast<const float*>(stage + r * COLS * 4 + (((col >> 2) ^ (r & (CHUNKS - 1))) << 4) + (col & 3) * 4);
      };
      if (lane < COLS && n < g.n) {
        for (int64_t i = lo + wave; i < g.states; i += NW) {
          const int64_t o0 = g.offsets[i], o1 = g.offsets[i + 1];
          if (o0 >= m_end) break;
          const int r0 = (int)(o0 > m0 ? o0 - m0 : 0), r1 = (int)(o1 < m_end ? o1 - m0 : rows_left);
          // eight sums side by side: added up one after the other, 48 rows leave a rounding of 1e-7 (and their
          // LDS reads would wait for each other)
          float part[8] = {};
          int r = r0;
          for (; r + 8 <= r1; r += 8)
#pragma unroll
            for (int k = 0; k < 8; ++k) part[k] += staged(r + k);
#pragma unroll
          for (int k = 0; k < 7; ++k)
            if (r + k < r1) part[k] += staged(r + k);
          double sum = 0.0;
#pragma unroll
          for (int k = 0; k < 8; ++k) sum += (double)part[k];
          if (o0 >= m0 && o1 <= m_end) g.sums[i * g.n + n] = sum;
          else g.parts[((int64_t)tm * 2 + (o0 < m0 ? 0 : 1)) * g.n + n] = sum;
        }
      }
    }
  }
}

// The first layer's answers.  A workgroup keeps T of both players and the base of 64 states x 128 columns (registers, LDS)
// and goes through its cards: a product of 103 columns, the card's rows of `gone` against the card's columns of the
// weights, one 128-byte block of every row at a time as above, the next one (of the next card too) sent ahead.  (In two of
// a card's four steps the compiler cannot tell the buffers apart and waits for those loads before it reads the step's
// operands; they overlap with the products in the other two only.)  T read again for every card, as the epilogue of a
// product over cards, made the layer 560-590 us at 2240 states x 48 cards x 1536 (830 us with 16-byte loads of sixteen rows
// at a time), this 505-515; the matrix cores are busy 12 % of it.
// The cards are dealt to as many workgroups as fill the chip twice; those of one stripe of columns follow each other on
// one XCD and share the weights in its L2.
struct LnFirst {
  const char *gone, *cards;     // [samples], [52][width]
  const float *b_inv, *products, *base, *stats;
  const float2* weight;
  const int32_t* row_of;        // [52][states]
  int64_t states;
  int width, groups;
  char* out_split;
  float* out_inv;
};
constexpr int LN_FIRST_ROWS = 64, LN_FIRST_COLS = 128, LN_FIRST_THREADS = 512;
__global__ __launch_bounds__(LN_FIRST_THREADS, 4) void ln_first_kernel(LnFirst g) {
  constexpr int TM = 2, TN = 2, BM = LN_FIRST_ROWS, BN = LN_FIRST_COLS;
  constexpr int ROW_BYTES = LN_CARD_BLOCKS * LN_BLOCK_BYTES;
  __shared__ __align__(128) char buf0[(BM + BN) * LN_BLOCK_BYTES];
  __shared__ __align__(128) char buf1[(BM + BN) * LN_BLOCK_BYTES];
  __shared__ ln_float4 base_of[TM * TN][LN_FIRST_THREADS];  // a lane's own values: 80 KiB in all, two workgroups per CU
  const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int wm = wave >> 2, wn = wave & 3;                 // waves 2 x 4, 32 x 32 each
  const unsigned tiles = gridDim.x, xcd = blockIdx.x & 7, per = tiles >> 3, more = tiles & 7;
  const unsigned tile = xcd * per + (xcd < more ? xcd : more) + (blockIdx.x >> 3);
  const unsigned tiles_m = (unsigned)((g.states + BM - 1) / BM);
  const unsigned tm = tile % tiles_m, group = tile / tiles_m % g.groups, tn = tile / tiles_m / g.groups;
  const int64_t m0 = (int64_t)tm * BM;
  const int n0 = (int)tn * BN;
  const int rows_left = (int)(g.states - m0 < BM ? g.states - m0 : BM), cols_left = g.width - n0 < BN ? g.width - n0 : BN;
  const int c0 = (int)(group * P2_CARDS / g.groups), c1 = (int)((group + 1) * P2_CARDS / g.groups);

  // fetches: thread k takes 16 bytes of row k / 8 of the samples, and of rows k / 8 and 64 + k / 8 of the weights
  const int fetch_row = wave * 8 + (lane >> 3);
  const uint32_t chunk = (uint32_t)(((lane & 7) ^ ((fetch_row >> 1) & 7)) * 16);
  const int64_t state_row = m0 + (fetch_row < rows_left ? fetch_row : rows_left - 1);
  uint32_t off_b[2];
#pragma unroll
  for (int i = 0; i < 2; ++i) {
    const int r = fetch_row + 64 * i;
    off_b[i] = (uint32_t)((r < cols_left ? r : cols_left - 1) * ROW_BYTES) + chunk;
  }
  auto sample_of = [&](int c) {                            // (a card that is on the board: any row, it is not stored)
    const int32_t s = g.row_of[(int64_t)c * g.states + state_row];
    return (uint32_t)(s < 0 ? 0 : s) * (uint32_t)ROW_BYTES + chunk;
  };
  auto fetch = [&](char* buf, int c, uint32_t off_a, int block) {
    const int at = block * LN_BLOCK_BYTES;
    const char* pb = g.cards + ((int64_t)c * g.width + n0) * ROW_BYTES + at;
    ln_to_lds(g.gone + at + off_a, buf + wave * 8 * LN_BLOCK_BYTES);
    ln_to_lds(pb + off_b[0], buf + (BM + wave * 8) * LN_BLOCK_BYTES);
    ln_to_lds(pb + off_b[1], buf + (BM + 64 + wave * 8) * LN_BLOCK_BYTES);
    __builtin_amdgcn_sched_barrier(0);
  };
  uint32_t off_a = sample_of(c0);
  fetch(buf0, c0, off_a, 0);

  const int fr = lane & 15, fq = lane >> 4, turn = (fr >> 1) & 7;
  ln_float4 t0[TM][TN], t1[TM][TN], bi[TN];
#pragma unroll
  for (int j = 0; j < TN; ++j) {
    const int n = n0 + (wn * TN + j) * 16 + fq * 4, nn = n < g.width ? n : 0;      // width is a multiple of 32
    bi[j] = *reinterpret_cast<const ln_float4*>(g.b_inv + nn);
    bi[j] *= 1.0f / LN_SAMPLE_SCALE;
#pragma unroll
    for (int i = 0; i < TM; ++i) {
      const int r = (wm * TM + i) * 16 + fr;
      const int64_t at = (m0 + (r < rows_left ? r : 0)) * g.width + nn;
      t0[i][j] = *reinterpret_cast<const ln_float4*>(g.products + at);
      t1[i][j] = *reinterpret_cast<const ln_float4*>(g.products + g.states * g.width + at);
      base_of[i * TN + j][threadIdx.x] = *reinterpret_cast<const ln_float4*>(g.base + at);
    }
  }
  const LnScale scale = ln_scale(g.stats[0] + g.stats[1]);
  const int64_t out_bytes = (int64_t)(g.width / 32) * LN_BLOCK_BYTES;

  for (int c = c0; c < c1; ++c) {
    ln_float4 acc[TM][TN] = {};
    auto multiply = [&](const char* buf) {
      const int ch = (fq ^ turn) * 16, cl = ((4 + fq) ^ turn) * 16;
      const char* la = buf + (wm * TM * 16 + fr) * LN_BLOCK_BYTES;
      const char* lb = buf + (BM + wn * TN * 16 + fr) * LN_BLOCK_BYTES;
      ln_half8 wh[TN], wl[TN];
#pragma unroll
      for (int j = 0; j < TN; ++j) {
        wl[j] = *reinterpret_cast<const ln_half8*>(lb + j * 16 * LN_BLOCK_BYTES + cl);
        wh[j] = *reinterpret_cast<const ln_half8*>(lb + j * 16 * LN_BLOCK_BYTES + ch);
      }
#pragma unroll
      for (int i = 0; i < TM; ++i) {
        const ln_half8 xh = *reinterpret_cast<const ln_half8*>(la + i * 16 * LN_BLOCK_BYTES + ch);
        const ln_half8 xl = *reinterpret_cast<const ln_half8*>(la + i * 16 * LN_BLOCK_BYTES + cl);
#pragma unroll
        for (int j = 0; j < TN; ++j) {
          acc[i][j] = __builtin_amdgcn_mfma_f32_16x16x32_f16(wl[j], xh, acc[i][j], 0, 0, 0);
          acc[i][j] = __builtin_amdgcn_mfma_f32_16x16x32_f16(wh[j], xl, acc[i][j], 0, 0, 0);
          acc[i][j] = __builtin_amdgcn_mfma_f32_16x16x32_f16(wh[j], xh, acc[i][j], 0, 0, 0);
        }
      }
    };
    int32_t row[TM];
    float2 wt[TM];
#pragma unroll
    for (int i = 0; i < TM; ++i) {
      const int r = (wm * TM + i) * 16 + fr;
      row[i] = r < rows_left ? g.row_of[(int64_t)c * g.states + m0 + r] : -1;
    }
    const int next = c + 1 < c1 ? c + 1 : c;
    static_assert(LN_CARD_BLOCKS == 4, "a card is two rounds of the two buffers");
    p2_sync_loads();
    fetch(buf1, c, off_a, 1);
    multiply(buf0);
    p2_sync_loads();
    fetch(buf0, c, off_a, 2);
    const uint32_t off_next = sample_of(next);
#pragma unroll
    for (int i = 0; i < TM; ++i) wt[i] = row[i] >= 0 ? g.weight[row[i]] : make_float2(0.f, 0.f);
    multiply(buf1);
    p2_sync_loads();
    fetch(buf1, c, off_a, 3);
    multiply(buf0);
    p2_sync_loads();
    off_a = off_next;
    fetch(buf0, next, off_a, 0);
    multiply(buf1);
#pragma unroll
    for (int i = 0; i < TM; ++i) {
      if (row[i] < 0) continue;
#pragma unroll
      for (int j = 0; j < TN; ++j) {
        const int n = n0 + (wn * TN + j) * 16 + fq * 4;
        if (n >= g.width) continue;
        const ln_float4 bs = base_of[i * TN + j][threadIdx.x];
        ln_half4 hi, lo;
#pragma unroll
        for (int e = 0; e < 4; ++e) {
          const float v = fmaf(t0[i][j][e], wt[i].x, fmaf(t1[i][j][e], wt[i].y, bs[e])) - acc[i][j][e] * bi[j][e];
          _Float16 h, l;
          ln_split(ln_relu(v) * scale.up, h, l);
          hi[e] = h;
          lo[e] = l;
        }
        char* at = g.out_split + row[i] * out_bytes + (n >> 5) * LN_BLOCK_BYTES + (n & 31) * 2;
        *reinterpret_cast<ln_half4*>(at) = hi;
        *reinterpret_cast<ln_half4*>(at + 64) = lo;
        if (n == 0) g.out_inv[row[i]] = scale.down;
      }
    }
  }
  p2_sync_loads();                                         // the last fetch has landed before the LDS is given back
}

// The samples whose first layer is taken whole: those of `whole` (a device count of them).  Their ranges are masked,
// normalised and split on the way into LDS, 64 samples against 128 columns a tile, and multiplied by the ranges' columns
// as LN_PLAIN does; the board's columns come from `base` and `columns`.  Runs behind ln_first_kernel, which wrote the
// same rows of `out_split` from zero weights.  A fixed number of workgroups takes the tiles in turn, each XCD a run of
// them, columns outermost, so that it keeps its columns' weights in its L2.  Where the tiles leave workgroups over, a
// tile's steps are cut into as many parts as there are workgroups for, and another launch adds them up (the last
// workgroup of a tile doing that, behind fences of the whole device, took 50 us more).
// 3 x 1536, ms a call, float32 on the vector units (four samples at a time) -> here: 2240 states with three hands per
// range (up to 12 of 48 samples whole) 21.4 -> 5.4, with one hand 9.8 -> 4.4, smooth ranges 3.7; 35 states with three
// hands 0.66 -> 0.31 (a tile in one part 0.39), smooth 0.27.  The network layer by layer: 20.4 and 0.56.  Bound: for few
// samples the chain of steps, 1.2 us each; for many the splitting, which the vector units do again for every stripe of
// columns.
struct LnWhole {
  const float* pre_beliefs;
  const int64_t *root_indices, *board;
  int64_t source_rows;
  const LnSample* samples;
  const int32_t *whole, *whole_count;
  const char* ranges;           // [2][width] split rows
  const float *b_inv, *bias, *base, *columns, *stats;
  int width;
  ln_float4* parts;             // [LN_WHOLE_GRID][4][LN_WHOLE_THREADS]
  char* out_split;
  float* out_inv;
};
constexpr int LN_WHOLE_ROWS = 64, LN_WHOLE_COLS = 128, LN_WHOLE_THREADS = 512, LN_WHOLE_GRID = 512;
// A tile of the ranges' share becomes rows of `out_split`: element e of sum[i][j] is row (wave / 4 TM + i) 16 + lane % 16,
// column (wave % 4 TN + j) 16 + 4 (lane / 16) + e.
constexpr int LN_WHOLE_TM = 2, LN_WHOLE_TN = 2;
__device__ __forceinline__ void ln_whole_store(const LnWhole& g, const ln_float4 (&sum)[LN_WHOLE_TM][LN_WHOLE_TN], int count,
                                               int m0, int n0) {
  constexpr int TM = LN_WHOLE_TM, TN = LN_WHOLE_TN;
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  const int wm = wave >> 2, wn = wave & 3, fr = lane & 15, fq = lane >> 4;
  const LnScale scale = ln_scale(g.stats[0] + g.stats[1]);
  const int64_t out_bytes = (int64_t)(g.width / 32) * LN_BLOCK_BYTES;
#pragma unroll
  for (int i = 0; i < TM; ++i) {
    const int r = m0 + (wm * TM + i) * 16 + fr;
    if (r >= count) continue;
    const int32_t s = g.whole[r];
    const LnSample sm = g.samples[s];
#pragma unroll
    for (int j = 0; j < TN; ++j) {
      const int n = n0 + (wn * TN + j) * 16 + fq * 4;
      if (n >= g.width) continue;
      const ln_float4 bi = *reinterpret_cast<const ln_float4*>(g.b_inv + n);
      ln_float4 rest;                                    // what does not come from the ranges
      if (sm.card >= 0) {
        rest = *reinterpret_cast<const ln_float4*>(g.base + (int64_t)sm.state * g.width + n);
        rest += *reinterpret_cast<const ln_float4*>(g.columns + (int64_t)sm.card * g.width + n);
      } else {
        rest = *reinterpret_cast<const ln_float4*>(g.bias + n);
      }
      ln_half4 hi, lo;
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        const float v = sum[i][j][e] * (bi[e] * (1.0f / LN_SAMPLE_SCALE)) + rest[e];
        _Float16 h, l;
        ln_split(ln_relu(v) * scale.up, h, l);
        hi[e] = h;
        lo[e] = l;
      }
      char* at = g.out_split + s * out_bytes + (n >> 5) * LN_BLOCK_BYTES + (n & 31) * 2;
      *reinterpret_cast<ln_half4*>(at) = hi;
      *reinterpret_cast<ln_half4*>(at + 64) = lo;
      if (n == 0) g.out_inv[s] = scale.down;
    }
  }
}

// Into how many parts the steps of a tile are cut, each a divisor of them that leaves an even number: as many as there are
// workgroups for.
__device__ __forceinline__ unsigned ln_whole_split(unsigned tiles) {
  unsigned split = 14;
  while (split > 1 && tiles * split > LN_WHOLE_GRID) split = split == 14 ? 7 : split == 7 ? 6 : split / 2;
  return split;
}

__global__ __launch_bounds__(LN_WHOLE_THREADS, 4) void ln_whole_kernel(LnWhole g) {
  constexpr int TM = LN_WHOLE_TM, TN = LN_WHOLE_TN, BM = LN_WHOLE_ROWS, BN = LN_WHOLE_COLS, STEPS = 2 * LN_RANGE_BLOCKS;
  static_assert(STEPS % 2 == 0, "steps in pairs, a buffer each");
  __shared__ __align__(128) char buf0[(BM + BN) * LN_BLOCK_BYTES];
  __shared__ __align__(128) char buf1[(BM + BN) * LN_BLOCK_BYTES];
  const int count = *g.whole_count;
  const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int wm = wave >> 2, wn = wave & 3;                 // waves 2 x 4, 32 x 32 each
  const int fr = lane & 15, fq = lane >> 4, turn = (fr >> 1) & 7;
  const int64_t row_bytes = LN_RANGE_BLOCKS * LN_BLOCK_BYTES;
  const unsigned tiles_m = (unsigned)((count + BM - 1) / BM), tiles_n = (unsigned)((g.width + BN - 1) / BN);
  const unsigned split = ln_whole_split(tiles_m * tiles_n);
  const int steps = STEPS / (int)split;
  const unsigned items = tiles_m * tiles_n * split, xcd = blockIdx.x & 7, per = items >> 3, more = items & 7;
  const unsigned mine = per + (xcd < more ? 1 : 0), start = xcd * per + (xcd < more ? xcd : more);
  for (unsigned turn_of = blockIdx.x >> 3; turn_of < mine; turn_of += gridDim.x >> 3) {
    const unsigned item = start + turn_of, part = item % split, tile = item / split, tm = tile % tiles_m, tn = tile / tiles_m;
    const int first = (int)part * steps, m0 = (int)tm * BM, n0 = (int)tn * BN;
    const int cols_left = g.width - n0 < BN ? g.width - n0 : BN;

    // this thread's part of the samples: row threadIdx.x / 8, four hands of every block
    const int a_row = threadIdx.x >> 3, a_col = (threadIdx.x & 7) * 4;
    const float* range = g.stats;                          // (of an input of zeros: one number, not used)
    bool dealt = false;
    float inv[2] = {0.f, 0.f}, uniform = 0.f;
    uint64_t gone = 0;
    if (m0 + a_row < count) {
      const LnSample sm = g.samples[g.whole[m0 + a_row]];
      const int64_t root = g.root_indices ? g.root_indices[sm.state] : sm.state;
      if (sm.card >= 0 && root >= 0 && root < g.source_rows) {
        int bcards[5];
        const int left = P2_CARDS - chance_board(g.board + root * 5, bcards, gone) - 1;
        gone |= 1ull << sm.card;
        uniform = 1.0f / fmaxf((float)(left * (left - 1) / 2), 1.0f);
        range = g.pre_beliefs + root * (2 * P2_H);
        dealt = true;
        inv[0] = sm.inv0;
        inv[1] = sm.inv1;
      }
    }
    float x[4];
    uint32_t ca[4], cb[4];                                 // the hands' cards
    auto load = [&](int step) {
      const int p = step >= LN_RANGE_BLOCKS, h = (step - p * LN_RANGE_BLOCKS) * 32 + a_col;
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        const int hand = h + e < P2_H ? h + e : 0;         // (selected, not branched on: the loads go out together)
        ca[e] = p2_combo.a[hand];
        cb[e] = p2_combo.b[hand];
        x[e] = range[dealt ? p * P2_H + hand : 0];
      }
    };
    auto store = [&](char* buf, int step) {
      const int p = step >= LN_RANGE_BLOCKS, h = (step - p * LN_RANGE_BLOCKS) * 32 + a_col;
      const float scaled = p ? inv[1] : inv[0];
      ln_half4 hi, lo;
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        const bool off = (((gone >> ca[e]) | (gone >> cb[e])) & 1ull) | !dealt | (h + e >= P2_H);
        const float v = off ? 0.f : (scaled < 0.f ? uniform : x[e] * scaled);
        _Float16 a, b;
        ln_split(v * LN_SAMPLE_SCALE, a, b);
        hi[e] = a;
        lo[e] = b;
      }
      char* row = buf + a_row * LN_BLOCK_BYTES;
      const int chunk = a_col >> 3, half = (a_col & 4) * 2, swap = (a_row >> 1) & 7;
      *reinterpret_cast<ln_half4*>(row + ((chunk ^ swap) << 4) + half) = hi;
      *reinterpret_cast<ln_half4*>(row + (((chunk + 4) ^ swap) << 4) + half) = lo;
    };
    // and of the weights: 16 bytes of rows threadIdx.x / 8 and 64 + threadIdx.x / 8
    uint32_t off_b[2];
#pragma unroll
    for (int i = 0; i < 2; ++i) {
      const int r = a_row + 64 * i;
      off_b[i] = (uint32_t)((r < cols_left ? r : cols_left - 1) * (int)row_bytes + (((lane & 7) ^ ((a_row >> 1) & 7)) * 16));
    }
    auto fetch = [&](char* buf, int step) {
      const int p = step >= LN_RANGE_BLOCKS;
      const char* from = g.ranges + ((int64_t)p * g.width + n0) * row_bytes + (step - p * LN_RANGE_BLOCKS) * LN_BLOCK_BYTES;
      ln_to_lds(from + off_b[0], buf + (BM + wave * 8) * LN_BLOCK_BYTES);
      ln_to_lds(from + off_b[1], buf + (BM + 64 + wave * 8) * LN_BLOCK_BYTES);
      load(step);
      __builtin_amdgcn_sched_barrier(0);
    };
    ln_float4 acc[TM][TN] = {}, sum[TM][TN] = {};
    // A step's operands are read before the next step's loads go out: behind them the compiler waits for those first.
    ln_half8 wh[TN], wl[TN], xh[TM], xl[TM];
    auto take = [&](const char* buf) {
      const int ch = (fq ^ turn) * 16, cl = ((4 + fq) ^ turn) * 16;
      const char* la = buf + (wm * TM * 16 + fr) * LN_BLOCK_BYTES;
      const char* lb = buf + (BM + wn * TN * 16 + fr) * LN_BLOCK_BYTES;
#pragma unroll
      for (int j = 0; j < TN; ++j) {
        wl[j] = *reinterpret_cast<const ln_half8*>(lb + j * 16 * LN_BLOCK_BYTES + cl);
        wh[j] = *reinterpret_cast<const ln_half8*>(lb + j * 16 * LN_BLOCK_BYTES + ch);
      }
#pragma unroll
      for (int i = 0; i < TM; ++i) {
        xh[i] = *reinterpret_cast<const ln_half8*>(la + i * 16 * LN_BLOCK_BYTES + ch);
        xl[i] = *reinterpret_cast<const ln_half8*>(la + i * 16 * LN_BLOCK_BYTES + cl);
      }
      __builtin_amdgcn_sched_barrier(0);
    };
    auto multiply = [&]() {
#pragma unroll
      for (int i = 0; i < TM; ++i)
#pragma unroll
        for (int j = 0; j < TN; ++j) {
          ln_float4 t = __builtin_amdgcn_mfma_f32_16x16x32_f16(wl[j], xl[i], ln_float4{}, 0, 0, 0);
          t = __builtin_amdgcn_mfma_f32_16x16x32_f16(wl[j], xh[i], t, 0, 0, 0);
          t = __builtin_amdgcn_mfma_f32_16x16x32_f16(wh[j], xl[i], t, 0, 0, 0);
          acc[i][j] += __builtin_amdgcn_mfma_f32_16x16x32_f16(wh[j], xh[i], t, 0, 0, 0);
        }
      __builtin_amdgcn_sched_barrier(0);                   // (`store` waits for the loads)
    };
    auto carry = [&]() {
#pragma unroll
      for (int i = 0; i < TM; ++i)
#pragma unroll
        for (int j = 0; j < TN; ++j) {
          sum[i][j] += acc[i][j];
          acc[i][j] = ln_float4{};
        }
    };
    fetch(buf0, first);
    store(buf0, first);
    for (int step = first; step < first + steps; step += 2) {
      p2_sync_loads();                                     // `step` is there, and everyone is done with buf1
      take(buf0);
      fetch(buf1, step + 1);
      multiply();
      store(buf1, step + 1);
      p2_sync_loads();
      const int next = step + 2 < first + steps ? step + 2 : step + 1;   // past the end: a block nobody uses
      take(buf1);
      fetch(buf0, next);
      multiply();
      store(buf0, next);
      if ((step & 6) == 6) carry();
    }
    p2_sync_loads();                                       // everyone is done with the buffers
    carry();
    if (split > 1) {
      ln_float4* at = g.parts + (int64_t)item * (TM * TN) * LN_WHOLE_THREADS + threadIdx.x;
#pragma unroll
      for (int i = 0; i < TM; ++i)
#pragma unroll
        for (int j = 0; j < TN; ++j) at[(i * TN + j) * LN_WHOLE_THREADS] = sum[i][j];
      continue;
    }
    ln_whole_store(g, sum, count, m0, n0);
  }
}

// Adds up the parts of the tiles that ln_whole_kernel has cut, in their order, and finishes them.
__global__ __launch_bounds__(LN_WHOLE_THREADS) void ln_whole_parts_kernel(LnWhole g) {
  constexpr int TM = LN_WHOLE_TM, TN = LN_WHOLE_TN;
  const int count = *g.whole_count;
  const unsigned tiles_m = (unsigned)((count + LN_WHOLE_ROWS - 1) / LN_WHOLE_ROWS);
  const unsigned tiles = tiles_m * (unsigned)((g.width + LN_WHOLE_COLS - 1) / LN_WHOLE_COLS), split = ln_whole_split(tiles);
  const unsigned tile = blockIdx.x;
  if (split == 1 || tile >= tiles) return;
  const ln_float4* at = g.parts + (int64_t)tile * split * (TM * TN) * LN_WHOLE_THREADS + threadIdx.x;
  ln_float4 sum[TM][TN] = {};
#pragma unroll 2
  for (unsigned k = 0; k < split; ++k, at += (TM * TN) * LN_WHOLE_THREADS)
#pragma unroll
    for (int i = 0; i < TM; ++i)
#pragma unroll
      for (int j = 0; j < TN; ++j) sum[i][j] += at[(i * TN + j) * LN_WHOLE_THREADS];
  ln_whole_store(g, sum, count, (int)(tile % tiles_m) * LN_WHOLE_ROWS, (int)(tile / tiles_m) * LN_WHOLE_COLS);
}

// The means over the samples of each state as split rows: the last layer's input.
__global__ __launch_bounds__(LN_THREADS) void ln_means_kernel(const int64_t* __restrict__ offsets,
                                                               const double* __restrict__ sums,
                                                               const double* __restrict__ parts, int width, int tile_rows,
                                                               char* __restrict__ out, float* __restrict__ inv) {
  __shared__ float red[LN_THREADS / 64];
  const int64_t i = blockIdx.x, o0 = offsets[i], o1 = offsets[i + 1];
  const double count = o1 > o0 ? (double)(o1 - o0) : 1.0;
  const int64_t first = o0 / tile_rows, last = o1 > o0 ? (o1 - 1) / tile_rows : first;
  auto mean = [&](int k) {
    double v;
    if (o1 <= o0) v = 0.0;
    else if (first == last) v = sums[i * width + k];
    else {
      v = parts[(first * 2 + 1) * width + k];
      for (int64_t tile = first + 1; tile <= last; ++tile) v += parts[tile * 2 * width + k];
    }
    return v / count;
  };
  float mx = 0.f;
  for (int k = threadIdx.x; k < width; k += LN_THREADS) mx = fmaxf(mx, fabsf((float)mean(k)));
  const LnScale s = ln_scale(ln_block_max(mx, red));
  if (threadIdx.x == 0) inv[i] = s.down;
  for (int u = threadIdx.x; u < width / 8; u += LN_THREADS) {
    ln_half8 hi, lo;
#pragma unroll
    for (int q = 0; q < 8; ++q) {
      const double y = mean(8 * u + q) * (double)s.up;
      hi[q] = (_Float16)(float)y;
      lo[q] = (_Float16)(float)(y - (double)hi[q]);
    }
    char* at = out + i * (int64_t)(width / 32) * LN_BLOCK_BYTES + (8 * u >> 5) * LN_BLOCK_BYTES + (8 * u & 31) * 2;
    *reinterpret_cast<ln_half8*>(at) = hi;
    *reinterpret_cast<ln_half8*>(at + 64) = lo;
  }
}

// Rows per tile of the product over `m` rows and `n` columns, `batches` times (the rule of ln_gemm_kernel's comment).
static inline int ln_tile(int epi, int64_t m, int64_t n, int64_t batches) {
  const int64_t large = ((m + 255) / 256) * ((n + 255) / 256) * batches;
  const int64_t small = ((m + 127) / 128) * ((n + 127) / 128) * batches;
  return large >= 1024 && epi != LN_PLAIN ? 256 : (small >= 192 ? 128 : 64);
}

template <int EPI>
static int ln_launch(const LnGemm& g, hipStream_t stream) {
  const int tile = ln_tile(EPI, g.m, g.n, g.batches);
  const int64_t count = ((g.m + tile - 1) / tile) * ((g.n + tile - 1) / tile) * g.batches;
  if (count > 0x7FFFFFFF) return P2_EINVAL;
  const dim3 grid((unsigned)count);
  if constexpr (EPI != LN_PLAIN)
    if (tile == 256) hipLaunchKernelGGL((ln_gemm_kernel<EPI, 2, 4, 8, 4>), grid, dim3(512), 0, stream, g);
  if (tile == 128) hipLaunchKernelGGL((ln_gemm_kernel<EPI, 2, 2, 4, 4>), grid, dim3(256), 0, stream, g);
  if (tile == 64) hipLaunchKernelGGL((ln_gemm_kernel<EPI, 2, 2, 2, 2>), grid, dim3(256), 0, stream, g);
  P2_LAUNCH_CHECK();
  return 0;
}

// Where things lie in the workspace of a call: 256-byte aligned pieces, counted the same way for its size and its use.
struct LnWorkspace {
  uintptr_t base;
  int64_t size;
  explicit LnWorkspace(void* at) : base((uintptr_t)at), size(0) {}
  template <typename T>
  T* take(int64_t count) {
    T* p = reinterpret_cast<T*>(base + (uintptr_t)size);
    size += (count * (int64_t)sizeof(T) + 255) / 256 * 256;
    return p;
  }
};

struct LnPlan {
  float* out_max[2];                       // these two and the count are cleared first, one run
  int32_t* whole_count;
  int64_t cleared;
  float *stats, *w_inv[LN_MAX_LAYERS], *w_bound[LN_MAX_LAYERS], *bias[LN_MAX_LAYERS], *unit[LN_MAX_LAYERS];
  char *first_ranges, *first_cards, *weights[LN_MAX_LAYERS];
  float *first_board, *products, *base;
  char *ranges, *gone, *hidden[2], *means;
  float *ranges_inv, *hidden_inv[2], *means_inv;
  double *sums, *parts;
  float2* weight;
  LnSample* samples;
  int32_t *row_of, *whole;
  ln_float4* whole_parts;
  int64_t size;
};

// `widths[0..layers-1]`: the layers' answers.
static LnPlan ln_plan(void* base, int64_t states, int64_t samples, const int32_t* widths, int layers) {
  LnPlan p;
  LnWorkspace w(base);
  int widest = 0;
  for (int l = 0; l + 1 < layers; ++l) widest = widths[l] > widest ? widths[l] : widest;
  for (int k = 0; k < 2; ++k) p.out_max[k] = w.take<float>(samples);
  p.whole_count = w.take<int32_t>(1);
  p.cleared = w.size;
  p.stats = w.take<float>(2 * layers);
  for (int l = 0; l < layers; ++l) {
    p.w_inv[l] = w.take<float>(widths[l]);
    p.w_bound[l] = w.take<float>(widths[l]);
    p.bias[l] = w.take<float>(widths[l]);
    p.unit[l] = w.take<float>(widths[l]);
    p.weights[l] = l ? w.take<char>((int64_t)widths[l] * (widths[l - 1] / 32) * LN_BLOCK_BYTES) : nullptr;
  }
  for (int k = 0; k < 2; ++k) {
    p.hidden[k] = w.take<char>(samples * (widest / 32) * LN_BLOCK_BYTES);
    p.hidden_inv[k] = w.take<float>(samples);
  }
  // Nothing is written to the second buffer of activations before the first layer is done: its pieces share the space.
  LnWorkspace early(p.hidden[1]);
  const int64_t w0 = widths[0];
  p.first_ranges = early.take<char>(2 * w0 * LN_RANGE_BLOCKS * LN_BLOCK_BYTES);
  p.first_cards = early.take<char>(P2_CARDS * w0 * LN_CARD_BLOCKS * LN_BLOCK_BYTES);
  p.first_board = early.take<float>(P2_CARDS * w0);
  p.products = early.take<float>(2 * states * w0);
  p.base = early.take<float>(states * w0);
  p.ranges = early.take<char>(2 * states * LN_RANGE_BLOCKS * LN_BLOCK_BYTES);
  p.ranges_inv = early.take<float>(2 * states);
  p.gone = early.take<char>(samples * LN_CARD_BLOCKS * LN_BLOCK_BYTES);
  p.weight = early.take<float2>(samples);
  p.samples = early.take<LnSample>(samples);
  p.row_of = early.take<int32_t>(P2_CARDS * states);
  p.whole = early.take<int32_t>(samples);
  p.whole_parts = early.take<ln_float4>((int64_t)LN_WHOLE_GRID * 4 * LN_WHOLE_THREADS);
  const int64_t early_end = (int64_t)((uintptr_t)p.hidden[1] - (uintptr_t)base) + early.size;
  if (w.size < early_end) w.size = early_end;
  const int last = widths[layers - 2];
  const int64_t tiles = (samples + 63) / 64;               // of the smallest kind
  p.sums = w.take<double>(states * last);
  p.parts = w.take<double>(tiles * 2 * last);
  p.means = w.take<char>(states * (last / 32) * LN_BLOCK_BYTES);
  p.means_inv = w.take<float>(states);
  p.size = w.size;
  return p;
}

__global__ __launch_bounds__(LN_THREADS) void ln_clear_kernel(uint4* __restrict__ at, int64_t count) {
  for (int64_t k = (int64_t)blockIdx.x * LN_THREADS + threadIdx.x; k < count; k += (int64_t)gridDim.x * LN_THREADS)
    at[k] = make_uint4(0u, 0u, 0u, 0u);
}
static inline unsigned ln_clear_grid(int64_t units) {
  const int64_t blocks = (units + LN_THREADS - 1) / LN_THREADS;
  return (unsigned)(blocks < 256 ? blocks : 256);
}

static bool ln_network_ok(const int32_t* widths, int layers) {
  if (!widths || layers < 3 || layers > LN_MAX_LAYERS || widths[layers - 1] != 2 * P2_H) return false;
  for (int l = 0; l + 1 < layers; ++l)
    if (widths[l] < 32 || widths[l] > 65536 || widths[l] % 32) return false;
  return true;
}
static bool ln_counts_ok(int64_t states, int64_t samples) {
  return states >= 0 && samples >= 0 && states <= 0x7FFFFF && samples <= LN_MAX_SAMPLES;
}
}  // namespace p2

extern "C" {

int64_t p2hip_chance_network_workspace(int64_t n, int64_t total_samples, const int32_t* host_widths, int layers) {
  if (!p2::ln_network_ok(host_widths, layers) || !p2::ln_counts_ok(n, total_samples)) return -1;
  return p2::ln_plan(nullptr, n, total_samples, host_widths, layers).size;
}

int p2hip_chance_network(const float* pre_beliefs, const int64_t* root_indices, const int64_t* board, int64_t n,
                         const int64_t* sample_offsets, int64_t source_rows, int64_t total_samples,
                         const float* const* host_weights, const float* const* host_biases, const int32_t* host_widths,
                         int layers, void* workspace, int64_t workspace_bytes, float* expected, void* stream) {
  using namespace p2;
  const float* const* weights = host_weights;
  const float* const* biases = host_biases;
  const int32_t* widths = host_widths;
  if (!ln_network_ok(widths, layers) || !ln_counts_ok(n, total_samples) || source_rows < 0) return P2_EINVAL;
  if (n == 0 || total_samples == 0) return 0;
  if (!pre_beliefs || !board || !sample_offsets || !weights || !biases || !workspace || !expected) return P2_EINVAL;
  if ((((uintptr_t)workspace & 255u) | ((uintptr_t)expected & 15u) | ((uintptr_t)pre_beliefs & 3u)) != 0) return P2_EINVAL;
  for (int l = 0; l < layers; ++l)
    if (!weights[l] || (((uintptr_t)weights[l] | (uintptr_t)biases[l]) & 15u) != 0) return P2_EINVAL;
  const LnPlan p = ln_plan(workspace, n, total_samples, widths, layers);
  if (workspace_bytes < p.size) return P2_EINVAL;
  hipStream_t s = (hipStream_t)stream;
  const int w0 = widths[0];
  {
    LnFirstWeights a = {};
    for (int l = 0; l < layers; ++l) {
      const LnLayerWeights g = {weights[l], biases[l], l ? p.unit[l - 1] : nullptr, p.weights[l], p.w_inv[l], p.w_bound[l],
                                p.bias[l], p.unit[l], l ? (int)widths[l - 1] : LN_INPUT, l + 1 < layers};
      if (l == 0) {
        a.layer = g;
        a.ranges = p.first_ranges; a.cards = p.first_cards; a.board = p.first_board;
        a.clear = (uint4*)workspace; a.clear_units = p.cleared / 16;
        a.width = w0; a.clear_blocks = (int)ln_clear_grid(a.clear_units);
        hipLaunchKernelGGL(ln_first_weights_kernel, dim3((unsigned)(w0 + a.clear_blocks)), dim3(LN_THREADS), 0, s, a);
      } else {
        hipLaunchKernelGGL(ln_weights_kernel, dim3((unsigned)widths[l]), dim3(LN_THREADS), 0, s, g);
      }
      P2_LAUNCH_CHECK();
    }
  }
  hipLaunchKernelGGL(ln_states_kernel, dim3((unsigned)n), dim3(LN_THREADS), 0, s, pre_beliefs, root_indices, board,
                     sample_offsets, source_rows, total_samples, p.ranges, p.ranges_inv, p.gone, p.weight, p.samples,
                     p.row_of, p.whole, p.whole_count);
  P2_LAUNCH_CHECK();
  {
    LnBounds b = {};
    for (int l = 0; l < layers; ++l) { b.bound[l] = p.w_bound[l]; b.bias[l] = p.bias[l]; b.rows[l] = widths[l]; }
    hipLaunchKernelGGL(ln_base_kernel, dim3((unsigned)(layers + n)), dim3(LN_THREADS), 0, s, b, layers, p.stats,
                       root_indices, board, source_rows, p.first_board, w0, p.base);
    P2_LAUNCH_CHECK();
  }
  int rc;
  {
    LnGemm g = {};
    g.a = p.ranges; g.b = p.first_ranges; g.a_inv = p.ranges_inv; g.b_inv = p.w_inv[0];
    g.m = n; g.n = w0; g.blocks = LN_RANGE_BLOCKS; g.batches = 2; g.out = p.products;
    if ((rc = ln_launch<LN_PLAIN>(g, s)) != 0) return rc;
  }
  {
    LnFirst g = {};
    g.gone = p.gone; g.cards = p.first_cards; g.b_inv = p.w_inv[0]; g.products = p.products; g.base = p.base;
    g.stats = p.stats; g.weight = p.weight; g.row_of = p.row_of; g.states = n; g.width = w0;
    g.out_split = p.hidden[0]; g.out_inv = p.hidden_inv[0];
    const int64_t squares = ((n + LN_FIRST_ROWS - 1) / LN_FIRST_ROWS) * ((w0 + LN_FIRST_COLS - 1) / LN_FIRST_COLS);
    const int64_t want = 512 / squares;
    g.groups = (int)(want < 1 ? 1 : (want > P2_CARDS ? P2_CARDS : want));
    if (squares * g.groups > 0x7FFFFFFF) return P2_EINVAL;
    hipLaunchKernelGGL(ln_first_kernel, dim3((unsigned)(squares * g.groups)), dim3(LN_FIRST_THREADS), 0, s, g);
    P2_LAUNCH_CHECK();
  }
  {
    const LnWhole g = {pre_beliefs, root_indices, board, source_rows, p.samples, p.whole, p.whole_count, p.first_ranges,
                       p.w_inv[0], p.bias[0], p.base, p.first_board, p.stats, w0, p.whole_parts, p.hidden[0], p.hidden_inv[0]};
    hipLaunchKernelGGL(ln_whole_kernel, dim3(LN_WHOLE_GRID), dim3(LN_WHOLE_THREADS), 0, s, g);
    P2_LAUNCH_CHECK();
    hipLaunchKernelGGL(ln_whole_parts_kernel, dim3(LN_WHOLE_GRID / 2), dim3(LN_WHOLE_THREADS), 0, s, g);
    P2_LAUNCH_CHECK();
  }
  for (int l = 1; l + 1 < layers; ++l) {
    const int in = (l - 1) & 1, out = l & 1;
    LnGemm g = {};
    g.a = p.hidden[in]; g.b = p.weights[l]; g.a_inv = p.hidden_inv[in]; g.b_inv = p.w_inv[l]; g.bias = p.bias[l];
    g.m = total_samples; g.n = widths[l]; g.blocks = widths[l - 1] / 32; g.batches = 1;
    if (l + 2 < layers) {
      const bool measured = l + 3 < layers;                // the hidden layer after this one needs a bound on its answer
      if (measured && l > 2) {                             // this buffer's maxima have been used: start again
        const int64_t units = (total_samples + 3) / 4;     // (the piece is 256-byte aligned at both ends)
        hipLaunchKernelGGL(ln_clear_kernel, dim3(ln_clear_grid(units)), dim3(LN_THREADS), 0, s, (uint4*)p.out_max[out], units);
        P2_LAUNCH_CHECK();
      }
      g.a_max = l > 1 ? p.out_max[in] : nullptr; g.first_stats = p.stats; g.stats = p.stats + 2 * l;
      g.out_split = p.hidden[out]; g.out_inv = p.hidden_inv[out]; g.out_max = measured ? p.out_max[out] : nullptr;
      if ((rc = ln_launch<LN_HIDDEN>(g, s)) != 0) return rc;
    } else {
      g.offsets = sample_offsets; g.states = n; g.sums = p.sums; g.parts = p.parts;
      if ((rc = ln_launch<LN_MEAN>(g, s)) != 0) return rc;
      hipLaunchKernelGGL(ln_means_kernel, dim3((unsigned)n), dim3(LN_THREADS), 0, s, sample_offsets, p.sums, p.parts,
                         (int)widths[l], ln_tile(LN_MEAN, total_samples, widths[l], 1), p.means, p.means_inv);
      P2_LAUNCH_CHECK();
    }
  }
  LnGemm g = {};
  const int l = layers - 1;
  g.a = p.means; g.b = p.weights[l]; g.a_inv = p.means_inv; g.b_inv = p.w_inv[l]; g.bias = p.bias[l];
  g.m = n; g.n = widths[l]; g.blocks = widths[l - 1] / 32; g.batches = 1; g.out = expected;
  return ln_launch<LN_PLAIN>(g, s);
}

}  // extern "C"
