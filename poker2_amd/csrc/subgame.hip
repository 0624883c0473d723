// What a search writes before its first iteration and reads after its last, without a pass of torch per step: the
// constant rows of a new state, the hands a board allows, the uniform initial policy with the reaches and ranges that
// follow from it, leaf values as the start of a backup, and the check for numbers that are not finite
// (src/p2/search/sparse_cfr_evaluator.py:240-306, cfr_evaluator.py:603-955).
// Bound: the rows they write (a workgroup per row).  192 three-raise river roots (20 160 nodes), us, torch -> here:
// constant rows 540 -> 205, allowed hands 930 -> 40 (both with the gaps between small launches), initial policy and
// what follows 2900 -> 300, a check 250 -> 44, leaf rows 150 -> 64 each.
#pragma once
#include "common.h"
#include "cfr_families.hip"

namespace p2 {

__device__ __forceinline__ void sub_fill(float* __restrict__ base, int64_t row, float v) {
  const float2 x[UB_PPT] = {make_float2(v, v), make_float2(v, v), make_float2(v, v)};
  fam_store(base, row, x);
}

// Rows of a new state that are one number: uniform policy 1 / children of the parent (0 for roots), reaches 1 for roots
// and 0 below, values +-reward at folds (player 0, 1) and 0 elsewhere.
__global__ __launch_bounds__(UB_BLOCK) void subgame_rows_kernel(
    const int64_t* __restrict__ parent_index, const int64_t* __restrict__ child_count, const uint8_t* __restrict__ fold,
    const float* __restrict__ reward, int64_t n_roots, float* __restrict__ uniform, float* __restrict__ reach,
    float* __restrict__ reach_avg, float* __restrict__ latest, float* __restrict__ values_avg) {
  const int64_t r = blockIdx.x;
  const bool root = r < n_roots;
  const float share = root ? 0.f : 1.0f / (float)child_count[parent_index[r]];
  const float won = fold[r] ? reward[r] : 0.f;
  sub_fill(uniform, r, share);
#pragma unroll
  for (int p = 0; p < 2; ++p) {
    sub_fill(reach, 2 * r + p, root ? 1.f : 0.f);
    sub_fill(reach_avg, 2 * r + p, root ? 1.f : 0.f);
    const float v = fold[r] ? (p ? -won : won) : 0.f;
    sub_fill(latest, 2 * r + p, v);
    sub_fill(values_avg, 2 * r + p, v);
  }
}

// allowed[r][h] = no card of h on the board of r's root; prob[r] uniform over these hands.
__global__ __launch_bounds__(UB_BLOCK) void allowed_hands_kernel(const int64_t* __restrict__ board,
                                                                  const int64_t* __restrict__ root_index,
                                                                  uint8_t* __restrict__ allowed, float* __restrict__ prob) {
  const int64_t r = blockIdx.x;
  const int64_t* b5 = board + root_index[r] * 5;
  uint64_t bits = 0;
#pragma unroll
  for (int j = 0; j < 5; ++j) {
    const int64_t c = b5[j];
    if (c >= 0 && c < P2_CARDS) bits |= 1ull << c;
  }
  const int left = P2_CARDS - __popcll(bits), hands = left * (left - 1) / 2;
  const float each = 1.0f / fmaxf((float)hands, 1.0f);
  uchar2* m2 = reinterpret_cast<uchar2*>(allowed + r * P2_H);
  float2* p2v = p2_row2(prob, r);
  for (int i = threadIdx.x; i < P2_HPAIRS; i += UB_BLOCK) {
    bool ok[2];
#pragma unroll
    for (int q = 0; q < 2; ++q) {
      const int h = 2 * i + q;
      ok[q] = !(((bits >> p2_combo.a[h]) | (bits >> p2_combo.b[h])) & 1ull);
    }
    m2[i] = make_uchar2(ok[0], ok[1]);
    p2v[i] = make_float2(ok[0] ? each : 0.f, ok[1] ? each : 0.f);
  }
}

// The initial policy of a model without one (uniform over the legal actions) and what follows from it, for every row at
// once: policy and average policy, reach and average reach, ranges and average ranges.  A row walks down from its root
// (`roots`: the roots' ranges as given): at every step the actor's range times the policy, then both normalised over the
// allowed hands, as the level-by-level program does (cfr_evaluator.py:830-886).  That program normalises every row again
// while it goes deeper, so a row of level k is normalised depth - k more times at the end, a root depth times (once
// without levels): same roundings.
struct SubStep { float policy; int actor; };
__global__ __launch_bounds__(UB_BLOCK) void uniform_start_kernel(
    const float* __restrict__ roots, const uint8_t* __restrict__ allowed, const float* __restrict__ allowed_prob,
    const int64_t* __restrict__ parent_index, const int64_t* __restrict__ prev_actor, const int64_t* __restrict__ root_index,
    const uint8_t* __restrict__ legal, int actions, int64_t n_roots, int depth, float eps, float* __restrict__ policy,
    float* __restrict__ policy_avg, float* __restrict__ reach, float* __restrict__ reach_avg, float* __restrict__ beliefs,
    float* __restrict__ beliefs_avg) {
  __shared__ float red[2][2][OPS_WAVES];
  __shared__ SubStep way[FAM_MAX_DEPTH];
  const int64_t c = blockIdx.x, root = root_index[c];
  float2 x[2][UB_PPT], b[2][UB_PPT];
  uchar2 al[UB_PPT];
#pragma unroll
  for (int p = 0; p < 2; ++p) {
    fam_load((const float*)reach, 2 * root + p, x[p]);
    fam_load(roots, 2 * root + p, b[p]);
  }
  const uchar2* m2 = reinterpret_cast<const uchar2*>(allowed + c * P2_H);
#pragma unroll
  for (int j = 0; j < UB_PPT; ++j) {
    const int i = threadIdx.x + j * UB_BLOCK;
    al[j] = m2[i < P2_HPAIRS ? i : 0];
  }
  int steps = 0;
  for (int64_t r = c; r >= n_roots && steps < FAM_MAX_DEPTH; ++steps) {
    const int64_t parent = parent_index[r];
    int count = 0;
    for (int a = 0; a < actions; ++a) count += legal[parent * actions + a] != 0;
    if (threadIdx.x == 0) way[steps] = {count ? 1.0f / (float)count : 0.f, (int)prev_actor[r]};
    r = parent;
  }
  p2_sync_lds();
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  int turn = 0;
  auto normalise = [&]() {
#pragma unroll
    for (int p = 0; p < 2; ++p) {
      float local = 0.f;
#pragma unroll
      for (int j = 0; j < UB_PPT; ++j) {
        b[p][j].x = al[j].x ? b[p][j].x : 0.f;
        b[p][j].y = al[j].y ? b[p][j].y : 0.f;
        if (threadIdx.x + j * UB_BLOCK < P2_HPAIRS) local += b[p][j].x + b[p][j].y;
      }
      local = p2_wave_sum(local);
      if (lane == 0) red[turn][p][wave] = local;
    }
    p2_sync_lds();                                          // (two sets of sums: the next round writes the other one)
#pragma unroll
    for (int p = 0; p < 2; ++p) {
      float total = 0.f;
#pragma unroll
      for (int w = 0; w < OPS_WAVES; ++w) total += red[turn][p][w];
      if (total > eps) {
#pragma unroll
        for (int j = 0; j < UB_PPT; ++j) b[p][j] = make_float2(b[p][j].x / total, b[p][j].y / total);
      } else {
        fam_load(allowed_prob, c, b[p]);
      }
    }
    turn ^= 1;
  };
  float own = 0.f;
  for (int s = steps - 1; s >= 0; --s) {
    const SubStep st = way[s];
    own = st.policy;
#pragma unroll
    for (int j = 0; j < UB_PPT; ++j) {
      if (st.actor) {
        b[1][j].x *= own; b[1][j].y *= own; x[1][j].x *= own; x[1][j].y *= own;
      } else {
        b[0][j].x *= own; b[0][j].y *= own; x[0][j].x *= own; x[0][j].y *= own;
      }
    }
    normalise();
  }
  const int again = depth > 0 ? depth - steps : 1;
  for (int k = 0; k < again; ++k) normalise();
  sub_fill(policy, c, own);
  sub_fill(policy_avg, c, own);
#pragma unroll
  for (int p = 0; p < 2; ++p) {
    if (steps) {
#pragma unroll
      for (int j = 0; j < UB_PPT; ++j) x[p][j] = make_float2(al[j].x ? x[p][j].x : 0.f, al[j].y ? x[p][j].y : 0.f);
      fam_store(reach, 2 * c + p, x[p]);
    }
    fam_store(reach_avg, 2 * c + p, x[p]);
    fam_store(beliefs, 2 * c + p, b[p]);
    fam_store(beliefs_avg, 2 * c + p, b[p]);
  }
}

// out[r] = leaf[r] ? values[r], clamped to [-1, 1] if asked : 0, rows of both players.
__global__ __launch_bounds__(UB_BLOCK) void leaf_rows_kernel(const float* __restrict__ values,
                                                              const uint8_t* __restrict__ leaf, int clamp,
                                                              float* __restrict__ out) {
  const int64_t r = blockIdx.x;
  float2 v[2][UB_PPT] = {};
  if (leaf[r]) {
#pragma unroll
    for (int p = 0; p < 2; ++p) fam_load(values, 2 * r + p, v[p]);
  }
  auto cut = [&](float a) { return clamp ? (a < -1.f ? -1.f : (a > 1.f ? 1.f : a)) : a; };   // NaN stays
#pragma unroll
  for (int p = 0; p < 2; ++p) {
#pragma unroll
    for (int j = 0; j < UB_PPT; ++j) v[p][j] = make_float2(cut(v[p][j].x), cut(v[p][j].y));
    fam_store(out, 2 * r + p, v[p]);
  }
}

// *found becomes 1 if some element is infinite or NaN (it starts at 0).
__global__ __launch_bounds__(FLAT_BLOCK) void nonfinite_kernel(const uint2* __restrict__ x, int64_t npairs,
                                                                int32_t* __restrict__ found) {
  bool bad = false;
  P2_FLAT_LOOP(i, npairs) {
    const uint2 v = x[i];
    bad = bad || (v.x & 0x7F800000u) == 0x7F800000u || (v.y & 0x7F800000u) == 0x7F800000u;
  }
  if (__any(bad) && (threadIdx.x & 63) == 0) *found = 1;
}

}  // namespace p2

extern "C" {

int p2hip_subgame_rows(const int64_t* parent_index, const int64_t* child_count, const uint8_t* fold_mask,
                       const float* reward, int64_t n_roots, int64_t total, float* uniform, float* reach, float* reach_avg,
                       float* latest, float* values_avg, void* stream) {
  P2_REQ(n_roots >= 0 && total >= n_roots && total <= 0x7FFFFFFF);
  if (total == 0) return 0;
  P2_REQ(parent_index && child_count && fold_mask && reward && uniform && reach && reach_avg && latest && values_avg);
  P2_REQ(p2_aligned8(uniform) && p2_aligned8(reach) && p2_aligned8(reach_avg) && p2_aligned8(latest) &&
         p2_aligned8(values_avg));
  hipLaunchKernelGGL(p2::subgame_rows_kernel, dim3((unsigned)total), dim3(p2::UB_BLOCK), 0, P2_ST, parent_index, child_count,
                     fold_mask, reward, n_roots, uniform, reach, reach_avg, latest, values_avg);
  P2_LAUNCH_CHECK();
  return 0;
}

int p2hip_allowed_hands(const int64_t* board, const int64_t* root_index, int64_t total, uint8_t* allowed, float* prob,
                        void* stream) {
  P2_REQ(total >= 0 && total <= 0x7FFFFFFF);
  if (total == 0) return 0;
  P2_REQ(board && root_index && allowed && prob && p2_aligned8(prob) && (reinterpret_cast<uintptr_t>(allowed) & 1u) == 0);
  hipLaunchKernelGGL(p2::allowed_hands_kernel, dim3((unsigned)total), dim3(p2::UB_BLOCK), 0, P2_ST, board, root_index,
                     allowed, prob);
  P2_LAUNCH_CHECK();
  return 0;
}

int p2hip_uniform_start(const float* roots, const uint8_t* allowed, const float* allowed_prob, const int64_t* parent_index,
                        const int64_t* prev_actor, const int64_t* root_index, const uint8_t* legal_mask, int actions,
                        int64_t n_roots, int64_t total, int depth, float eps, float* policy, float* policy_avg,
                        float* reach, float* reach_avg, float* beliefs, float* beliefs_avg, void* stream) {
  P2_REQ(n_roots >= 0 && total >= n_roots && total <= 0x7FFFFFFF && actions >= 1 && depth >= 0 && depth <= p2::FAM_MAX_DEPTH);
  if (total == 0) return 0;
  P2_REQ(roots && allowed && allowed_prob && parent_index && prev_actor && root_index && legal_mask && policy && policy_avg &&
         reach && reach_avg && beliefs && beliefs_avg && roots != beliefs);
  P2_REQ(p2_aligned8(roots) && p2_aligned8(allowed_prob) && p2_aligned8(policy) && p2_aligned8(policy_avg) &&
         p2_aligned8(reach) && p2_aligned8(reach_avg) && p2_aligned8(beliefs) && p2_aligned8(beliefs_avg) &&
         (reinterpret_cast<uintptr_t>(allowed) & 1u) == 0);
  hipLaunchKernelGGL(p2::uniform_start_kernel, dim3((unsigned)total), dim3(p2::UB_BLOCK), 0, P2_ST, roots, allowed,
                     allowed_prob, parent_index, prev_actor, root_index, legal_mask, actions, n_roots, depth, eps, policy,
                     policy_avg, reach, reach_avg, beliefs, beliefs_avg);
  P2_LAUNCH_CHECK();
  return 0;
}

int p2hip_leaf_rows(const float* values, const uint8_t* leaf_mask, int64_t total, int clamp, float* out, void* stream) {
  P2_REQ(total >= 0 && total <= 0x7FFFFFFF);
  if (total == 0) return 0;
  P2_REQ(values && leaf_mask && out && p2_aligned8(values) && p2_aligned8(out));
  hipLaunchKernelGGL(p2::leaf_rows_kernel, dim3((unsigned)total), dim3(p2::UB_BLOCK), 0, P2_ST, values, leaf_mask, clamp, out);
  P2_LAUNCH_CHECK();
  return 0;
}

int p2hip_any_nonfinite(const float* x, int64_t n, int32_t* found, void* stream) {
  P2_REQ(n >= 0 && (n & 1) == 0);
  if (n == 0) return 0;
  P2_REQ(x && found && p2_aligned8(x) && p2_aligned4(found));
  const int64_t pairs = n / 2, blocks = (pairs + p2::FLAT_BLOCK - 1) / p2::FLAT_BLOCK;
  hipLaunchKernelGGL(p2::nonfinite_kernel, dim3((unsigned)(blocks < 16384 ? blocks : 16384)), dim3(p2::FLAT_BLOCK), 0, P2_ST,
                     (const uint2*)x, pairs, found);
  P2_LAUNCH_CHECK();
  return 0;
}

}  // extern "C"
