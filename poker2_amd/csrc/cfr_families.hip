// The launch-per-operation path, a family at a time: what the reference runs as several operations over whole tensors
// (fused_sparse_cfr_evaluator.py:201-398) as one launch per method, or per level of the tree where a level needs the one
// above or below it.  A workgroup takes a parent with its children, which are neighbouring rows; what the operations
// of cfr_ops.hip and unblocked.hip hand to each other through tensors of the tree's size (positive regrets and their
// sums, the actor's ranges and values per parent, marginals, opponent weights) stays in its registers and LDS.  Every
// number goes through the same roundings as there.
// Bound: memory where a launch has the whole tree (4-5 TB/s of rows), the chain of one family where it has a level.  192
// roots of mixed streets to depth 5 (8400 nodes), us, operations -> here: regrets and their update 154 -> 69, regret
// matching 69 -> 19, average policy 94 -> 43, reach and ranges of all levels 130 -> 105, expected values of five levels 199
// -> 104 (a family on eight waves instead of four 122), showdown rows with their gather and scatter 65 -> 20.
#pragma once
#include "common.h"
#include "unblocked.hip"
#include "cfr_ops.hip"

namespace p2 {

static_assert(UB_BLOCK == OPS_BLOCK && UB_PPT == OPS_PAIRS_PER_THREAD, "a lane's pairs of a row");
constexpr int FAM_MAX_CHILDREN = 8;
// (Where a kernel keeps MAXC children in registers or LDS, a family larger than the caller's max_children is left alone.)

__device__ __forceinline__ void fam_load(const float* __restrict__ base, int64_t row, float2 (&v)[UB_PPT]) {
  const float2* r = p2_row2(base, row);
#pragma unroll
  for (int j = 0; j < UB_PPT; ++j) {
    const int i = threadIdx.x + j * UB_BLOCK;
    v[j] = r[i < P2_HPAIRS ? i : 0];                        // no branch; what lies past the end is never used
  }
}
__device__ __forceinline__ void fam_store(float* __restrict__ base, int64_t row, const float2 (&v)[UB_PPT]) {
  float2* r = p2_row2(base, row);
#pragma unroll
  for (int j = 0; j < UB_PPT; ++j) {
    const int i = threadIdx.x + j * UB_BLOCK;
    if (i < P2_HPAIRS) r[i] = v[j];
  }
}
// Children k < MAXC of a family; places past its end hold the last child again.
template <int MAXC>
__device__ __forceinline__ void fam_load_children(const float* __restrict__ base, int64_t first, int count,
                                                  float2 (&v)[MAXC][UB_PPT]) {
#pragma unroll
  for (int k = 0; k < MAXC; ++k) fam_load(base, first + (k < count ? k : count - 1), v[k]);
}
// Sum over the children, one after the other.
template <int MAXC>
__device__ __forceinline__ void fam_sum(const float2 (&v)[MAXC][UB_PPT], int count, float2 (&sum)[UB_PPT]) {
#pragma unroll
  for (int j = 0; j < UB_PPT; ++j) sum[j] = make_float2(0.f, 0.f);
#pragma unroll
  for (int k = 0; k < MAXC; ++k)
    if (k < count)
#pragma unroll
      for (int j = 0; j < UB_PPT; ++j) { sum[j].x += v[k][j].x; sum[j].y += v[k][j].y; }
}

// r[c] = unblocked(beliefs[p][other player]) * (achieved[c][actor] - expected[p][actor]), 0 for rows below `bottom`:
// stored as `regrets`, or (UPDATE) added to the cumulative regrets as dcfr_update_kernel does.
struct FamUpdate {
  float *cumulative, *weights;
  const float *ta_num, *tb_num, *ta_den, *tb_den;
  int apply_dcfr, cfr_plus;
};
struct FamDiscount { float an, bn, ad, bd; };
__device__ __forceinline__ void fam_update(const FamUpdate& u, const FamDiscount& d, float r, float& c, float& w) {
  if (u.apply_dcfr) {
    const bool positive = c > 0.f;
    const float num = positive ? d.an : d.bn, den = positive ? d.ad : d.bd;
    c = c * num;
    c = c / den;
    w = w * num;
    w = w / den;
  }
  w = w + 1.0f;
  c = c + r;
  if (u.cfr_plus) c = fmaxf(c, 0.f);
}
__device__ __forceinline__ void fam_update_row(const FamUpdate& u, const FamDiscount& d, int64_t row,
                                               const float2 (&r)[UB_PPT], float2 (&c)[UB_PPT], float2 (&w)[UB_PPT]) {
#pragma unroll
  for (int j = 0; j < UB_PPT; ++j) {
    fam_update(u, d, r[j].x, c[j].x, w[j].x);
    fam_update(u, d, r[j].y, c[j].y, w[j].y);
  }
  fam_store(u.cumulative, row, c);
  fam_store(u.weights, row, w);
}
template <bool UPDATE>
__global__ __launch_bounds__(UB_BLOCK) void family_regrets_kernel(
    const float* __restrict__ achieved, const float* __restrict__ expected, const float* __restrict__ beliefs,
    const int64_t* __restrict__ to_act, const int64_t* __restrict__ prev_actor, const int64_t* __restrict__ child_offsets,
    const int64_t* __restrict__ child_count, int64_t bottom, int64_t top, float* __restrict__ regrets, FamUpdate u) {
  __shared__ __align__(8) float t[UB_STRIDE];
  __shared__ double cs[P2_CARDS];
  const int64_t p = blockIdx.x;
  FamDiscount d = {1.f, 1.f, 1.f, 1.f};
  if (UPDATE && u.apply_dcfr) d = {*u.ta_num, *u.tb_num, *u.ta_den, *u.tb_den};
  float2 cum[UB_PPT], wsum[UB_PPT];
  if (p < bottom) {
    const float2 none[UB_PPT] = {};
    if constexpr (UPDATE) {
      fam_load((const float*)u.cumulative, p, cum);
      fam_load((const float*)u.weights, p, wsum);
      fam_update_row(u, d, p, none, cum, wsum);
    } else {
      fam_store(regrets, p, none);
    }
  }
  const int count = p < top ? (int)child_count[p] : 0;
  if (count <= 0) return;
  const int64_t first = child_offsets[p], actor = to_act[p];
  float2 range[UB_PPT], e[UB_PPT], a[UB_PPT];
  fam_load(beliefs, 2 * p + (actor ^ 1), range);
  fam_load(expected, 2 * p + actor, e);
  fam_load(achieved, 2 * first + prev_actor[first], a);
  if constexpr (UPDATE) {
    fam_load((const float*)u.cumulative, first, cum);
    fam_load((const float*)u.weights, first, wsum);
  }
  stage_row(range, t);
  CardLane cl;
  HandCards hc;
  card_lane_init(cl);
  hand_cards_init(hc);
  p2_sync_lds();
  card_sums_fixed(cl, t, UB_STRIDE, 1, cs);
  const double total = card_total(cs);
  float2 w[UB_PPT];
#pragma unroll
  for (int j = 0; j < UB_PPT; ++j)
    w[j] = make_float2(unblocked_of(range[j].x, cs, total, hc.ab[j][0]), unblocked_of(range[j].y, cs, total, hc.ab[j][1]));
  for (int k = 0; k < count; ++k) {
    float2 next[UB_PPT], r[UB_PPT], next_cum[UB_PPT], next_wsum[UB_PPT];
    const int64_t c = first + (k + 1 < count ? k + 1 : k);
    fam_load(achieved, 2 * c + prev_actor[c], next);
    if constexpr (UPDATE) {
      fam_load((const float*)u.cumulative, c, next_cum);
      fam_load((const float*)u.weights, c, next_wsum);
    }
#pragma unroll
    for (int j = 0; j < UB_PPT; ++j) r[j] = make_float2(w[j].x * (a[j].x - e[j].x), w[j].y * (a[j].y - e[j].y));
    if constexpr (UPDATE) fam_update_row(u, d, first + k, r, cum, wsum);
    else fam_store(regrets, first + k, r);
#pragma unroll
    for (int j = 0; j < UB_PPT; ++j) {
      a[j] = next[j];
      if constexpr (UPDATE) { cum[j] = next_cum[j]; wsum[j] = next_wsum[j]; }
    }
  }
}

// policy[c] = max(cumulative[c], 0) / their sum over the family, fallback[c] where that is at most eps.
template <int MAXC>
__global__ __launch_bounds__(UB_BLOCK) void family_regret_matching_kernel(const float* __restrict__ cumulative,
                                                                           const float* __restrict__ fallback,
                                                                           const int64_t* __restrict__ child_offsets,
                                                                           const int64_t* __restrict__ child_count,
                                                                           float eps, float* __restrict__ policy) {
  const int64_t count64 = child_count[blockIdx.x];
  if (count64 <= 0 || count64 > MAXC) return;
  const int count = (int)count64;
  const int64_t first = child_offsets[blockIdx.x];
  float2 v[MAXC][UB_PPT], sum[UB_PPT];
  fam_load_children(cumulative, first, count, v);
#pragma unroll
  for (int k = 0; k < MAXC; ++k)
#pragma unroll
    for (int j = 0; j < UB_PPT; ++j)                        // like torch.clamp: NaN stays
      v[k][j] = make_float2(v[k][j].x < 0.f ? 0.f : v[k][j].x, v[k][j].y < 0.f ? 0.f : v[k][j].y);
  fam_sum(v, count, sum);
#pragma unroll
  for (int k = 0; k < MAXC; ++k) {
    if (k >= count) break;
    float2 f[UB_PPT];
    bool need = false;                                      // the fallback is read where some lane of the wave needs it
#pragma unroll
    for (int j = 0; j < UB_PPT; ++j) need = need || !(sum[j].x > eps) || !(sum[j].y > eps);
    if (__any(need)) fam_load(fallback, first + k, f);
#pragma unroll
    for (int j = 0; j < UB_PPT; ++j)
      v[k][j] = make_float2(sum[j].x > eps ? v[k][j].x / fmaxf(sum[j].x, eps) : f[j].x,
                            sum[j].y > eps ? v[k][j].y / fmaxf(sum[j].y, eps) : f[j].y);
    fam_store(policy, first + k, v[k]);
  }
}

// The reach-weighted mix of the average policy with the current one, then divided by its sum over the family where that
// is above eps; rows below `bottom` zero.
template <int MAXC>
__global__ __launch_bounds__(UB_BLOCK) void family_average_policy_kernel(
    const float* __restrict__ policy, float* __restrict__ policy_avg, const float* __restrict__ reach,
    const float* __restrict__ reach_avg, const int64_t* __restrict__ to_act, const int64_t* __restrict__ child_offsets,
    const int64_t* __restrict__ child_count, const float* __restrict__ old_p, const float* __restrict__ new_p,
    const float* __restrict__ tot_p, int64_t bottom, int64_t top, float eps) {
  const int64_t p = blockIdx.x;
  if (p < bottom) {
    const float2 none[UB_PPT] = {};
    fam_store(policy_avg, p, none);
  }
  const int64_t count64 = p < top ? child_count[p] : 0;
  if (count64 <= 0 || count64 > MAXC) return;
  const int count = (int)count64;
  const int64_t first = child_offsets[p], row = 2 * p + to_act[p];
  float2 r[UB_PPT], ra[UB_PPT], cur[MAXC][UB_PPT], avg[MAXC][UB_PPT], sum[UB_PPT];
  fam_load(reach, row, r);
  fam_load(reach_avg, row, ra);
  fam_load_children(policy, first, count, cur);
  fam_load_children((const float*)policy_avg, first, count, avg);
  const float o = *old_p, n = *new_p, tot = *tot_p;
  auto mix = [&](float rr, float rra, float c, float a) {
    const float reach_a = rra * o, reach_n = rr * n;
    const float num = reach_a * a + reach_n * c, den = reach_a + reach_n;
    const float unweighted = (o * a + n * c) / tot;
    return den > eps ? num / den : unweighted;
  };
#pragma unroll
  for (int k = 0; k < MAXC; ++k)
#pragma unroll
    for (int j = 0; j < UB_PPT; ++j)
      avg[k][j] = make_float2(mix(r[j].x, ra[j].x, cur[k][j].x, avg[k][j].x), mix(r[j].y, ra[j].y, cur[k][j].y, avg[k][j].y));
  fam_sum(avg, count, sum);
#pragma unroll
  for (int k = 0; k < MAXC; ++k) {
    if (k >= count) break;
#pragma unroll
    for (int j = 0; j < UB_PPT; ++j)
      avg[k][j] = make_float2(sum[j].x > eps ? avg[k][j].x / fmaxf(sum[j].x, eps) : avg[k][j].x,
                              sum[j].y > eps ? avg[k][j].y / fmaxf(sum[j].y, eps) : avg[k][j].y);
    fam_store(policy_avg, first + k, avg[k]);
  }
}

// Every row below the roots: the reach of both players, the root's times the policies of their actions on the way down
// (in that order: the roundings of a pass down the levels), zero where the hand is not allowed; and their ranges, root
// range x reach normalised, allowed_prob where the sum is at most eps.  The nodes of a root share their allowed hands.
// A row reads the policies on its way instead of the reach above it, so that all levels are one launch: they are read by
// many rows and come from the caches (8400 rows: five launches of 22 us, a level at a time, or one of 105; neighbouring rows
// on one XCD, so that they share the policies in its L2: 113, the stores like neighbours on different XCDs better).  From
// some 20 000 rows on the levels are faster, and the evaluator takes those.
constexpr int FAM_MAX_DEPTH = 64;
constexpr int FAM_BATCH = 4;                                // rows of policy requested together
__global__ __launch_bounds__(UB_BLOCK) void tree_reach_beliefs_kernel(
    float* __restrict__ reach, const float* __restrict__ policy, const uint8_t* __restrict__ allowed,
    const float* __restrict__ allowed_prob, const int64_t* __restrict__ parent_index,
    const int64_t* __restrict__ prev_actor, const int64_t* __restrict__ root_index, float* __restrict__ beliefs,
    int64_t n_roots, float eps) {
  __shared__ float red[2][OPS_WAVES];
  __shared__ uint32_t way[FAM_MAX_DEPTH];                   // rows from this one up to below the root, 2 row + actor
  const int64_t c = blockIdx.x + n_roots;
  const int64_t root = root_index[c];
  float2 x[2][UB_PPT], b[2][UB_PPT];
  uchar2 al[UB_PPT];
#pragma unroll
  for (int p = 0; p < 2; ++p) {
    fam_load((const float*)reach, 2 * root + p, x[p]);
    fam_load((const float*)beliefs, 2 * root + p, b[p]);
  }
  const uchar2* m2 = reinterpret_cast<const uchar2*>(allowed + c * P2_H);
#pragma unroll
  for (int j = 0; j < UB_PPT; ++j) {
    const int i = threadIdx.x + j * UB_BLOCK;
    al[j] = m2[i < P2_HPAIRS ? i : 0];
  }
  int steps = 0;
  for (int64_t r = c; r >= n_roots && steps < FAM_MAX_DEPTH; r = parent_index[r]) {
    if (threadIdx.x == 0) way[steps] = (uint32_t)(2 * r + prev_actor[r]);
    ++steps;
  }
  p2_sync_lds();
  for (int first = steps - 1; first >= 0; first -= FAM_BATCH) {
    float2 pol[FAM_BATCH][UB_PPT];
    uint32_t at[FAM_BATCH];
#pragma unroll
    for (int q = 0; q < FAM_BATCH; ++q) {
      at[q] = way[first - q >= 0 ? first - q : 0];          // past the end: the last one again, not used
      fam_load(policy, at[q] >> 1, pol[q]);
    }
#pragma unroll
    for (int q = 0; q < FAM_BATCH; ++q) {
      if (first - q < 0) break;
      if (at[q] & 1) {
#pragma unroll
        for (int j = 0; j < UB_PPT; ++j) { x[1][j].x *= pol[q][j].x; x[1][j].y *= pol[q][j].y; }
      } else {
#pragma unroll
        for (int j = 0; j < UB_PPT; ++j) { x[0][j].x *= pol[q][j].x; x[0][j].y *= pol[q][j].y; }
      }
    }
  }
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
#pragma unroll
  for (int p = 0; p < 2; ++p) {
    float local = 0.f;
#pragma unroll
    for (int j = 0; j < UB_PPT; ++j) {
      x[p][j] = make_float2(al[j].x ? x[p][j].x : 0.f, al[j].y ? x[p][j].y : 0.f);
      b[p][j] = make_float2(b[p][j].x * x[p][j].x, b[p][j].y * x[p][j].y);
      if (threadIdx.x + j * UB_BLOCK < P2_HPAIRS) local += b[p][j].x + b[p][j].y;
    }
    fam_store(reach, 2 * c + p, x[p]);
    local = p2_wave_sum(local);
    if (lane == 0) red[p][wave] = local;
  }
  p2_sync_lds();
#pragma unroll
  for (int p = 0; p < 2; ++p) {
    float total = 0.f;
#pragma unroll
    for (int w = 0; w < OPS_WAVES; ++w) total += red[p][w];
    if (total > eps) {
#pragma unroll
      for (int j = 0; j < UB_PPT; ++j) b[p][j] = make_float2(b[p][j].x / total, b[p][j].y / total);
    } else {
      fam_load(allowed_prob, c, b[p]);
    }
    fam_store(beliefs, 2 * c + p, b[p]);
  }
}

// Parents base .. base + gridDim.x - 1, all of one level: their values from their children's.  The actor's weight of a
// child is its policy, the other player's the share of the actor's compatible range that goes there:
// unblocked(range x policy) / unblocked(range), 0 where the latter is at most eps.
template <int MAXC>
__global__ __launch_bounds__(UB_BLOCK) void level_expected_values_kernel(
    float* __restrict__ values, const float* __restrict__ policy, const float* __restrict__ beliefs,
    const int64_t* __restrict__ to_act, const int64_t* __restrict__ child_offsets,
    const int64_t* __restrict__ child_count, int64_t base, float eps) {
  __shared__ __align__(8) float t[MAXC + 1][UB_STRIDE];
  __shared__ double cs[(MAXC + 1) * P2_CARDS];
  __shared__ double totals[MAXC + 1];
  const int64_t p = base + blockIdx.x;
  const int64_t count64 = child_count[p];
  if (count64 <= 0 || count64 > MAXC) return;               // a leaf keeps its values
  const int count = (int)count64;
  const int64_t first = child_offsets[p];
  const int actor = (int)to_act[p];
  float2 range[UB_PPT], w[MAXC][UB_PPT], own[UB_PPT], other[UB_PPT];
  fam_load(beliefs, 2 * p + actor, range);
  fam_load_children(policy, first, count, w);
  fam_load((const float*)values, 2 * first + actor, own);
  fam_load((const float*)values, 2 * first + (actor ^ 1), other);
  HandCards hc;
  hand_cards_init(hc);
  stage_row(range, t[0]);
#pragma unroll
  for (int k = 0; k < MAXC; ++k) {
    if (k >= count) break;
    float2 marginal[UB_PPT];
#pragma unroll
    for (int j = 0; j < UB_PPT; ++j) marginal[j] = make_float2(range[j].x * w[k][j].x, range[j].y * w[k][j].y);
    stage_row(marginal, t[k + 1]);
  }
  p2_sync_lds();
  card_sums_multi(t[0], UB_STRIDE, count + 1, cs);
  for (int v = threadIdx.x >> 6; v <= count; v += UB_WAVES) {   // a vector's total in one wave, not in every one
    const double total = card_total(cs + v * P2_CARDS);
    if ((threadIdx.x & 63) == 0) totals[v] = total;
  }
  p2_sync_lds();
  float2 den[UB_PPT], sum_own[UB_PPT], sum_other[UB_PPT];
#pragma unroll
  for (int j = 0; j < UB_PPT; ++j) {
    den[j] = make_float2(unblocked_of(range[j].x, cs, totals[0], hc.ab[j][0]),
                         unblocked_of(range[j].y, cs, totals[0], hc.ab[j][1]));
    sum_own[j] = sum_other[j] = make_float2(0.f, 0.f);
  }
#pragma unroll
  for (int k = 0; k < MAXC; ++k) {
    if (k >= count) break;
    float2 next_own[UB_PPT], next_other[UB_PPT];
    const int64_t c = first + (k + 1 < count ? k + 1 : k);
    fam_load((const float*)values, 2 * c + actor, next_own);
    fam_load((const float*)values, 2 * c + (actor ^ 1), next_other);
    const double* csk = cs + (k + 1) * P2_CARDS;
    const double total = totals[k + 1];
#pragma unroll
    for (int j = 0; j < UB_PPT; ++j) {
      const float m0 = range[j].x * w[k][j].x, m1 = range[j].y * w[k][j].y;
      const float o0 = den[j].x > eps ? unblocked_of(m0, csk, total, hc.ab[j][0]) / den[j].x : 0.f;
      const float o1 = den[j].y > eps ? unblocked_of(m1, csk, total, hc.ab[j][1]) / den[j].y : 0.f;
      sum_own[j].x += own[j].x * w[k][j].x;
      sum_own[j].y += own[j].y * w[k][j].y;
      sum_other[j].x += other[j].x * o0;
      sum_other[j].y += other[j].y * o1;
      own[j] = next_own[j];
      other[j] = next_other[j];
    }
  }
  fam_store(values, 2 * p + actor, sum_own);
  fam_store(values, 2 * p + (actor ^ 1), sum_other);
}

}  // namespace p2

extern "C" {

int p2hip_family_regrets(const float* achieved, const float* expected, const float* beliefs, const int64_t* to_act,
                         const int64_t* prev_actor, const int64_t* child_offsets, const int64_t* child_count,
                         int64_t bottom, int64_t top, float* regrets, void* stream) {
  const int64_t rows = bottom > top ? bottom : top;
  P2_REQ(bottom >= 0 && top >= 0 && rows <= 0x7FFFFFFF);
  if (rows == 0) return 0;
  P2_REQ(achieved && expected && beliefs && to_act && prev_actor && child_offsets && child_count && regrets);
  P2_REQ(p2_aligned8(achieved) && p2_aligned8(expected) && p2_aligned8(beliefs) && p2_aligned8(regrets));
  hipLaunchKernelGGL(p2::family_regrets_kernel<false>, dim3((unsigned)rows), dim3(p2::UB_BLOCK), 0, P2_ST, achieved,
                     expected, beliefs, to_act, prev_actor, child_offsets, child_count, bottom, top, regrets, p2::FamUpdate{});
  P2_LAUNCH_CHECK();
  return 0;
}

int p2hip_family_regret_update(const float* achieved, const float* expected, const float* beliefs, const int64_t* to_act,
                               const int64_t* prev_actor, const int64_t* child_offsets, const int64_t* child_count,
                               int64_t bottom, int64_t top, float* cumulative, float* weights, const float* t_alpha_num,
                               const float* t_beta_num, const float* t_alpha_den, const float* t_beta_den, int apply_dcfr,
                               int cfr_plus, void* stream) {
  const int64_t rows = bottom > top ? bottom : top;
  P2_REQ(bottom >= 0 && top >= 0 && rows <= 0x7FFFFFFF);
  if (rows == 0) return 0;
  P2_REQ(achieved && expected && beliefs && to_act && prev_actor && child_offsets && child_count && cumulative && weights);
  P2_REQ(!apply_dcfr || (t_alpha_num && t_beta_num && t_alpha_den && t_beta_den));
  P2_REQ(p2_aligned8(achieved) && p2_aligned8(expected) && p2_aligned8(beliefs) && p2_aligned8(cumulative) &&
         p2_aligned8(weights));
  const p2::FamUpdate u = {cumulative, weights, t_alpha_num, t_beta_num, t_alpha_den, t_beta_den, apply_dcfr, cfr_plus};
  hipLaunchKernelGGL(p2::family_regrets_kernel<true>, dim3((unsigned)rows), dim3(p2::UB_BLOCK), 0, P2_ST, achieved, expected,
                     beliefs, to_act, prev_actor, child_offsets, child_count, bottom, top, (float*)nullptr, u);
  P2_LAUNCH_CHECK();
  return 0;
}

int p2hip_family_regret_matching(const float* cumulative, const float* fallback, const int64_t* child_offsets,
                                 const int64_t* child_count, int64_t top, int max_children, float eps, float* policy,
                                 void* stream) {
  P2_REQ(top >= 0 && top <= 0x7FFFFFFF && max_children >= 0 && max_children <= p2::FAM_MAX_CHILDREN);
  if (top == 0) return 0;
  P2_REQ(cumulative && fallback && child_offsets && child_count && policy);
  P2_REQ(p2_aligned8(cumulative) && p2_aligned8(fallback) && p2_aligned8(policy));
  auto kernel = max_children <= 5 ? p2::family_regret_matching_kernel<5> : p2::family_regret_matching_kernel<8>;
  hipLaunchKernelGGL(kernel, dim3((unsigned)top), dim3(p2::UB_BLOCK), 0, P2_ST, cumulative, fallback, child_offsets,
                     child_count, eps, policy);
  P2_LAUNCH_CHECK();
  return 0;
}

int p2hip_family_average_policy(const float* policy, float* policy_avg, const float* reach, const float* reach_avg,
                                const int64_t* to_act, const int64_t* child_offsets, const int64_t* child_count,
                                const float* old_w, const float* new_w, const float* total_w, int64_t bottom, int64_t top,
                                int max_children, float eps, void* stream) {
  const int64_t rows = bottom > top ? bottom : top;
  P2_REQ(bottom >= 0 && top >= 0 && rows <= 0x7FFFFFFF && max_children >= 0 && max_children <= p2::FAM_MAX_CHILDREN);
  if (rows == 0) return 0;
  P2_REQ(policy && policy_avg && reach && reach_avg && to_act && child_offsets && child_count && old_w && new_w && total_w);
  P2_REQ(p2_aligned8(policy) && p2_aligned8(policy_avg) && p2_aligned8(reach) && p2_aligned8(reach_avg));
  auto kernel = max_children <= 5 ? p2::family_average_policy_kernel<5> : p2::family_average_policy_kernel<8>;
  hipLaunchKernelGGL(kernel, dim3((unsigned)rows), dim3(p2::UB_BLOCK), 0, P2_ST, policy, policy_avg, reach, reach_avg,
                     to_act, child_offsets, child_count, old_w, new_w, total_w, bottom, top, eps);
  P2_LAUNCH_CHECK();
  return 0;
}

int p2hip_tree_reach_beliefs(float* reach, const float* policy, const uint8_t* allowed, const float* allowed_prob,
                             const int64_t* parent_index, const int64_t* prev_actor, const int64_t* root_index,
                             float* beliefs, int64_t n_roots, int64_t total, int depth, float eps, void* stream) {
  P2_REQ(n_roots >= 0 && total >= n_roots && total <= 0x3FFFFFFF && depth >= 0 && depth <= p2::FAM_MAX_DEPTH);
  if (total == n_roots) return 0;
  P2_REQ(reach && policy && allowed && allowed_prob && parent_index && prev_actor && root_index && beliefs);
  P2_REQ(p2_aligned8(reach) && p2_aligned8(policy) && p2_aligned8(allowed_prob) && p2_aligned8(beliefs) &&
         (reinterpret_cast<uintptr_t>(allowed) & 1u) == 0);
  hipLaunchKernelGGL(p2::tree_reach_beliefs_kernel, dim3((unsigned)(total - n_roots)), dim3(p2::UB_BLOCK), 0, P2_ST, reach,
                     policy, allowed, allowed_prob, parent_index, prev_actor, root_index, beliefs, n_roots, eps);
  P2_LAUNCH_CHECK();
  return 0;
}

int p2hip_level_expected_values(float* values, const float* policy, const float* beliefs, const int64_t* to_act,
                                const int64_t* child_offsets, const int64_t* child_count, int64_t base, int64_t n,
                                int max_children, float eps, void* stream) {
  P2_REQ(base >= 0 && n >= 0 && n <= 0x7FFFFFFF && max_children >= 0 && max_children <= p2::FAM_MAX_CHILDREN);
  if (n == 0) return 0;
  P2_REQ(values && policy && beliefs && to_act && child_offsets && child_count);
  P2_REQ(p2_aligned8(values) && p2_aligned8(policy) && p2_aligned8(beliefs));
  auto kernel = max_children <= 5 ? p2::level_expected_values_kernel<5> : p2::level_expected_values_kernel<8>;
  hipLaunchKernelGGL(kernel, dim3((unsigned)n), dim3(p2::UB_BLOCK), 0, P2_ST, values, policy, beliefs, to_act,
                     child_offsets, child_count, base, eps);
  P2_LAUNCH_CHECK();
  return 0;
}

}  // extern "C"
