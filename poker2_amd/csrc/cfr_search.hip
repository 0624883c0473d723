// The iteration of a search on a few roots, fused per family: what cfr_iteration_kernel does in three walks over a
// work item's families is one top-down walk here, and a bottom-up walk over the families that have a child with
// children of its own.  Per family:
//   opponent's unblocked mass at the parent, regrets, discounting, regret matching -> policy, which stays in LDS;
//   average-policy mix, reach, ranges (rows with children only);
//   the showdown child, its two ranges handed over through LDS: neither is ever stored;
//   if every child is a leaf whose value is known by now: the backup, from the same policy and the values just made.
// A lean iteration with two reach_avg buffers (see cfr_iter.hip), the same arithmetic in the same order: the state
// is bit-identical to that kernel's.
//
// The regret part reads the parent's ranges as the previous iteration left them, which the family above would
// overwrite: the ranges alternate between two buffers like reach_avg does (leaf_prev read, leaf_next written).
//
// What bounds it: with few roots nothing fills the chip, and an iteration lasts as long as its longest chain of
// families, each a chain of dependent steps.  Twelve waves take a family (one pair of hands per lane, four waves for
// the prefix of the sorted ranges while eight take the card scans), rows are requested one child ahead, the parent's
// before the first barrier, and a tier of work items costs one launch downwards and one upwards.  Microseconds per
// iteration, three walks -> one over the same work items: three-raise river tree (105 nodes) 1 root 299 -> 211 (141
// with the tree cut at every level), 64 roots 386 -> 270; depth-2 tree 1 root 81 -> 57, 128 roots 110 -> 95; 64 mixed
// roots to depth 5 368 -> 240.  All these are roots with equal stacks, or happen to have no parent with two showdown
// children: one such parent keeps the batch on the three walks.  Tried: all children's rows requested at once instead
// of one child ahead (211 -> 231; with a branch per child 218).
//
// Why only few roots: the showdown's tables leave room for two workgroups per CU at most, and the barriers of a
// family (fourteen) drain what rows are in flight.  4096 roots: 11.3 ms per iteration against 9.7 of the three walks,
// although it moves 5 % fewer bytes (45.3 GB against 47.4); as four waves with six hands per lane and 256
// registers the same walk took 11.7 ms there and 291 us on one root.
#pragma once
#include "cfr_iter.hip"

namespace p2 {

// Twelve waves, one pair of hands per lane: waves 3w, 3w + 1, 3w + 2 own the three runs (64, 64 and 38 pairs) that a
// lane of wave w owns in cfr_iteration_kernel, so that sums over hands can be taken in the same order.
constexpr int SR_BLOCK = 768;
constexpr int SR_WAVES = SR_BLOCK / 64;
constexpr int SR_MAXC = 5;   // children per parent: more take the three-walk kernel
static_assert(SR_WAVES == 3 * IT_WAVES, "three runs per wave of the three-walk kernel");

constexpr int SR_SUMS = 13;
struct SearchFam {      // one family: FamWin's entries, and the stakes of its showdown child
  int p, first, ca, kinds;
  int rs;
  float pot0, pot1, scale;
};
struct SearchLds {
  float pol[SR_MAXC][IT_VSTRIDE];      // the children's new policies; a lane reads only its own pair: no barrier
  union {
    float vecs[SR_MAXC + 3][IT_VSTRIDE];   // the last two: the showdown child's values, in the lanes' own pairs
    ShowdownLds sd;
    float part[SR_SUMS][SR_BLOCK];
  } u;
  double cs[(SR_MAXC + 1) * P2_CARDS];
  float red[SR_SUMS][IT_WAVES];
  SearchFam fam[64];                   // a window of the item's family list
};
static_assert(sizeof(ShowdownLds) >= sizeof(float) * (SR_MAXC + 3) * IT_VSTRIDE &&
                  sizeof(float2) * 2 * P2_H <= sizeof(float) * (SR_MAXC + 1) * IT_VSTRIDE,
              "values of the showdown child: inside the union, behind the sorted ranges and their prefix");

struct SearchRows {
  const float* leaf_prev;   // [total,2,H] beliefs (beliefs_avg under cfr_avg) of the previous iteration
  float* leaf_next;         // the buffer this iteration writes
};

// A copy of a per-lane value that the optimiser cannot relate to the original: what is computed from it stays
// inside the loop iteration instead of occupying registers through the whole walk (the table slice's LDS addresses,
// the offsets of a card's combos).
template <class T>
__device__ __forceinline__ T fresh(T x) {
  asm volatile("" : "+v"(x));
  return x;
}

__device__ __forceinline__ int wave_of_block() { return __builtin_amdgcn_readfirstlane((int)threadIdx.x >> 6); }

struct SLane {
  uint32_t off;  // byte offset of the pair in a row, clamped into it where the lane has none
  bool ok;       // the lane has a pair
  uint32_t ab;   // cards of the two hands: a0 | b0 << 8 | a1 << 16 | b1 << 24
};
__device__ __forceinline__ void slane_init(SLane& ln) {
  const int lane = threadIdx.x & 63, wave = wave_of_block();
  const int run = wave % 3, q = run * 64 + lane, i = (wave / 3) * IT_WAVE_PAIRS + q;
  ln.ok = run < 2 || (q < IT_WAVE_PAIRS && i < P2_HPAIRS);
  const int idx = ln.ok ? i : P2_HPAIRS - 1, h = 2 * idx;
  ln.off = (uint32_t)idx * 8u;
  ln.ab = (uint32_t)p2_combo.a[h] | ((uint32_t)p2_combo.b[h] << 8) | ((uint32_t)p2_combo.a[h + 1] << 16) |
          ((uint32_t)p2_combo.b[h + 1] << 24);
}
// (unsigned byte offsets: a row's address stays in scalar registers, the lane adds 32 bits)
__device__ __forceinline__ float2 sld(const float* base, int64_t row, const SLane& ln, int mask = -1) {
  const char* at = reinterpret_cast<const char*>(base + row * P2_H);
  const float2 v = *reinterpret_cast<const float2*>(at + (ln.off & (uint32_t)mask));
  return ln.ok ? v : make_float2(0.f, 0.f);
}
__device__ __forceinline__ void sst(float* base, int64_t row, float2 v, const SLane& ln) {
  if (ln.ok) *reinterpret_cast<float2*>(reinterpret_cast<char*>(base + row * P2_H) + ln.off) = v;
}
__device__ __forceinline__ void sput(float* vec, float2 v, const SLane& ln) {
  if (ln.ok) *reinterpret_cast<float2*>(reinterpret_cast<char*>(vec) + ln.off) = v;
}
__device__ __forceinline__ float2 sget(const float* vec, const SLane& ln) {
  const float2 v = *reinterpret_cast<const float2*>(reinterpret_cast<const char*>(vec) + ln.off);
  return ln.ok ? v : make_float2(0.f, 0.f);
}
__device__ __forceinline__ float2 sunblocked(float2 t, const double* cs, double S, uint32_t ab) {
  const double x = S - cs[ab & 0xFFu] - cs[(ab >> 8) & 0xFFu] + (double)t.x;
  const double y = S - cs[(ab >> 16) & 0xFFu] - cs[ab >> 24] + (double)t.y;
  return make_float2(fmaxf((float)x, 0.f), fmaxf((float)y, 0.f));
}

// Sums of N per-lane values over the block, in the order of cfr_iteration_kernel's block_sums: a lane's three runs,
// the lanes of a wave, the four waves.  The values pass through LDS, where N * 4 wave scans are dealt to twelve waves.
template <int N>
__device__ __forceinline__ void search_sums(float (&v)[N], SearchLds& L) {
  const int tid = fresh((int)threadIdx.x), lane = tid & 63, wave = wave_of_block();
#pragma unroll
  for (int q = 0; q < N; ++q) L.u.part[q][tid] = v[q];
  p2_sync_lds();
#pragma unroll
  for (int t0 = 0; t0 < N * IT_WAVES; t0 += SR_WAVES) {
    const int task = t0 + wave;
    if (task < N * IT_WAVES) {
      const int q = task / IT_WAVES, w = task % IT_WAVES;
      const float* x = &L.u.part[q][w * 192 + lane];
      const float s = p2_wave_sum(x[0] + x[64] + x[128]);
      if (lane == 0) L.red[q][w] = s;
    }
  }
  p2_sync_lds();
#pragma unroll
  for (int q = 0; q < N; ++q) {
    float s = 0.f;
#pragma unroll
    for (int w = 0; w < IT_WAVES; ++w) s += L.red[q][w];
    v[q] = s;
  }
}

// A lane's slice of the board's strength table: two consecutive sorted positions of its own (663 lanes), and the card
// lists of the cards its wave scans (waves 4..11: card wave - 4 + 8 * i), two 16-bit entries to a register.
constexpr int SR_SCAN_WAVE0 = 4, SR_SCAN_WAVES = SR_WAVES - SR_SCAN_WAVE0, SR_SCANS = 7;
static_assert(SR_SCANS * SR_SCAN_WAVES >= P2_CARDS && SR_SCAN_WAVE0 == SD_WAVES, "cards dealt to the scanning waves");
struct SearchTable {
  uint32_t perm, ab, lr[2], cidx[2], clist[(SR_SCANS + 1) / 2];
};
__device__ __forceinline__ void search_table(const uint8_t* __restrict__ tab, SearchTable& T) {
  const int t = (int)threadIdx.x < P2_HPAIRS ? (int)threadIdx.x : 0;
  T.perm = reinterpret_cast<const uint32_t*>(tab + SD_OFF_PERM)[t];
  const uint32_t* lr = reinterpret_cast<const uint32_t*>(tab + SD_OFF_LR) + 2 * t;
  T.lr[0] = lr[0]; T.lr[1] = lr[1];
  const uint32_t* cx = reinterpret_cast<const uint32_t*>(tab + SD_OFF_CIDX) + 2 * t;
  T.cidx[0] = cx[0]; T.cidx[1] = cx[1];
  const uint16_t* clist = reinterpret_cast<const uint16_t*>(tab + SD_OFF_CLIST);
  const int lane = threadIdx.x & 63, wave = wave_of_block();
  uint32_t cl[SR_SCANS + 1];
#pragma unroll
  for (int i = 0; i < SR_SCANS; ++i) {
    const int c = wave - SR_SCAN_WAVE0 + SR_SCAN_WAVES * i;
    const uint32_t x = clist[(c >= 0 && c < P2_CARDS ? c : 0) * 51 + (lane < 51 ? lane : 50)];
    cl[i] = lane < 51 && c >= 0 && c < P2_CARDS ? x : 0xFFFFu;
  }
  cl[SR_SCANS] = 0xFFFFu;
#pragma unroll
  for (int q = 0; q < (SR_SCANS + 1) / 2; ++q) T.clist[q] = cl[2 * q] | (cl[2 * q + 1] << 16);
  const int h0 = (int)(T.perm & 0x7FFFu), h1 = (int)((T.perm >> 16) & 0x7FFFu);
  T.ab = (uint32_t)p2_combo.a[h0] | ((uint32_t)p2_combo.b[h0] << 8) | ((uint32_t)p2_combo.a[h1] << 16) |
         ((uint32_t)p2_combo.b[h1] << 24);
}

// Showdown values of both players from the ranges in L.u.vecs[0] / [1]; EVs in combo order in L.u.sd.v, as (hero 0,
// hero 1).  showdown_eval's arithmetic: four waves take the prefix of the sorted ranges with its six positions per
// lane while the other eight take the card scans.  Begins behind a barrier that covers the ranges, ends with one.
__device__ __forceinline__ void search_showdown(const SearchTable& T0, SearchLds& L, float pot0, float pot1, float scale) {
  ShowdownLds& s = L.u.sd;
  const int tid = fresh((int)threadIdx.x), lane = tid & 63, wave = wave_of_block();
  const bool mine = tid < P2_HPAIRS;
  const uint32_t perm = fresh(T0.perm);
  const uint32_t p0 = perm & 0xFFFFu, p1 = perm >> 16;
  const int h0 = (int)(p0 & 0x7FFFu), h1 = (int)(p1 & 0x7FFFu);
  const float2 va = make_float2(L.u.vecs[1][h0], L.u.vecs[0][h0]), vb = make_float2(L.u.vecs[1][h1], L.u.vecs[0][h1]);
  p2_sync_lds();
  if (mine) {
    s.v[2 * tid] = va;
    s.v[2 * tid + 1] = vb;
  }
  p2_sync_lds();
  auto scan_cards = [&](int from) {
    float2 x[4];
#pragma unroll
    for (int q = 0; q < 4; ++q) {
      const int i = from + q < SR_SCANS ? from + q : SR_SCANS - 1;
      const uint32_t cl = fresh(T0.clist[i / 2]), pos = i & 1 ? cl >> 16 : cl & 0xFFFFu;
      const float2 y = s.v[pos < (uint32_t)P2_H ? pos : 0u];
      x[q] = make_float2(pos < (uint32_t)P2_H ? y.x : 0.f, pos < (uint32_t)P2_H ? y.y : 0.f);
    }
    p2_wave_scan_incl4(x[0].x, x[0].y, x[1].x, x[1].y);
    p2_wave_scan_incl4(x[2].x, x[2].y, x[3].x, x[3].y);
#pragma unroll
    for (int q = 0; q < 4; ++q) {
      const int c = wave - SR_SCAN_WAVE0 + SR_SCAN_WAVES * (from + q);
      if (from + q < SR_SCANS && c < P2_CARDS) {
        if (lane < 51) s.Pc[c][lane + 1] = x[q];
        if (lane == 0) s.Pc[c][0] = make_float2(0.f, 0.f);
      }
    }
  };
  const int k0 = tid * SD_PPT;
  float local[2] = {0.f, 0.f}, incl[2] = {0.f, 0.f};
  if (wave < SR_SCAN_WAVE0) {
#pragma unroll
    for (int i = 0; i < SD_PPT; ++i) {
      const float2 y = s.v[k0 < P2_H ? k0 + i : 0];   // 1326 = 221 * 6: a lane is inside the table or past its end
      local[0] += k0 < P2_H ? y.x : 0.f;
      local[1] += k0 < P2_H ? y.y : 0.f;
    }
#pragma unroll
    for (int p = 0; p < 2; ++p) {
      incl[p] = p2_wave_scan_incl(local[p]);
      if (lane == 63) s.part[p][wave] = incl[p];
    }
  } else {
    scan_cards(0);
  }
  p2_sync_lds();
  if (wave < SR_SCAN_WAVE0) {
    float base0 = 0.f, base1 = 0.f;
    for (int w = 0; w < wave; ++w) { base0 += s.part[0][w]; base1 += s.part[1][w]; }
    float run0 = base0 + (incl[0] - local[0]), run1 = base1 + (incl[1] - local[1]);
#pragma unroll
    for (int i = 0; i < SD_PPT; ++i) {
      if (k0 + i <= P2_H) s.P[k0 + i] = make_float2(run0, run1);
      const float2 y = s.v[k0 < P2_H ? k0 + i : 0];
      run0 += k0 < P2_H ? y.x : 0.f;
      run1 += k0 < P2_H ? y.y : 0.f;
    }
  } else {
    scan_cards(4);
  }
  p2_sync_lds();
  if (mine) {
    const float r0 = pot0 / scale, r1 = pot1 / scale;
    const uint32_t ab = fresh(T0.ab);
    // s.v is dead by now: the card scans that read it are behind the barrier
    s.v[h0] = showdown_hand(s, p0, fresh(T0.lr[0]), fresh(T0.cidx[0]), ab & 0xFFFFu, va.x, va.y, r0, r1);
    s.v[h1] = showdown_hand(s, p1, fresh(T0.lr[1]), fresh(T0.cidx[1]), ab >> 16, vb.x, vb.y, r0, r1);
  }
  p2_sync_lds();
}

// The window of 64 families that starts at list position `base`, by the first wave.  Begins and ends with a barrier.
__device__ __forceinline__ void search_window(SearchLds& L, const IterArgs& A, int64_t pp0, int nfam, int base) {
  p2_sync_lds();
  if (threadIdx.x < 64) {
    FamWin F;
    fam_load<SR_MAXC, true, true>(F, A, pp0, nfam, base);
    SearchFam f = {F.p, F.first, F.ca, F.kinds, F.rs, 0.f, 0.f, 1.f};
    const uint32_t k = (uint32_t)F.kinds, sd = (k >> 1) & 0x5555u & ~(k >> 16);
    if (base + (int)threadIdx.x < nfam && sd) {
      const int64_t c = F.first + (__builtin_ctz(sd) >> 1);
      f.pot0 = A.potential[2 * c];
      f.pot1 = A.potential[2 * c + 1];
      f.scale = A.scale[c];
    }
    L.fam[threadIdx.x] = f;
  }
  p2_sync_lds();
}
__device__ __forceinline__ Fam search_fam(const SearchLds& L, int slot) {
  const SearchFam& x = L.fam[slot];
  Fam f;
  f.p = __builtin_amdgcn_readfirstlane(x.p);
  f.first = __builtin_amdgcn_readfirstlane(x.first);
  const int ca = __builtin_amdgcn_readfirstlane(x.ca);
  f.cnt = ca & 0xFF;
  f.actor = (ca >> 8) & 0xFF;
  f.kinds = __builtin_amdgcn_readfirstlane(x.kinds);
  f.rs = __builtin_amdgcn_readfirstlane(x.rs);
  return f;
}

template <bool CA>
__global__ __launch_bounds__(SR_BLOCK, 3) void cfr_search_kernel(IterArgs A, SearchRows B) {
  constexpr int MAXC = SR_MAXC;
  __shared__ SearchLds L;
  const int64_t w = blockIdx.x;
  const int64_t r = A.item_root ? A.item_root[w] : w;
  const bool top = A.item_top ? A.item_top[w] != 0 : true;
  const int64_t pp0 = A.root_parent_offsets[w];
  const int nfam = (int)(A.root_parent_offsets[w + 1] - pp0);

  SLane ln;
  slane_init(ln);
  int base = 0;
  search_window(L, A, pp0, nfam, base);

  const float f_an = A.fscal[0], f_bn = A.fscal[1], f_ad = A.fscal[2], f_bd = A.fscal[3];
  const float mix_old = A.fscal[4], mix_new = A.fscal[5], mix_total = A.fscal[6], mix_inv = A.fscal[7];
  const float y_ad = p2_recip_wide(f_ad), y_bd = p2_recip_wide(f_bd), y_mix = p2_recip_wide(mix_total);
  const int64_t t_now = A.iscal[0];
  const bool apply_dcfr = A.iscal[1] != 0, cfr_plus = A.iscal[2] != 0, avg_copy = A.iscal[3] != 0;
  const bool update_avg = A.iscal[5] != 0, linear = A.iscal[7] != 0;

  auto mixed_value = [&](float2 old, float2 now) {
    return make_float2((old.x * mix_old + now.x * mix_new) * mix_inv, (old.y * mix_old + now.y * mix_new) * mix_inv);
  };

  // Backup of one family.  `ab`: the actor's range at the parent; the children's policies are in L.pol; `sdbits`
  // marks the showdown child whose values wait in LDS (0: every child's values are read).
  auto backup = [&](const Fam& f, bool root_family, float2 ab, int sdbits) {
    const int64_t p = f.p, first = f.first;
    const int cnt = f.cnt, actor = f.actor;
    sput(L.u.vecs[0], ab, ln);
    float2 v0, v1, a0, a1;      // the next child's values and running averages: one child ahead
    auto request = [&](int k) {
      const int64_t c = first + k;
      const int m = const_mask(f, k);
      v0 = v1 = a0 = a1 = make_float2(0.f, 0.f);
      if (!((sdbits >> (2 * k)) & 1)) {
        v0 = sld(A.latest, c * 2, ln, m);
        v1 = sld(A.latest, c * 2 + 1, ln, m);
      }
      if (update_avg) {
        a0 = sld(A.values_avg, c * 2, ln, m);
        a1 = sld(A.values_avg, c * 2 + 1, ln, m);
      }
    };
    request(0);
#pragma unroll 1
    for (int k = 0; k < cnt; ++k) sput(L.u.vecs[1 + k], mul2(ab, sget(L.pol[k], ln)), ln);
    p2_sync_lds();
    card_sums_block<SR_BLOCK>(L.u.vecs[0], IT_VSTRIDE, cnt + 1, L.cs, fresh((int)threadIdx.x));
    const uint32_t cards = fresh(ln.ab);
    const float2 dn = sunblocked(ab, L.cs, card_total(L.cs), cards);
    float2 vp[2] = {make_float2(0.f, 0.f), make_float2(0.f, 0.f)};
#pragma unroll 1
    for (int k = 0; k < cnt; ++k) {
      const int64_t c = first + k;
      float2 u0 = v0, u1 = v1;
      const float2 b0 = a0, b1 = a1;
      if (k + 1 < cnt) request(k + 1);
      if ((sdbits >> (2 * k)) & 1) {
        u0 = sget(L.u.vecs[MAXC + 1], ln);
        u1 = sget(L.u.vecs[MAXC + 2], ln);
      }
      if (update_avg) {
        const float2 x0 = mixed_value(b0, u0), x1 = mixed_value(b1, u1);
        if (const_mask(f, k) == 0) {
          if (threadIdx.x == 0) {
            p2_row2(A.values_avg, c * 2)[0] = x0;
            p2_row2(A.values_avg, c * 2 + 1)[0] = x1;
          }
        } else {
          sst(A.values_avg, c * 2, x0, ln);
          sst(A.values_avg, c * 2 + 1, x1, ln);
        }
      }
      const float2 pk = sget(L.pol[k], ln);
      const float2 nm = sunblocked(mul2(ab, pk), L.cs + (1 + k) * P2_CARDS, card_total(L.cs + (1 + k) * P2_CARDS), cards);
      const float2 wo = make_float2(dn.x > 1e-5f ? p2_div(nm.x, dn.x) : 0.f, dn.y > 1e-5f ? p2_div(nm.y, dn.y) : 0.f);
      const float2 w0 = actor == 0 ? pk : wo, w1 = actor == 0 ? wo : pk;
      vp[0].x += u0.x * w0.x; vp[0].y += u0.y * w0.y;
      vp[1].x += u1.x * w1.x; vp[1].y += u1.y * w1.y;
    }
    sst(A.latest, p * 2, vp[0], ln);
    sst(A.latest, p * 2 + 1, vp[1], ln);
    if (root_family && update_avg) {   // the root is nobody's child: its average values move here
#pragma unroll
      for (int pl = 0; pl < 2; ++pl)
        sst(A.values_avg, p * 2 + pl, mixed_value(sld(A.values_avg, p * 2 + pl, ln), vp[pl]), ln);
    }
    p2_sync_lds();  // the staged vectors and L.cs are rewritten by the next family
  };

  if (A.phases & PHASE_12) {
    const bool take_sample = A.t_sample[r] == t_now;
    // the root's leaf ranges (CA: the average ones) scale every leaf range below it
    const float2 la0 = sld(B.leaf_prev, r * 2, ln), la1 = sld(B.leaf_prev, r * 2 + 1, ln);
    if (top) {
      sst(B.leaf_next, r * 2, la0, ln);
      sst(B.leaf_next, r * 2 + 1, la1, ln);
    }
    const uchar2 am = *reinterpret_cast<const uchar2*>(A.allowed + r * P2_H + (ln.off >> 2));
    const bool am0 = am.x != 0, am1 = am.y != 0;
    auto allowed2 = [&](float2 v) { return make_float2(am0 ? v.x : 0.f, am1 ? v.y : 0.f); };
    SearchTable table = {};
    if (A.tables && A.root_showdown_offsets[w + 1] > A.root_showdown_offsets[w])
      search_table(A.tables + r * SD_TABLE_BYTES, table);
    if (top) {
      // the root row's regret is zero (never positive): only its weight sum moves
      float2 ws = sld(A.wsum, r, ln);
      if (apply_dcfr) {
        ws = make_float2(ws.x * f_bn, ws.y * f_bn);
        ws = make_float2(p2_quotient(ws.x, f_bd, y_bd), p2_quotient(ws.y, f_bd, y_bd));
      }
      sst(A.wsum, r, make_float2(ws.x + 1.0f, ws.y + 1.0f), ln);
    }
    for (int i = 0; i < nfam; ++i) {
      if (i >= base + 64) search_window(L, A, pp0, nfam, base = i);
      const Fam f = search_fam(L, i - base);
      ln.off = fresh(ln.off);
      ln.ab = fresh(ln.ab);
      const int64_t p = f.p, first = f.first;
      const int cnt = f.cnt, actor = f.actor;
      const bool root_family = top && i == 0;
      const int has_children = f.kinds & 0x5555, whole = (f.kinds >> 16) & 0x5555;
      const int sdbits = A.tables ? (f.kinds >> 1) & 0x5555 & ~whole : 0;
      const int opp_rows = (root_family ? 0x5555 : 0) | whole;
      const bool bottom = (has_children | whole) == 0;
      const int64_t row_act = range_row(f, actor), row_opp = range_row(f, 1 - actor);

      // ---- every row of the regret and the mixing part is requested here
      const float2 bo = sld(B.leaf_prev, row_opp, ln), ex = sld(A.latest, p * 2 + actor, ln);
      float2 ach, cum, wsum;      // one child ahead
      auto request = [&](int k) {
        ach = sld(A.latest, (first + k) * 2 + actor, ln, const_mask(f, k));
        cum = sld(A.cum, first + k, ln);
        wsum = sld(A.wsum, first + k, ln);
      };
      request(0);
      const float2 rn_act = sld(A.reach, row_act, ln), ran_act = sld(A.reach_avg, row_act, ln);
      const float2 ra_old = sld(A.reach_avg_prev, row_act, ln);
      float2 rn_opp = make_float2(0.f, 0.f), ran_opp = make_float2(0.f, 0.f);
      if (root_family || (!CA && (sdbits | whole))) rn_opp = allowed2(sld(A.reach, row_opp, ln));
      if (root_family || (CA && (sdbits | whole))) ran_opp = allowed2(sld(A.reach_avg, row_opp, ln));

      // ---- regrets, discounting, regret matching
      sput(L.u.vecs[0], bo, ln);
      p2_sync_lds();
      card_sums_block<SR_BLOCK>(L.u.vecs[0], IT_VSTRIDE, 1, L.cs, fresh((int)threadIdx.x));
      float2 wgt = sunblocked(bo, L.cs, card_total(L.cs), fresh(ln.ab));
      if (linear && actor == (int)(t_now & 1)) wgt = make_float2(0.f, 0.f);   // this player's regrets are skipped at this t
      float2 sum = make_float2(0.f, 0.f);
#pragma unroll 1
      for (int k = 0; k < cnt; ++k) {
        float cc[2] = {cum.x, cum.y}, ww[2] = {wsum.x, wsum.y};
        const float rg[2] = {wgt.x * (ach.x - ex.x), wgt.y * (ach.y - ex.y)};
        if (k + 1 < cnt) request(k + 1);
#pragma unroll
        for (int e = 0; e < 2; ++e) {
          if (apply_dcfr) {
            const bool positive = cc[e] > 0.f;
            const float num = positive ? f_an : f_bn, den = positive ? f_ad : f_bd;
            const float inv = positive ? y_ad : y_bd;
            cc[e] = cc[e] * num;
            cc[e] = p2_quotient(cc[e], den, inv);
            ww[e] = ww[e] * num;
            ww[e] = p2_quotient(ww[e], den, inv);
          }
          ww[e] = ww[e] + 1.0f;
          cc[e] = cc[e] + rg[e];
          if (cfr_plus) cc[e] = fmaxf(cc[e], 0.f);
        }
        sst(A.cum, first + k, make_float2(cc[0], cc[1]), ln);
        sst(A.wsum, first + k, make_float2(ww[0], ww[1]), ln);
        const float2 pos = make_float2(fmaxf(cc[0], 0.f), fmaxf(cc[1], 0.f));
        sput(L.pol[k], pos, ln);
        sum.x += pos.x;
        sum.y += pos.y;
      }
      float2 pav[MAXC];
      if (!avg_copy) {
#pragma unroll
        for (int k = 0; k < MAXC; ++k)
          if (k < cnt) pav[k] = sld(A.policy_avg, first + k, ln);
      }
      // ---- the new policy, and the average policy mixed with it
      const float uniform = 1.0f / (float)cnt;
      float2 psum = make_float2(0.f, 0.f);
#pragma unroll
      for (int k = 0; k < MAXC; ++k) {
        if (k < cnt) {
          if (take_sample) sst(A.policy_sample, first + k, sld(A.policy, first + k, ln), ln);
          const float2 pos = sget(L.pol[k], ln);
          float2 pol;
          pol.x = p2_matched(pos.x, sum.x, uniform);
          pol.y = p2_matched(pos.y, sum.y, uniform);
          sst(A.policy, first + k, pol, ln);
          sput(L.pol[k], pol, ln);
          if (avg_copy) {
            pav[k] = pol;
          } else {
            const float rr[2] = {rn_act.x, rn_act.y}, rao[2] = {ra_old.x, ra_old.y};
            const float cc[2] = {pol.x, pol.y}, aa[2] = {pav[k].x, pav[k].y};
            float o[2];
#pragma unroll
            for (int e = 0; e < 2; ++e) {
              const float reach_a = rao[e] * mix_old, reach_n = rr[e] * mix_new;
              const float num = reach_a * aa[e] + reach_n * cc[e];
              const float den = reach_a + reach_n;
              const float unweighted = p2_quotient(mix_old * aa[e] + mix_new * cc[e], mix_total, y_mix);
              o[e] = den > 1e-5f ? p2_div(num, den) : unweighted;
            }
            pav[k] = make_float2(o[0], o[1]);
            psum.x += o[0];
            psum.y += o[1];
          }
        }
      }
      // ---- sums of the ranges: 0 the opponent's leaf range, 1 the actor's range at the parent, 2 + k the
      // children's leaf ranges; CA: 7 + k the children's ranges, 12 the opponent's
      constexpr int NS = CA ? SR_SUMS : 7;
      float sums[NS];
#pragma unroll
      for (int q = 0; q < NS; ++q) sums[q] = 0.f;
      const float2 la_act = actor == 0 ? la0 : la1, la_opp = actor == 0 ? la1 : la0;
      // the root's ranges behind `beliefs`
      const float2 rb_act = CA ? sld(A.beliefs, r * 2 + actor, ln) : la_act;
      const float2 rb_opp = CA && root_family ? sld(A.beliefs, r * 2 + 1 - actor, ln) : make_float2(0.f, 0.f);
      const float2 x_par = allowed2(rn_act);
      float2 lo = mul2(la_opp, CA ? ran_opp : rn_opp);   // the opponent's leaf range, the same at every child
      sums[0] = lo.x + lo.y;
      {
        const float2 va = mul2(rb_act, x_par);
        sums[1] = va.x + va.y;
        if (CA) {
          const float2 vb = mul2(rb_opp, rn_opp);
          sums[NS - 1] = vb.x + vb.y;
        }
      }
#pragma unroll
      for (int k = 0; k < MAXC; ++k) {
        if (k < cnt) {
          if (!avg_copy) {
            if (psum.x > 1e-5f) pav[k].x = p2_div(pav[k].x, fmaxf(psum.x, 1e-5f));
            if (psum.y > 1e-5f) pav[k].y = p2_div(pav[k].y, fmaxf(psum.y, 1e-5f));
          }
          sst(A.policy_avg, first + k, pav[k], ln);
          pav[k] = allowed2(mul2(ran_act, pav[k]));    // the child's average reach from here on
          const float2 x = mul2(rb_act, allowed2(mul2(rn_act, sget(L.pol[k], ln)))), y = mul2(la_act, pav[k]);
          sums[2 + k] = CA ? y.x + y.y : x.x + x.y;
          if (CA) sums[(CA ? 7 : 2) + k] = x.x + x.y;
        }
      }
      search_sums<NS>(sums, L);
      // ---- rows other families read: reach, average reach, ranges of children that have children
      auto normalised = [&](float2 v, float s) {
        return s > 1e-5f ? make_float2(p2_div(v.x, s), p2_div(v.y, s)) : sld(A.allowed_prob, r, ln);
      };
      if (sdbits | opp_rows) lo = normalised(lo, sums[0]);
      float2 own = make_float2(0.f, 0.f);  // the showdown child's range of the actor
#pragma unroll
      for (int k = 0; k < MAXC; ++k) {
        if (k < cnt) {
          const int64_t c = first + k;
          const bool inner = (has_children >> (2 * k)) & 1, sd = (sdbits >> (2 * k)) & 1;
          const float2 x = allowed2(mul2(rn_act, sget(L.pol[k], ln)));
          if (inner) {
            sst(A.reach, c * 2 + actor, x, ln);
            sst(A.reach_avg, c * 2 + actor, pav[k], ln);
            if (root_family) {
              sst(A.reach, c * 2 + 1 - actor, rn_opp, ln);
              sst(A.reach_avg, c * 2 + 1 - actor, ran_opp, ln);
            }
            if (CA) {
              sst(A.beliefs, c * 2 + actor, normalised(mul2(rb_act, x), sums[(CA ? 7 : 2) + k]), ln);
              if (root_family) sst(A.beliefs, c * 2 + 1 - actor, normalised(mul2(rb_opp, rn_opp), sums[NS - 1]), ln);
            }
          }
          if (inner || sd || ((whole >> (2 * k)) & 1)) {
            const float2 o = normalised(mul2(la_act, CA ? pav[k] : x), sums[2 + k]);
            if (sd) {
              own = o;
            } else {
              sst(B.leaf_next, c * 2 + actor, o, ln);
              if ((opp_rows >> (2 * k)) & 1) sst(B.leaf_next, c * 2 + 1 - actor, lo, ln);
            }
          }
        }
      }
      // ---- the showdown child: both ranges through LDS into strength order, values from there
      if (sdbits) {
        const SearchFam& stakes = L.fam[i - base];
        const float pot0 = readlane_f(stakes.pot0, 0), pot1 = readlane_f(stakes.pot1, 0), scl = readlane_f(stakes.scale, 0);
        const int64_t c = first + (__builtin_ctz((unsigned)sdbits) >> 1);
        sput(L.u.vecs[actor], own, ln);
        sput(L.u.vecs[1 - actor], lo, ln);
        p2_sync_lds();
        search_showdown(table, L, pot0, pot1, scl);
        const float2* ev = &L.u.sd.v[ln.off >> 2];
        const float2 x = ev[0], y = ev[1];
        const float2 v0 = make_float2(x.x, y.x), v1 = make_float2(x.y, y.y);
        sst(A.latest, c * 2, v0, ln);
        sst(A.latest, c * 2 + 1, v1, ln);
        sput(L.u.vecs[MAXC + 1], v0, ln);   // over the per-card prefixes, dead since the last barrier
        sput(L.u.vecs[MAXC + 2], v1, ln);
        p2_sync_lds();   // the buffers just read are staged over
      }
      if (bottom) backup(f, root_family, root_family ? rb_act : normalised(mul2(rb_act, x_par), sums[1]), sdbits);
    }
  }

  if (A.phases & PHASE_3) {
    for (int i = nfam - 1; i >= 0; --i) {
      if (i < base || i >= base + 64) search_window(L, A, pp0, nfam, base = i > 63 ? i - 63 : 0);
      const Fam f = search_fam(L, i - base);
      if (((f.kinds | (f.kinds >> 16)) & 0x5555) == 0) continue;   // backed up in the first walk
      const float2 ab = sld(CA ? A.beliefs : B.leaf_next, range_row(f, f.actor), ln);
      float2 pk[MAXC];
#pragma unroll
      for (int k = 0; k < MAXC; ++k)
        if (k < f.cnt) pk[k] = sld(A.policy, f.first + k, ln);
#pragma unroll
      for (int k = 0; k < MAXC; ++k)
        if (k < f.cnt) sput(L.pol[k], pk[k], ln);
      backup(f, top && i == 0, ab, 0);
    }
  }
}

}  // namespace p2
extern "C" {

int p2hip_cfr_iteration_shared(const P2HipIterArgs* host_args, const int32_t* range_rows, const float* leaf_prev,
                               float* leaf_next, int64_t n_items, int max_children, int phases, void* stream) {
  constexpr int FUSED = 64, FUSED_CFR_AVG = 128;
  if (phases & ~511) return P2_EINVAL;
  p2::IterArgs a = {};
  const int bad = p2_iteration_args(host_args, n_items, max_children, phases, a);
  if (bad) return bad;
  if (!p2_aligned4(range_rows) || !p2_aligned8(leaf_prev) || !p2_aligned8(leaf_next)) return P2_EINVAL;
  a.range_rows = range_rows;
  if (!(phases & FUSED)) {
    if ((phases & FUSED_CFR_AVG) || leaf_next) return P2_EINVAL;
    a.leaf_prev = leaf_prev;
    if (n_items == 0) return 0;
    return p2_launch_iteration(a, n_items, max_children, phases & 63, stream);
  }
  // one walk per family: a lean iteration between two reach_avg and two range buffers
  if (max_children > p2::SR_MAXC || (phases & 15 & ~3) || !(phases & p2::PHASE_LEAN) || !(phases & p2::PHASE_CONST) ||
      (phases & p2::PHASE_WHOLE) || !range_rows || !leaf_prev || !leaf_next || leaf_prev == leaf_next ||
      (n_items > 0 && !a.reach_avg_prev))
    return P2_EINVAL;
  if (n_items == 0) return 0;
  const p2::SearchRows rows = {leaf_prev, leaf_next};
  const dim3 grid((unsigned)n_items), block(p2::SR_BLOCK);
  if (phases & FUSED_CFR_AVG)
    hipLaunchKernelGGL((p2::cfr_search_kernel<true>), grid, block, 0, (hipStream_t)stream, a, rows);
  else
    hipLaunchKernelGGL((p2::cfr_search_kernel<false>), grid, block, 0, (hipStream_t)stream, a, rows);
  P2_LAUNCH_CHECK();
  return 0;
}

}  // extern "C"
