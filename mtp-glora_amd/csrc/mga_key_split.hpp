// Splitting the last work items of an attention launch over their keys.
//
// The forward and dQ launches hand each XCD a contiguous share of the items,
// one workgroup per slot (a CU, or half of one); an item walks its whole tile
// list. When the items of a share are not a multiple of the slots, the last
// round leaves slots idle for as long as a full walk: 8 items on 32 slots (a
// 512-row chunk) use a quarter of the GPU. The r items of that round are
// therefore split into parts of their tile lists, where that ends earlier
// (split_ends_first); a part is a workgroup of its own and writes fp32 partial
// results, which a small kernel combines in the order of the parts.
#pragma once

#include <algorithm>
#include <cmath>
#include <functional>

#include "mga_common.hpp"

namespace mga {

// Items 0 .. k - 1 of each XCD's share run whole, the other r in ns parts:
// part 0 takes first / 1024 of an item's tile list, the later ones equal
// shares of the rest. Workgroup t of an XCD: the whole items, then every
// item's part 0, then the other parts.
struct KeySplit {
  int k;
  int r;
  int ns;
  int first;
  float *ws;   // parts, [item * ns + part][XCD][wave][part_floats]

  // number of workgroups per XCD
  __host__ __device__ int groups() const { return k + r * ns; }
  // workgroup t: its item (within the share) and part, -1 = the whole list
  __device__ __forceinline__ void locate(int t, int &item, int &part) const {
    item = t;
    part = -1;
    if (t < k) return;
    const int u = t - k;
    if (u < r) {
      part = 0;
    } else {
      const int v = u - r;
      item = k + v / (ns - 1);
      part = 1 + v % (ns - 1);
    }
  }
  // first entry of a part's share of n tile-list entries (part ns: n)
  __host__ __device__ __forceinline__ int begin(int part, int n) const {
    if (part == 0) return 0;
    const int f = (n * first + 512) >> 10;
    return f + (n - f) * (part - 1) / (ns - 1);
  }
  // a part's index among the parts in ws
  __device__ __forceinline__ int64_t slot(int item, int part, int xcd) const {
    return ((int64_t)(item - k) * ns + part) * 8 + xcd;
  }
};

// fp32 words of one wave's part of the forward: O^T, offset and row sum per lane.
template <int HD>
constexpr int kPartFloats = HD * 32 + 128;
inline int part_floats(int head_dim) { return head_dim * 32 + 128; }

inline KeySplit no_split(int nmax) { return KeySplit{nmax, 0, 1, 1024, nullptr}; }

// Key tiles of the longest item of the last round: an XCD whose share lies in
// whole kv heads (longest items first) ends with the items of a head's first
// rows.
inline int last_round_tiles(int S, int P, int Hkv, int nslice, int rows, int r) {
  const int last = Hkv % 8 == 0 ? rows * ((r + nslice - 1) / nslice) : S;
  return (P + std::min(S, last) + kBlock - 1) / kBlock;
}

// nmax: items of the largest share; slots: workgroups an XCD runs at once;
// ntile: key tiles of the longest item of the last round; part_cost, merge_cost: what a part
// costs beyond its tiles and what the combining launch costs, in tiles. Of
// two shapes per ns the plan takes the one with the least time to the end:
// * equal parts, run in rounds of the slots;
// * r < slots: a long first part for r of the slots, short ones in rounds on
//   the other slots - r, so long that both end together (24 items on 32
//   slots: 3/4 of each item in one piece, the rest three to a free slot).
// A part keeps at least min_part tiles; kMaxPartRounds bounds the
// workspace (133 KB a part at head_dim 128).
constexpr int kMaxParts = 16, kMaxPartRounds = 4;
inline KeySplit key_split_plan(int nmax, int slots, int ntile, float part_cost, float merge_cost, int min_part) {
  KeySplit best = no_split(nmax);
  slots = std::max(slots, 1);
  const int r = nmax % slots;
  if (r == 0) return best;
  const float T = (float)ntile;
  float best_cost = T;   // the last round unsplit
  for (int ns = 2; ns <= kMaxParts && r * ns <= kMaxPartRounds * slots; ++ns) {
    if (ntile >= min_part * ns) {
      const int rounds = (r * ns + slots - 1) / slots;
      const float cost = rounds * ((float)((ntile + ns - 1) / ns) + part_cost) + merge_cost;
      if (cost < best_cost) {
        best_cost = cost;
        best = KeySplit{nmax - r, r, ns, 1024 / ns, nullptr};
      }
    }
    const int rounds = (r * (ns - 1) + slots - r - 1) / (slots - r);   // of the short parts
    const float per = (float)rounds / (ns - 1);
    const float big = (per * T + (rounds - 1) * part_cost) / (1.f + per);   // big + part_cost = short parts' end
    if (big < T && (T - big) / (ns - 1) >= min_part) {
      const float cost = std::ceil(big) + part_cost + merge_cost;
      if (cost < best_cost) {
        best_cost = cost;
        best = KeySplit{nmax - r, r, ns, (int)(1024.f * big / T), nullptr};
      }
    }
  }
  return best;
}

// Time until the last workgroup of an XCD ends: they start in order, each on
// the slot that is free first.
class SlotClock {
 public:
  explicit SlotClock(int slots) : n_(std::min(std::max(slots, 1), kMost)) { std::fill(t_, t_ + n_, 0.f); }
  void run(float cost) {
    std::pop_heap(t_, t_ + n_, std::greater<float>());
    t_[n_ - 1] += cost;
    end_ = std::max(end_, t_[n_ - 1]);
    std::push_heap(t_, t_ + n_, std::greater<float>());
  }
  float end() const { return end_; }

 private:
  static constexpr int kMost = 256;
  int n_;
  float t_[kMost];   // a heap, the slot free first on top
  float end_ = 0.f;
};

// The items of the first XCD's share, which holds the longest lists: rows row
// blocks of a kv head's nslice head slices, last rows first.
struct QShare {
  int S, P, nslice, rows, nmax, slots, head_dim;
  int tiles(int o) const {   // key tiles of item o
    const int nqb = (S + rows - 1) / rows, qb = nqb - 1 - o % (nslice * nqb) / nslice;
    return (P + std::min((qb + 1) * rows, S) + kBlock - 1) / kBlock;
  }
};

// Whether the split launch ends before the one that would run without it: the
// items from k1 on as two-group workgroups, half a list each, in a launch of
// their own. key_split_plan takes the last round's items as equally long and
// the slots as free at the same time; where the chunk's own keys are a large
// share of the lists, the slots that end early level the whole items by
// themselves. So both launches are run through SlotClock (up to 2.5 us of host
// time), in key tiles: a whole item costs its list + 1; a part 1.05 of its
// share + 2 (the parts of an item stream K and V apart from each other); two
// groups half the longest list + 4 (head_dim 64: 2.5), + 12 behind another
// launch, whose end they wait for; 4-wave workgroups, two slots a CU, run in 0.9
// of the time where no CU gets two. Of 412 16-bit launches timed with and without
// their plan (11 geometries, 124 to 5 900 rows, 0 to 20 000 prefix keys) 32 were
// slower split, by up to 15%: 872 rows x 32 heads on 1 500 keys, forward 57.0 ->
// 60.6 us, dQ 63.3 -> 68.7; 3 248 rows on 1 500, 191 -> 207 and 250 -> 265 us;
// 3 624 on 2 500, 265 -> 284 and 350 -> 369 us. With this rule one is left (3 361
// rows on 11 280, head_dim 64, dQ 571 -> 589 us), and ten that gained 3 to 17%
// run whole.
inline bool split_ends_first(const KeySplit &sp, const QShare &f, int k1, float merge_cost) {
  constexpr float kItem = 1.f, kPart = 2.f, kPartPace = 1.05f, kTwoGroupsBehind = 12.f;
  constexpr float kLonePace = 0.9f, kGain = 1.02f;
  const float two_groups = f.head_dim == 64 ? 2.5f : 4.f;
  constexpr int kRounds = 7;   // the rounds before the last that are looked at
  const int o0 = std::max(0, sp.k - kRounds * f.slots);
  const bool two_a_cu = f.slots > device_cu_count() / 8;
  auto pace = [&](int workgroups) { return two_a_cu && workgroups <= f.slots / 2 ? kLonePace : 1.f; };
  SlotClock whole(f.slots), split(f.slots);
  for (int o = o0; o < k1; ++o) whole.run(kItem + f.tiles(o));
  float unsplit = whole.end() * pace(k1 - o0);
  if (k1 < f.nmax) unsplit += (k1 > 0 ? kTwoGroupsBehind : two_groups) + 0.5f * f.tiles(k1);
  for (int o = o0; o < sp.k; ++o) split.run(kItem + f.tiles(o));
  for (int o = sp.k; o < f.nmax; ++o) split.run(kPart + kPartPace * sp.begin(1, f.tiles(o)));
  for (int o = sp.k; o < f.nmax; ++o)
    for (int p = 1; p < sp.ns; ++p)
      split.run(kPart + kPartPace * (sp.begin(p + 1, f.tiles(o)) - sp.begin(p, f.tiles(o))));
  return kGain * (split.end() * pace(sp.groups() - o0) + merge_cost) < unsplit;
}

}  // namespace mga
