// batch_items.hpp - the work items of a batch launch: strips x row chunks of
// every instance, dealt to the XCDs.  Host code only.
#pragma once

#include <algorithm>
#include <array>
#include <cstdint>
#include <utility>
#include <vector>

namespace sps {

struct BatchItem {
  int inst, y0, ty, strip;
};
struct BatchSides {
  int X, Y, R;  // R: radius of the instance's step
};

// Strip geometry of the 2-values-per-lane stream (fused_tile.hpp): a wave
// covers (64 - 2*HL)*2 columns and HL halo lanes per side carry the K*R
// columns the K fused steps reach.
constexpr int kBatchVec = 2;
constexpr int batch_halo_lanes(int K, int R) {
  return (K * R + kBatchVec - 1) / kBatchVec;
}
constexpr int batch_strip_width(int K, int R) {
  return (64 - 2 * batch_halo_lanes(K, R)) * kBatchVec;
}

// cost of streaming a chunk of ty rows, K steps: the rows and the fill, a
// radius-two row 10 to a radius-one row's 9
constexpr int batch_item_cost(int K, int R, int ty) {
  return (ty + 2 * K * R) * (R == 2 ? 10 : 9);
}

constexpr int kBatchXcds = 8;
using BatchLists = std::array<std::vector<BatchItem>, kBatchXcds>;

// Every XCD's items at item height `rows`, the costliest first: whole instances,
// or contiguous pieces of one that is more than 1/64 of the batch, of like total
// cost.
inline BatchLists batch_lists(const std::vector<BatchSides>& inst, int K, int rows) {
  struct Unit {
    int64_t cost;
    std::vector<BatchItem> items;
  };
  auto cost = [&](const BatchItem& it) {
    return (int64_t)batch_item_cost(K, inst[it.inst].R, it.ty);
  };
  std::vector<Unit> units;
  int64_t total = 0;
  for (size_t i = 0; i < inst.size(); ++i) {
    const int W = batch_strip_width(K, inst[i].R), X = inst[i].X, Y = inst[i].Y;
    units.push_back(Unit{0, {}});
    for (int st = 0; st * W < X; ++st)
      for (int y0 = 0; y0 < Y; y0 += rows) {
        const BatchItem it{(int)i, y0, std::min(rows, Y - y0), st};
        units.back().items.push_back(it);
        units.back().cost += cost(it);
      }
    total += units.back().cost;
  }
  std::vector<Unit> pieces;
  for (Unit& u : units) {
    if (u.cost * 64 <= total) {
      pieces.push_back(std::move(u));
      continue;
    }
    pieces.push_back(Unit{0, {}});
    for (const BatchItem& it : u.items) {
      if (pieces.back().cost * 64 > total) pieces.push_back(Unit{0, {}});
      pieces.back().items.push_back(it);
      pieces.back().cost += cost(it);
    }
  }
  // the largest first, each to the XCD with the least so far
  std::stable_sort(pieces.begin(), pieces.end(),
                   [](const Unit& a, const Unit& b) { return a.cost > b.cost; });
  BatchLists xcd;
  std::array<int64_t, kBatchXcds> load{};
  for (const Unit& u : pieces) {
    const size_t least = std::min_element(load.begin(), load.end()) - load.begin();
    load[least] += u.cost;
    xcd[least].insert(xcd[least].end(), u.items.begin(), u.items.end());
  }
  for (auto& x : xcd)
    std::stable_sort(x.begin(), x.end(), [&](const BatchItem& a, const BatchItem& b) {
      return cost(a) > cost(b);
    });
  return xcd;
}

// How long a launch of the lists at item height `rows` takes, in the unit of
// batch_item_cost: an XCD's workgroups of four items go to its 32 CUs in turn,
// one item to each SIMD, and the fullest SIMD ends last; a lone item's rows cost
// 1.5 of a shared one's (their latency shows).  Counts the items of batch_lists
// by cost instead of listing them.
inline double batch_launch_cost(const std::vector<BatchSides>& inst, int K, int rows) {
  struct Run {
    int cost;
    int64_t count;
  };
  struct Piece {
    int64_t cost;
    Run run[2];
  };
  auto strips_of = [&](const BatchSides& s) {
    const int W = batch_strip_width(K, s.R);
    return (s.X + W - 1) / W;
  };
  int64_t total = 0;
  std::vector<Piece> whole, pieces;
  whole.reserve(inst.size());
  for (const BatchSides& s : inst) {
    const int64_t n = strips_of(s), rest = s.Y % rows;
    const Run full{batch_item_cost(K, s.R, rows), n * (s.Y / rows)},
        last{rest ? batch_item_cost(K, s.R, (int)rest) : 0, rest ? n : 0};
    whole.push_back(Piece{full.cost * full.count + last.cost * last.count, {full, last}});
    total += whole.back().cost;
  }
  pieces.reserve(whole.size());
  for (size_t i = 0; i < whole.size(); ++i) {
    const Piece& u = whole[i];
    if (u.cost * 64 <= total) {
      pieces.push_back(u);
      continue;
    }
    const Piece none{0, {{u.run[0].cost, 0}, {u.run[1].cost, 0}}};
    pieces.push_back(none);
    const int64_t n = strips_of(inst[i]);
    for (int64_t st = 0; st < n; ++st)
      for (int which = 0; which < 2; ++which)
        for (int64_t c = 0; c < u.run[which].count / n; ++c) {
          if (pieces.back().cost * 64 > total) pieces.push_back(none);
          pieces.back().cost += u.run[which].cost;
          ++pieces.back().run[which].count;
        }
  }
  std::stable_sort(pieces.begin(), pieces.end(),
                   [](const Piece& a, const Piece& b) { return a.cost > b.cost; });
  std::array<int64_t, kBatchXcds> load{};
  std::array<std::vector<Run>, kBatchXcds> runs;
  for (const Piece& u : pieces) {
    const size_t least = std::min_element(load.begin(), load.end()) - load.begin();
    load[least] += u.cost;
    for (const Run& r : u.run) {
      if (r.count == 0) continue;
      auto same = std::find_if(runs[least].begin(), runs[least].end(),
                               [&](const Run& q) { return q.cost == r.cost; });
      if (same == runs[least].end()) runs[least].push_back(r);
      else same->count += r.count;
    }
  }
  double longest = 0;
  for (auto& x : runs) {
    std::sort(x.begin(), x.end(), [](const Run& a, const Run& b) { return a.cost > b.cost; });
    std::array<int64_t, 128> simd{};
    size_t p = 0;
    for (const Run& r : x) {
      longest = std::max(longest, 1.5 * r.cost);
      if (r.count >= 128)
        for (int64_t& v : simd) v += r.cost * (r.count / 128);
      for (int64_t q = r.count % 128; q > 0; --q, ++p) simd[p % 128] += r.cost;
    }
    longest = std::max(longest, (double)*std::max_element(simd.begin(), simd.end()));
  }
  return longest;
}

// Item height before any tuning: of the heights that split a side of the batch
// evenly, the one whose launch is the shortest (the tallest of equals).  A launch
// lasts at least the mean load of a SIMD and 1.5 of its costliest item: the 32
// heights of the least such bounds are tried, as long as the bound is below the
// best launch found.
inline int batch_rows(const std::vector<BatchSides>& inst, int K) {
  std::vector<std::array<int, 3>> kinds;  // strips, Y, R; then how many of each
  std::vector<int64_t> count;
  std::vector<std::array<int, 3>> all;
  for (const BatchSides& i : inst) {
    const int W = batch_strip_width(K, i.R);
    all.push_back({(i.X + W - 1) / W, i.Y, i.R});
  }
  std::sort(all.begin(), all.end());
  for (const auto& k : all) {
    if (kinds.empty() || kinds.back() != k) {
      kinds.push_back(k);
      count.push_back(0);
    }
    ++count.back();
  }
  std::vector<bool> is(513, false);
  for (const auto& k : kinds)
    for (int m = 1; m <= k[1]; ++m) {
      const int rows = (k[1] + m - 1) / m;
      if (rows < 4) break;
      is[std::min(rows, 512)] = true;
    }
  std::vector<std::pair<double, int>> bound;
  for (int rows = 512; rows >= 4; --rows) {
    if (!is[rows]) continue;
    int64_t sum = 0;
    int most = 0;
    for (size_t k = 0; k < kinds.size(); ++k) {
      const int Y = kinds[k][1], R = kinds[k][2];
      if (Y / rows) most = std::max(most, batch_item_cost(K, R, rows));
      if (Y % rows) most = std::max(most, batch_item_cost(K, R, Y % rows));
      sum += count[k] * kinds[k][0] *
             ((int64_t)(Y / rows) * batch_item_cost(K, R, rows) +
              (Y % rows ? batch_item_cost(K, R, Y % rows) : 0));
    }
    bound.push_back({std::max((double)sum / 1024, 1.5 * most), rows});
  }
  std::stable_sort(bound.begin(), bound.end(),
                   [](const auto& a, const auto& b) { return a.first < b.first; });
  int best = 4;  // every side below four rows
  double least = 0;
  if (bound.size() > 32) bound.resize(32);
  for (const auto& b : bound) {
    if (least > 0 && b.first > least) break;
    const double c = batch_launch_cost(inst, K, b.second);
    if (least == 0 || c < least || (c == least && b.second > best)) {
      least = c;
      best = b.second;
    }
  }
  return best;
}

}  // namespace sps
