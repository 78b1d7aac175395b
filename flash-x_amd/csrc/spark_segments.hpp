// spark_segments.hpp -- z segments of the FP32-flux stage's column items (host
// code).
#pragma once
#include <algorithm>
#include <functional>
#include <map>
#include <queue>
#include <utility>
#include <vector>

namespace spark {

// one column of a stage region: the levels it updates and its cells per level
struct Column { int levels, cells; };

// the segments a column of n levels is cut into for segments of at most len
struct Cut { int parts, seg; };
inline Cut cut_column(int n, int len) {
  const int parts = (n + len - 1) / len;
  return Cut{parts, (n + parts - 1) / parts};
}

// Length of the z segments the columns of a stage are cut into, given in the
// order the workgroups take them.  A workgroup marches an item level by level,
// two levels more than it updates (the reconstruction below and the flux
// above), so few or unequal columns leave workgroups idle, and cutting them
// costs those two levels per segment.  The length with the shortest list
// schedule over the launch's `slots` workgroups wins, the whole column unless
// cutting gains 3 %.  A length is scheduled only where the total work or the
// longest item does not rule it out, the whole columns not at all where the
// bound on any list schedule leaves no other length a chance: on 4096 mixed
// blocks the eleven schedules of every plan, tuned candidates included, took
// 0.26 of the first step's 0.89 s, and the bounds decide all of them.
// *scheduled (optional) counts the schedules.
inline int z_segment(const std::vector<Column>& cols, int slots, int* scheduled = nullptr) {
  // a segment's time: its levels' barriers and its columns' tasks
  auto time = [](int seg, int cells) { return (seg + 2) * (1. + cells / 64.); };
  std::map<std::pair<int, int>, long> kinds;
  int longest = 1;
  for (const Column& c : cols) {
    kinds[{c.levels, c.cells}]++;
    longest = std::max(longest, c.levels);
  }
  // lower and upper bound of the schedule's end for a length
  auto bounds = [&](int len) {
    double total = 0., most = 0.;
    for (const auto& k : kinds) {
      const Cut c = cut_column(k.first.first, len);
      const double t = time(c.seg, k.first.second);
      total += t * c.parts * k.second;
      most = std::max(most, t);
    }
    // 1e-9: the schedule sums the same times in another order
    return std::make_pair(std::max(total / slots, most) * (1. - 1e-9), (total / slots + most) * (1. + 1e-9));
  };
  auto schedule = [&](int len) {
    if (scheduled) (*scheduled)++;
    std::priority_queue<double, std::vector<double>, std::greater<double>> busy;
    double end = 0.;
    for (const Column& col : cols) {
      const Cut c = cut_column(col.levels, len);
      const double t = time(c.seg, col.cells);
      for (int p = 0; p < c.parts; p++) {
        double at = 0.;
        if ((int)busy.size() == slots) {
          at = busy.top();
          busy.pop();
        }
        busy.push(at + t);
        end = std::max(end, at + t);
      }
    }
    return end;
  };
  const int lens[] = {24, 16, 12, 10, 8, 7, 6, 5, 4, 3};
  const double whole_most = bounds(longest).second;
  bool chance = false;
  for (int len : lens) chance = chance || (len < longest && bounds(len).first < 0.97 * whole_most);
  if (!chance) return longest;
  int pick = longest;
  double best = schedule(longest);
  for (int len : lens) {
    if (len >= longest) continue;
    const double bar = pick == longest ? 0.97 * best : best;
    if (bounds(len).first >= bar) continue;
    const double end = schedule(len);
    if (end < bar) {
      best = end;
      pick = len;
    }
  }
  return pick;
}

}  // namespace spark
