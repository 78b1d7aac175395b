// Checks spark::z_segment against a list schedule of every length (the rule it
// stands for) on random column sets, on the shapes at the edges of its bounds,
// and that large sets are decided without a schedule.  Prints "ok <cases>" or
// the first mismatch.
#include <cstdio>
#include <random>

#include "spark_segments.hpp"

static int every_schedule(const std::vector<spark::Column>& cols, int slots) {
  int longest = 1;
  for (const auto& c : cols) longest = std::max(longest, c.levels);
  int pick = longest;
  double best = 0.;
  for (int len : {longest, 24, 16, 12, 10, 8, 7, 6, 5, 4, 3}) {
    if (len > longest) continue;
    std::priority_queue<double, std::vector<double>, std::greater<double>> busy;
    double end = 0.;
    for (const auto& c : cols) {
      const int parts = (c.levels + len - 1) / len, seg = (c.levels + parts - 1) / parts;
      const double t = (seg + 2) * (1. + c.cells / 64.);
      for (int p = 0; p < parts; p++) {
        double at = 0.;
        if ((int)busy.size() == slots) {
          at = busy.top();
          busy.pop();
        }
        busy.push(at + t);
        end = std::max(end, at + t);
      }
    }
    if (len == longest || end < (pick == longest ? 0.97 : 1.) * best) {
      best = end;
      pick = len;
    }
  }
  return pick;
}

int main() {
  std::mt19937 r(20261205);
  long cases = 0, cut = 0;
  auto check = [&](const std::vector<spark::Column>& cols, int slots) {
    const int want = every_schedule(cols, slots), got = spark::z_segment(cols, slots);
    if (want != got)
      std::printf("%zu columns over %d slots: %d, want %d\n", cols.size(), slots, got, want);
    cases++;
    int longest = 1;
    for (const auto& c : cols) longest = std::max(longest, c.levels);
    cut += want != longest;
    return want == got;
  };
  for (int t = 0; t < 3000; t++) {
    const int slots = 8 << (r() % 7), n = 1 + r() % (t % 3 ? 200 : 4 * slots);
    std::vector<spark::Column> cols;
    const int kinds = 1 + r() % 4;
    std::vector<spark::Column> kind;
    for (int k = 0; k < kinds; k++) kind.push_back({1 + (int)(r() % 44), 4 + (int)(r() % 253)});
    for (int i = 0; i < n; i++) cols.push_back(kind[r() % kinds]);
    if (!check(cols, slots)) return 1;
  }
  for (int levels : {1, 2, 3, 4, 23, 24, 25, 28, 44})
    for (int n : {1, 511, 512, 513, 1024, 1025})
      if (!check(std::vector<spark::Column>(n, {levels, 196}), 512)) return 1;
  if (cut < cases / 10 || cut > cases - cases / 10) {
    std::printf("%ld of %ld cases cut: the sets do not cover both sides\n", cut, cases);
    return 1;
  }
  // many columns: decided by the bounds
  std::vector<spark::Column> many;
  for (int i = 0; i < 40000; i++) many.push_back({i % 8 ? 28 : 44, i % 3 ? 196 : 242});
  int scheduled = 0;
  if (spark::z_segment(many, 512, &scheduled) != 44 || scheduled != 0) {
    std::printf("%d schedules for %zu columns\n", scheduled, many.size());
    return 1;
  }
  std::printf("ok %ld\n", cases);
  return 0;
}
