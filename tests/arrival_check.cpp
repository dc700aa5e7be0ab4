// CPU check of the arrival counts of small launches (minim_amd/csrc/arrival.hpp),
// run by tests/test_tile_map.py: alone, exactly the last block of a launch finishes
// its sums, from any state that earlier launches left; and two launches whose
// blocks arrive mixed on one counter leave it good for the next.
#include <algorithm>
#include <cstdio>
#include <random>
#include <vector>

#include "arrival.hpp"

using namespace minim_amd;

static bool arrive(unsigned& counter, int nb, int b) {
  const unsigned w = arrival_weight(nb, b), before = counter;
  counter += w;
  return arrival_last(before, w);
}

int main() {
  std::mt19937 rng(1);
  int bad = 0;
  unsigned counter = 0u - 40 * kArrivals;  // passes the end of the 32 bits on the way
  auto alone = [&](int nb) {
    std::vector<int> order(nb);
    for (int b = 0; b < nb; b++) order[b] = b;
    std::shuffle(order.begin(), order.end(), rng);
    for (int k = 0; k < nb; k++) bad += arrive(counter, nb, order[k]) != (k == nb - 1);
  };
  for (int nb = 1; nb <= (int)kArrivals; nb++) alone(nb);
  for (int trial = 0; trial < 2000; trial++) {
    const int n1 = 1 + rng() % kArrivals, n2 = 1 + rng() % kArrivals;
    std::vector<std::pair<int, int>> order;
    for (int b = 0; b < n1; b++) order.push_back({n1, b});
    for (int b = 0; b < n2; b++) order.push_back({n2, b});
    std::shuffle(order.begin(), order.end(), rng);
    for (auto& o : order) arrive(counter, o.first, o.second);
    alone(1 + rng() % kArrivals);
  }
  std::printf("%d failures\n", bad);
  return bad ? 1 : 0;
}
