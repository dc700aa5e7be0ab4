// subclass_check.cpp -- classes derived from the library's potentials keep their
// own evaluations on the paths of the minimisers (no GPU: nothing is launched).
#include <cstdio>
#include <stdexcept>

#include "minim/BarAndHinge.h"
#include "minim/LjNd.h"

static int fails = 0;
#define EXPECT(c)                                        \
  do {                                                   \
    if (!(c)) {                                          \
      std::printf("FAILED line %d: %s\n", __LINE__, #c); \
      fails++;                                           \
    }                                                    \
  } while (0)

struct Walled : minim::Lj3d {
  mutable int calls = 0;
  void evaluate(int, const void*, const void*, double, double*, void*, void*) const override { calls++; }
};

struct Counting : minim::BarAndHinge {
  mutable int calls = 0;
  void evaluateAsync(int, const void*, const void*, double, bool, double*, void*, void*) const override { calls++; }
};

int main() {
  double x[3] = {}, g[3];
  minim::Lj3d lj;
  lj.setCutoff(2.5, {10, 10, 10}, 0.3);
  EXPECT(lj.fusesFire(3) && lj.fusesFire(0) && !lj.fusesFire(2));
  Walled w;
  w.setCutoff(2.5, {10, 10, 10}, 0.3);
  EXPECT(!w.fusesFire(3));
  w.evaluateAsync(minim::FP64, x, nullptr, 0.0, false, nullptr, g, nullptr);
  EXPECT(w.calls == 1);
  // an override of the asynchronous form that calls evaluate must not come back to itself
  Counting c;
  bool threw = false;
  try {
    c.evaluate(minim::FP64, x, nullptr, 0.0, nullptr, g, nullptr);
  } catch (const std::runtime_error&) {
    threw = true;  // not initialised
  }
  EXPECT(threw && c.calls == 0);
  std::printf("%s\n", fails ? "subclass check: FAILED" : "subclass check: ok");
  return fails ? 1 : 0;
}
