// hinge_angle_check.cpp -- BarAndHinge::setHingeTheta0 on the GPU: after each
// change, energy and gradient are those of a potential made with the same rest
// angles from the start, bit for bit, and a copy made before keeps its own.
#include <cmath>
#include <cstdio>
#include <vector>

#include "minim/BarAndHinge.h"

static int fails = 0;
#define EXPECT(c)                                        \
  do {                                                   \
    if (!(c)) {                                          \
      std::printf("FAILED line %d: %s\n", __LINE__, #c); \
      fails++;                                           \
    }                                                    \
  } while (0)

static const int side = 40;
static std::vector<std::vector<int>> tri;
static std::vector<double> x;

static minim::BarAndHinge make(const std::vector<int>& fixed) {
  minim::BarAndHinge p;
  p.setTriangulation(tri).setRigidity(1.0, 0.3).setLength0(1.0);
  p.setConstraints(fixed);
  return p;
}

// p's energy and gradient are those of a potential made with theta
static void same(const minim::BarAndHinge& p, const std::vector<double>& theta, const std::vector<int>& fixed,
                 const std::vector<double>& force, const char* what) {
  std::printf("%s\n", what);
  std::fflush(stdout);
  minim::BarAndHinge q = make(fixed);
  q.setTheta0(theta);
  if (!force.empty()) q.setForce(force);
  q.init(x);
  EXPECT(p.energy(x) == q.energy(x));
  EXPECT(p.gradient(x) == q.gradient(x));
}

int main() {
  std::vector<int> fixed;
  for (int i = 0; i < side; i++)
    for (int j = 0; j < side; j++) {
      x.insert(x.end(), {0.95 * (i - 0.5 * j), 0.87 * j, 0.1 * std::sin(1.3 * i + j)});
      for (int k = 0; k < 3 && i < 2; k++) fixed.push_back(3 * (i * side + j) + k);
      if (i + 1 < side && j + 1 < side) {
        const int a = i * side + j, b = a + side;
        tri.push_back({a, b, b + 1});
        tri.push_back({a, b + 1, a + 1});
      }
    }
  for (int uniform = 0; uniform < 2; uniform++) {
    minim::BarAndHinge p = make(fixed);
    if (uniform) p.setTheta0(3.0);
    p.init(x);
    std::vector<double> theta = p.theta0List();
    const int n = (int)theta.size();
    const minim::BarAndHinge before = p;
    const std::vector<double> theta0 = theta;
    for (int h : {0, n / 2, n / 2 + 1, n - 1, n / 2}) {  // 0: all of its nodes are fixed
      theta[h] += 0.25;
      p.setHingeTheta0(h, theta[h]);
      same(p, theta, fixed, {}, "changed");
    }
    same(before, theta0, fixed, {}, "the copy");
    p.setForce({0, 0, 0.01});
    theta[7 * side] = 2.5;
    p.setHingeTheta0(7 * side, 2.5);
    same(p, theta, fixed, {0, 0, 0.01}, "with a force set since");
    fixed.push_back((int)x.size() - 2);
    p.setConstraints(std::vector<int>{fixed.back()});
    theta[n - 2] = 3.5;
    p.setHingeTheta0(n - 2, 3.5);
    same(p, theta, fixed, {0, 0, 0.01}, "with a constraint set since");
    fixed.pop_back();
  }
  std::printf("%s\n", fails ? "hinge angle check: FAILED" : "hinge angle check: ok");
  return fails ? 1 : 0;
}
