// Checks the cluster tables of bah_mesh.hpp on the host: sheets, stars whose
// hub has more elements than a chunk holds, random and degenerate lists.
#include <cstdio>
#include <cstdlib>
#include <random>

#include "bah_mesh.hpp"

using namespace minim_amd;

#define REQUIRE(c)                                              \
  do {                                                          \
    if (!(c)) {                                                 \
      std::printf("%s:%d: %s (%s)\n", __FILE__, __LINE__, #c, name); \
      std::exit(1);                                             \
    }                                                           \
  } while (0)

static void check(const char* name, int n, const std::vector<int>& bar, const std::vector<int>& hin,
                  const std::vector<double>& x) {
  BaHLists l;
  l.nnode = n;
  l.bar = &bar;
  l.hinge = &hin;
  const int m = bah_mesh::parts(n);
  const auto ord = bah_mesh::order(x, m);
  const BaHMesh M = bah_mesh::build(l, ord, m);
  std::vector<int> owned(n, 0), counted[2], chunkCluster(M.chunk.size(), -1);
  counted[0].assign(bar.size() / 2, 0);
  counted[1].assign(hin.size() / 4, 0);
  // per node: the (element, corner) sequence its codes name
  std::vector<std::vector<int>> seq[2];
  seq[0].resize(n);
  seq[1].resize(n);
  size_t visits = 0;
  for (size_t k = 0; k < M.cluster.size(); k++) {
    int first = 1;
    for (int ci = M.cluster[k];; ci++) {
      REQUIRE(ci < (int)M.chunk.size());
      const BaHChunk& c = M.chunk[ci];
      visits++;
      REQUIRE(c.nOwn >= 1 && c.nOwn <= kBaHNodes && c.nNode >= c.nOwn && c.nNode <= kBaHTable);
      REQUIRE(c.nHinge <= kBaHHinges && c.nHingeOwn >= 0 && c.nHingeOwn <= c.nHinge);
      REQUIRE(c.node0 + c.nNode <= M.node.size() && c.own0 + c.nOwn <= n);
      REQUIRE(c.hinge0 + c.nHinge <= M.hingeId.size());
      REQUIRE(c.bcode0 + (size_t)c.nBarCode * c.nOwn <= M.bcode.size() && M.barId.size() == 4 * M.bcode.size());
      REQUIRE(c.hcode0 + (size_t)c.nHingeCode * c.nOwn <= M.hcode.size());
      for (int i = 0; i < c.nNode; i++) REQUIRE(M.node[c.node0 + i] >= 0 && M.node[c.node0 + i] < n);
      for (int i = 0; i < c.nOwn; i++) {
        REQUIRE(M.node[c.node0 + i] == ord[c.own0 + i]);
        owned[ord[c.own0 + i]] += first;
      }
      for (int e = 0; e < c.nHinge; e++) {
        for (int q = 0; q < 4; q++) {
          const int pos = M.hinge[(c.hinge0 + e) * 4 + q];
          REQUIRE(pos < c.nNode && M.node[c.node0 + pos] == hin[(size_t)M.hingeId[c.hinge0 + e] * 4 + q]);
        }
        if (e < c.nHingeOwn) counted[1][M.hingeId[c.hinge0 + e]]++;
      }
      for (int i = 0; i < c.nOwn; i++) {
        bool end = false;
        for (int q = 0; q < 4 * c.nBarCode; q++) {
          const size_t at = c.bcode0 + (size_t)(q / 4) * c.nOwn + i;
          const int code = M.bcode[at].c[q % 4], id = M.barId[4 * at + q % 4];
          if (code == kBaHNoBar) {
            end = true;
            REQUIRE(id == 0);
            continue;
          }
          REQUIRE(!end && (code >> 1) < c.nNode);
          const int k = code & 1;
          REQUIRE(bar[2 * (size_t)id + k] == ord[c.own0 + i]);
          REQUIRE(bar[2 * (size_t)id + 1 - k] == M.node[c.node0 + (code >> 1)]);
          counted[0][id] += k == 0;
          seq[0][ord[c.own0 + i]].push_back(id * 2 + k);
        }
        end = false;
        for (int q = 0; q < 4 * c.nHingeCode; q++) {
          const int code = M.hcode[c.hcode0 + (size_t)(q / 4) * c.nOwn + i].c[q % 4];
          if (code == kBaHNoHinge) {
            end = true;
            continue;
          }
          REQUIRE(!end);
          const int e = code % kBaHCol, k = code / (3 * kBaHCol);
          REQUIRE(e < c.nHinge && k < 4 && code == bah_slot(e, k));
          REQUIRE(M.hinge[(c.hinge0 + e) * 4 + k] == i);
          seq[1][ord[c.own0 + i]].push_back(M.hingeId[c.hinge0 + e] * 4 + k);
        }
      }
      first = 0;
      if (!c.more) break;
    }
  }
  REQUIRE(visits == M.chunk.size());
  for (int i = 0; i < n; i++) REQUIRE(owned[i] == 1);
  for (int t = 0; t < 2; t++) {
    for (int v : counted[t]) REQUIRE(v == 1);
    const auto& list = t ? hin : bar;
    std::vector<std::vector<int>> want(n);
    for (size_t q = 0; q < list.size(); q++) want[list[q]].push_back((int)q);
    REQUIRE(want == seq[t]);
  }
  std::printf("%s: %d nodes, %zu clusters, %zu chunks, hinges evaluated %.3f per hinge\n", name, n,
              M.cluster.size(), M.chunk.size(), hin.empty() ? 0.0 : 4.0 * M.hingeId.size() / hin.size());
}

static void sheet(int nx, int ny, double scale, const char* name) {
  std::vector<int> bar, hin;
  auto id = [&](int i, int j) { return i * ny + j; };
  auto in = [&](int i, int j) { return i >= 0 && j >= 0 && i < nx && j < ny; };
  for (int i = 0; i < nx; i++)
    for (int j = 0; j < ny; j++) {
      const int to[3][2] = {{i + 1, j}, {i, j + 1}, {i + 1, j + 1}};
      const int tip[3][2][2] = {{{i + 1, j + 1}, {i, j - 1}}, {{i + 1, j + 1}, {i - 1, j}}, {{i + 1, j}, {i, j + 1}}};
      for (int k = 0; k < 3; k++) {
        if (!in(to[k][0], to[k][1])) continue;
        bar.insert(bar.end(), {id(i, j), id(to[k][0], to[k][1])});
        if (in(tip[k][0][0], tip[k][0][1]) && in(tip[k][1][0], tip[k][1][1]))
          hin.insert(hin.end(), {id(tip[k][0][0], tip[k][0][1]), id(i, j), id(to[k][0], to[k][1]),
                                 id(tip[k][1][0], tip[k][1][1])});
      }
    }
  std::vector<double> x;
  for (int i = 0; i < nx; i++)
    for (int j = 0; j < ny; j++) x.insert(x.end(), {scale * 0.95 * (i - 0.5 * j), scale * 0.866 * j, 0.0});
  check(name, nx * ny, bar, hin, x);
}

int main() {
  sheet(2, 2, 1, "sheet 2x2");
  sheet(24, 24, 1, "sheet 24x24");
  sheet(37, 211, 1, "sheet 37x211");
  sheet(512, 300, 1, "sheet 512x300");
  sheet(300, 512, 0, "sheet 300x512, all nodes at one point");
  std::mt19937 r(5);
  for (int n : {1, 2, 3, 700, 5000}) {
    // a star: every bar and hinge at node 0, a few repeated or with equal nodes
    std::vector<int> bar, hin;
    std::vector<double> x(3 * (size_t)n, NAN);
    for (int k = 0; k < 2 * n; k++) bar.insert(bar.end(), {0, (int)(r() % n)});
    for (int k = 0; k < 3 * n; k++) hin.insert(hin.end(), {(int)(r() % n), 0, (int)(r() % n), (int)(r() % n)});
    check("star", n, bar, hin, x);
    check("no elements", n, {}, {}, x);
    bar.clear();
    hin.clear();
    for (int k = 0; k < 2 * n; k++) bar.insert(bar.end(), {(int)(r() % n), (int)(r() % n)});
    for (int k = 0; k < 2 * n; k++)
      hin.insert(hin.end(), {(int)(r() % n), (int)(r() % n), (int)(r() % n), (int)(r() % n)});
    for (auto& v : x) v = (double)(r() % 1000);
    check("random", n, bar, hin, x);
  }
  return 0;
}
