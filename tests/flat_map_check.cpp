// CPU check of the flat-chunk decomposition (minim_amd/csrc/pf_tile.hpp), run by
// tests/test_tile_map.py: every site owned exactly once, every site loaded inside
// the plane, every LDS slot within its array and filled, and the slots that a
// site's neighbours are read from holding its periodic neighbours.
#include <cstdio>
#include <vector>

#include "pf_tile.hpp"

using namespace minim_amd;

static int check(int X, int Y, int Z, int R, int H, int xchunk, int target) {
  TileGeom G;
  if (!tile_geom(X, Y, Z, R, xchunk, target, 8192, G, H)) return 1;
  const int T = kTileWaves * kTileZ, cap = flat_slots(R, H);
  const long YZ = (long)Y * Z;
  std::vector<int> owned((size_t)X * YZ, 0);
  int bad = 0;
  for (int L = 0; L < G.nblocks; L++) {
    std::vector<long> slot(cap, -1);
    std::vector<FlatThread> th(T);
    auto put = [&](int s, unsigned site) {
      if (s < 0 || s >= cap || site >= (unsigned long)YZ || slot[s] >= 0) bad++;
      else slot[s] = site;
    };
    for (int t = 0; t < T; t++) {
      flat_thread(G, L, t, th[t]);
      if (th[t].x0 < 0 || th[t].x1 > X || th[t].x0 >= th[t].x1) bad++;
      for (int r = 0; r < R; r++) put(th[t].slot[r], th[t].site[r]);
      for (int h = 0; h < H; h++) {
        if (th[t].hsite[h] >= (unsigned long)YZ) bad++;
        if (th[t].hslot[h] >= 0) put(th[t].hslot[h], th[t].hsite[h]);
      }
    }
    for (int t = 0; t < T; t++)
      for (int r = 0; r < R; r++) {
        const FlatThread& o = th[t];
        const int at[4] = {o.slot[r] - Z, o.slot[r] + Z, o.zm[r], o.zp[r]};
        for (int s : at)  // read by every lane, owned or not
          if (s < 0 || s >= cap || slot[s] < 0) bad++;
        if (!(o.own & (1u << r)) || bad) continue;
        for (int i = o.x0; i < o.x1; i++) owned[(size_t)i * YZ + o.site[r]]++;
        const long y = o.site[r] / Z, z = o.site[r] % Z;
        const long want[4] = {((y + Y - 1) % Y) * Z + z, ((y + 1) % Y) * Z + z, y * Z + (z + Z - 1) % Z,
                              y * Z + (z + 1) % Z};
        for (int k = 0; k < 4; k++) bad += slot[at[k]] != want[k];
      }
    if (bad) break;
  }
  for (int v : owned) bad += v != 1;
  if (bad) std::printf("%dx%dx%d R=%d H=%d xchunk=%d: %d failures\n", X, Y, Z, R, H, xchunk, bad);
  return bad ? 1 : 0;
}

int main() {
  const int shapes[][3] = {{1, 1, 1},  {1, 1, 7},    {1, 5, 3},    {3, 1, 1},   {2, 2, 2},   {4, 17, 65}, {2, 30, 128},
                           {5, 3, 100}, {9, 131, 97}, {7, 33, 126}, {1, 200, 70}, {3, 70, 63}, {2, 1, 128}, {2, 9, 129},
                           {5, 150, 141}, {3, 40, 192}, {2, 1, 192}};
  int fails = 0, n = 0;
  for (const auto& s : shapes)
    for (int R : {1, 2, 4})
      for (int H : {1, 2}) {
        if (s[2] > (H == 1 ? 128 : kFlatMaxZ)) continue;
        for (int xc : {0, 1, 3}) {
          fails += check(s[0], s[1], s[2], R, H, xc, 512);
          n++;
        }
      }
  // the rule never asks for more halo sites than a thread stages or slots than there are
  for (int Y = 1; Y < 400; Y += 7)
    for (int Z = 1; Z < 400; Z++)
      for (int R : {2, 4}) {
        const int H = flat_halo(Y, Z, R);
        if (H && (2 * Z > 256 * H || 256 * R + 2 * Z > flat_slots(R, H))) fails++;
      }
  std::printf("%d cases, %d failed\n", n, fails);
  return fails ? 1 : 0;
}
