// pf_tile.hpp -- work decomposition of the tiled PhaseField stencil kernel.
//
// Plain C++ (host and device) so that the mapping can be checked on the CPU:
// every site of the grid must be owned by exactly one thread, and every
// address a thread touches must lie inside the grid.
//
// The canonical grid is X x Y x Z (Z contiguous).  A block of 4 wavefronts
// owns a tile of 64 z-sites x TY = 4R y-rows and marches over a chunk of x
// planes.  Lane l of wavefront w owns column z = z0 + l and the R rows
// y0 + wR .. y0 + wR + R-1 of every plane of the chunk.  Each plane of the
// tile is staged in LDS with a one-site halo ring: LDS row j holds grid row
// y0 - 1 + j and LDS column c holds z0 - 1 + c (rows 0 .. TY+1, columns
// 0 .. 65).  Coordinates are wrapped periodically, so a tile that overhangs
// the grid (Y % TY or Z % 64 != 0, or dimensions smaller than the tile)
// still loads valid sites: its overhanging lanes/rows hold exactly the
// wrapped neighbours the last in-grid sites need, and only "owned" rows are
// stored or summed.
//
// Where such tiles leave many lanes outside the grid (Z just above a multiple of
// 64), a block takes 256 R consecutive sites of the plane's linear order instead
// (flat chunks): thread t owns sites t, t + 256, ...  Its LDS slot j holds site
// base - Z + j of the plane (wrapped), so the y neighbours lie Z slots away and
// the z neighbours one slot away, or Z - 1 at the ends of a grid row.
#pragma once

#ifndef MINIM_HD
#if defined(__HIPCC__) || defined(__HIP__)
#define MINIM_HD __host__ __device__
#else
#define MINIM_HD
#endif
#endif

namespace minim_amd {

constexpr int kTileZ = 64;     // sites per tile row: one per lane of a wavefront
constexpr int kTileWaves = 4;  // wavefronts per block, stacked in y
constexpr int kMaxTileR = 4;   // y rows per thread

struct TileGeom {
  int X, Y, Z;
  int R, TY;            // rows per thread, rows per tile (4R)
  int ntz, nty, ntile;  // tiles per plane
  int xchunk, nxc;      // x planes per block, chunks along x
  int nblocks;          // ntile * nxc, x-chunk major
  int flat;             // 0: tiles; else flat chunks, with so many halo sites per thread
};

// Flat chunks: LDS slots for R rows and H halo sites per thread.  With H = 2 the
// slots, not the threads, set the largest Z.
constexpr int kFlatMaxZ = 192;
MINIM_HD constexpr int flat_slots(int R, int H) { return kTileWaves * kTileZ * R + (H == 1 ? 256 : 2 * kFlatMaxZ); }

struct FlatThread {
  int x0, x1;                // planes [x0, x1) marched by this block
  unsigned site[kMaxTileR];  // in-plane index of own rows, wrapped into the grid
  int slot[kMaxTileR];       // their LDS slots
  unsigned own;              // bit r: own row r lies inside the grid
  int zm[kMaxTileR], zp[kMaxTileR];  // LDS slots of their z neighbours
  unsigned hsite[2];         // halo sites this thread stages (own row 0 when none)
  int hslot[2];              // and their slots (negative: none)
};

struct TileThread {
  int x0, x1;                // planes [x0, x1) marched by this block
  int lrow0, lcol;           // LDS slot of own row 0 (own rows are lrow0 .. lrow0+R-1)
  int hrow, hcol;            // LDS slot this thread fills with a halo site (hrow < 0: none)
  unsigned hsite;            // in-plane index of that halo site (own row 0 when none)
  unsigned site[kMaxTileR];  // in-plane index (y*Z + z) of own rows, wrapped into the grid
  unsigned own;              // bit r: own row r lies inside the grid (stored and summed)
};

MINIM_HD inline int wrap_mod(int v, int n) {
  const int r = v % n;
  return r < 0 ? r + n : r;
}

// x plane of a (possibly out-of-range) plane index v, periodic in X.  The
// kernel reads planes x0-1 .. x1+1 of its chunk, so v lies in [-1, X+1]; with
// X = 1 or 2 that is more than one period away.
MINIM_HD inline int tile_plane(int v, int X) { return wrap_mod(v, X); }

// Every x plane the tiled kernel reads for chunk [x0, x1): the three planes
// x0-1, x0, x0+1 of its prologue and plane i+2 fetched while plane i is
// computed, for i in [x0, x1).
MINIM_HD inline int tile_planes_read(int x0, int x1) { return 3 + (x1 - x0); }
MINIM_HD inline int tile_plane_read(int x0, int k, int X) {
  return k < 3 ? tile_plane(x0 - 1 + k, X) : tile_plane(x0 + 2 + (k - 3), X);
}

// L: logical block index (x-chunk major), t: thread index in the block.
MINIM_HD inline void tile_thread(const TileGeom& G, int L, int t, TileThread& o) {
  const int xc = L / G.ntile, tile = L - xc * G.ntile;
  const int ty_t = tile / G.ntz, tz_t = tile - ty_t * G.ntz;
  const int w = t / kTileZ, lane = t - w * kTileZ;
  const int y0 = ty_t * G.TY, z0 = tz_t * kTileZ;
  const int zl = z0 + lane;
  const int z = wrap_mod(zl, G.Z);
  o.own = 0;
  for (int r = 0; r < kMaxTileR; r++) {
    const int yl = y0 + w * G.R + r;
    o.site[r] = (unsigned)(wrap_mod(yl, G.Y) * G.Z + z);
    if (r < G.R && yl < G.Y && zl < G.Z) o.own |= 1u << r;
  }
  o.x0 = xc * G.xchunk;
  o.x1 = (o.x0 + G.xchunk < G.X) ? o.x0 + G.xchunk : G.X;
  o.lrow0 = w * G.R + 1;
  o.lcol = lane + 1;
  o.hrow = -1;
  o.hcol = 0;
  o.hsite = o.site[0];
  if (t < kTileZ) {  // row above the tile
    o.hrow = 0;
    o.hcol = t + 1;
    o.hsite = (unsigned)(wrap_mod(y0 - 1, G.Y) * G.Z + wrap_mod(z0 + t, G.Z));
  } else if (t < 2 * kTileZ) {  // row below
    o.hrow = G.TY + 1;
    o.hcol = t - kTileZ + 1;
    o.hsite = (unsigned)(wrap_mod(y0 + G.TY, G.Y) * G.Z + wrap_mod(z0 + t - kTileZ, G.Z));
  } else if (t < 2 * kTileZ + G.TY) {  // column before
    const int j = t - 2 * kTileZ;
    o.hrow = j + 1;
    o.hcol = 0;
    o.hsite = (unsigned)(wrap_mod(y0 + j, G.Y) * G.Z + wrap_mod(z0 - 1, G.Z));
  } else if (t < 2 * kTileZ + 2 * G.TY) {  // column after
    const int j = t - 2 * kTileZ - G.TY;
    o.hrow = j + 1;
    o.hcol = kTileZ + 1;
    o.hsite = (unsigned)(wrap_mod(y0 + j, G.Y) * G.Z + wrap_mod(z0 + kTileZ, G.Z));
  }
}

MINIM_HD inline void flat_thread(const TileGeom& G, int Lb, int t, FlatThread& o) {
  const int T = kTileWaves * kTileZ, L = T * G.R, YZ = G.Y * G.Z;
  const int xc = Lb / G.ntile, base = (Lb - xc * G.ntile) * L;
  o.x0 = xc * G.xchunk;
  o.x1 = (o.x0 + G.xchunk < G.X) ? o.x0 + G.xchunk : G.X;
  o.own = 0;
  for (int r = 0; r < kMaxTileR; r++) {
    const int j = r * T + t, f = base + j, s = f % YZ, z = s % G.Z;
    o.site[r] = (unsigned)s;
    o.slot[r] = G.Z + j;
    o.zm[r] = o.slot[r] + (z == 0 ? G.Z - 1 : -1);
    o.zp[r] = o.slot[r] + (z == G.Z - 1 ? 1 - G.Z : 1);
    if (r < G.R && f < YZ) o.own |= 1u << r;
  }
  for (int h = 0; h < 2; h++) {
    const int j = h * T + t;
    if (h < G.flat && j < 2 * G.Z) {
      o.hslot[h] = j < G.Z ? j : L + j;
      o.hsite[h] = (unsigned)wrap_mod(base - G.Z + o.hslot[h], YZ);
    } else {
      o.hslot[h] = -1;
      o.hsite[h] = o.site[0];
    }
  }
}

// Flat chunks where they leave less to do: sites computed (lanes outside the
// grid included) and sites staged count alike, and the tiles, whose y neighbours
// come from registers, keep the grids where flat chunks save under a tenth.
MINIM_HD inline int flat_halo(int Y, int Z, int R) {
  if (Z > kFlatMaxZ) return 0;
  const long L = kTileWaves * kTileZ * R, TY = kTileWaves * R;
  const long tiles = (long)((Z + kTileZ - 1) / kTileZ) * ((Y + TY - 1) / TY);
  const long chunks = ((long)Y * Z + L - 1) / L;
  const long tile_cost = tiles * (kTileZ * TY + (kTileZ + 2) * (TY + 2)), flat_cost = chunks * (2 * L + 2 * Z);
  if (10 * flat_cost >= 9 * tile_cost) return 0;
  return Z <= 128 ? 1 : 2;
}

// Blocks per CU, in quarters, below which the march does not keep the chip busy, by
// the bytes of a site: a lane of a one-fluid field has little to do per plane.
MINIM_HD constexpr int march_busy(int siteBytes) { return siteBytes <= 4 ? 11 : siteBytes <= 8 ? 10 : 8; }

// Tile geometry for R rows per thread (flat: from flat_halo).  xchunk > 0 forces
// the x-march length, else the march is as short as at most target_blocks blocks
// allow (two per CU by default), or, with busy (from march_busy), one chunk
// more where that takes the fullest CU less time: its blocks, but busy / 4 of
// them at least, times their planes and six more for the start of the march.
// Energy and gradient, one chunk fewer and one more: 160x150x141x3 in FP64 480
// blocks 38.8 us, 540 48.6; 190x180x187x3 504 62.8, 540 76.8; 64x320x896x3 280
// blocks 251, 560 216; 40x512x576x1 in FP32 288 blocks 40.9, 576 25.9.  Over 2,455
// launches of one to four fluids, 0.25 to 22 M sites, the choice is 0.1 % off the
// better one in the mean (2.2 % for at most, 9.6 % for at least the target) and
// 14 % at worst (65, 40).  Returns false when the grid cannot be launched (more
// than max_blocks blocks).
MINIM_HD inline bool tile_geom(int X, int Y, int Z, int R, int xchunk, int target_blocks, int max_blocks,
                               TileGeom& G, int flat = 0, int busy = 0) {
  G.X = X;
  G.Y = Y;
  G.Z = Z;
  G.R = R;
  G.TY = kTileWaves * R;
  G.ntz = (Z + kTileZ - 1) / kTileZ;
  G.nty = (Y + G.TY - 1) / G.TY;
  G.ntile = G.ntz * G.nty;
  G.flat = flat;
  if (flat) {
    const long L = kTileWaves * kTileZ * R;
    G.ntile = (int)(((long)Y * Z + L - 1) / L);
  }
  if (xchunk <= 0) {
    long nxc = target_blocks / G.ntile;
    if (nxc < 1) nxc = 1;
    if (nxc > X) nxc = X;
    xchunk = (int)((X + nxc - 1) / nxc);
    if (busy > 0 && nxc < X && G.ntile < target_blocks && target_blocks % G.ntile != 0) {
      const long CUs = 256;
      long cost[2];
      int chunk[2] = {xchunk, (int)((X + nxc) / (nxc + 1))};
      for (int k = 0; k < 2; k++) {
        const long blocks = (long)G.ntile * ((X + chunk[k] - 1) / chunk[k]), quarters = 4 * ((blocks + CUs - 1) / CUs);
        cost[k] = (quarters > busy ? quarters : busy) * (chunk[k] + 6);
      }
      if (cost[1] < cost[0]) xchunk = chunk[1];
    }
  }
  if (xchunk > X) xchunk = X;
  if (xchunk < 1) xchunk = 1;
  G.xchunk = xchunk;
  G.nxc = (X + xchunk - 1) / xchunk;
  while ((long)G.ntile * G.nxc > max_blocks && G.xchunk < X) {
    G.xchunk *= 2;
    if (G.xchunk > X) G.xchunk = X;
    G.nxc = (X + G.xchunk - 1) / G.xchunk;
  }
  G.nblocks = G.ntile * G.nxc;
  return (long)G.ntile * G.nxc <= max_blocks;
}

}  // namespace minim_amd
