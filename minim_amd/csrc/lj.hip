// lj.hip -- Lennard-Jones potential on MI355X.
//
// Reference semantics (LjNd::init / elementEnergyGradient,
// src/potentials/LjNd.cpp:12-53): one element per pair i<j, E = 4 eps (lj12 -
// lj6), g_i += dx * (-24 eps (2 lj12 - lj6) / r^2), g_j -= the same.  The
// reference stores N(N-1)/2 heap elements and scatters into g; here one block
// owns particle i and gathers over all j, so the gradient is written once per
// particle with no atomics and the energy is the FP64 sum of per-particle
// halves.
//
// Cutoff mode (no reference counterpart): truncated-and-shifted at rc in a
// periodic box, with a full Verlet list of radius rc+skin built from a cell
// list; the list is rebuilt when any particle has moved more than skin/2 from
// where the list was built.  Lists are built deterministically (cell contents
// sorted by particle id), so energies and gradients are reproducible.
#include <algorithm>
#include <climits>
#include <cmath>
#include <stdexcept>
#include <type_traits>
#include <typeinfo>
#include <vector>

#include "common.hpp"
#include "minim/LjNd.h"
#include "runtime.hpp"
#include "vec.hpp"

namespace minim_amd {
namespace {

template <typename T, int D>
__device__ inline void load_pos(const T* __restrict__ x, const T* __restrict__ d, T t, int i, T (&p)[D]) {
#pragma unroll
  for (int k = 0; k < D; k++) {
    T c = x[(size_t)i * D + k];
    if (d) {
      T s = t * d[(size_t)i * D + k];
      c = c + s;
    }
    p[k] = c;
  }
}

// All pairs, gather form: a block takes R particles at a time and spreads the
// other particles j over its threads, so that a cluster of N particles has
// N/R blocks of N/256 steps each; the block sums the R gradients in FP64 and
// one thread stores them.  Bound by FP64 issue (the division) when N is large
// and by the latency of one pass over the positions when it is small.  Energy and
// gradient, both on the device, in 3-D FP64: 9.6 us at 64 particles and 10 us at
// 1,000 (the host's two launches; the pairs take 6 us), 29 us at 4,096; one thread
// per particle with a serial loop over j (4 blocks for 1,000 particles), waited
// for by the host, took 45, 221 and 807 us.  Lanes add N/256 terms each and the block adds the lanes in
// FP64, so the gradient's error against 64 bits fell too (1,000 particles,
// 3-D: 1.2e-15 -> 6e-16 in FP64, 1.1e-6 -> 7.6e-7 in FP32).  MODE bit 1
// energy, bit 2 gradient.
//
// s2: 4^-k with 2^k <= sigma < 2^(k+1), and sig6 the sixth power of sigma / 2^k,
// so that 1 / r^6 stays in range wherever (sigma / r)^6 does (a power of two
// rounds nothing); where r^4 does not, the pair's force is zero.
template <typename T, int D, int R, int MODE>
__global__ __launch_bounds__(kBlock) void lj_allpairs_kernel(const T* __restrict__ x, const T* __restrict__ d, T t,
                                                             int N, T sig6, T eps, T s2, T* __restrict__ g,
                                                             RedScratch rs) {
  constexpr bool WE = MODE & 1, WG = MODE & 2;
  constexpr T most = sizeof(T) == 8 ? (T)1.79769313486231571e308 : (T)3.40282347e38f;
  constexpr int U = 4;  // positions requested before any is used
  __shared__ double lds[(kBlock / kWave) * (WG ? R * D : 1)];
  const int ngroup = (N + R - 1) / R;
  double ei = 0.0;
  for (int q = blockIdx.x; q < ngroup; q += gridDim.x) {
    T xi[R][D], gi[R][D];
#pragma unroll
    for (int r = 0; r < R; r++) {
      load_pos<T, D>(x, d, t, min(q * R + r, N - 1), xi[r]);
#pragma unroll
      for (int k = 0; k < D; k++) gi[r][k] = (T)0;
    }
    for (int j0 = threadIdx.x; j0 < N; j0 += U * kBlock) {
      T pj[U][D];
#pragma unroll
      for (int u = 0; u < U; u++) load_pos<T, D>(x, d, t, min(j0 + u * kBlock, N - 1), pj[u]);
#pragma unroll
      for (int u = 0; u < U; u++) {
        const int j = j0 + u * kBlock;
        if (j >= N) break;
#pragma unroll
        for (int r = 0; r < R; r++) {
          const int i = q * R + r;
          T dx[D], r2 = (T)0;
#pragma unroll
          for (int k = 0; k < D; k++) {
            dx[k] = xi[r][k] - pj[u][k];
            r2 = fma(dx[k], dx[k], r2);
          }
          if (j == i || i >= N) continue;
          const T q2 = s2 * r2, q4 = q2 * q2;
          const T ir6 = (T)1 / (q4 * q2);  // one division per pair
          const T lj6 = sig6 * ir6;
          const T lj12 = lj6 * lj6;
          if (WE) ei += 0.5 * (double)((T)4 * eps * (lj12 - lj6));
          if (WG) {
            const T f = (T)-24 * eps * s2 * ((T)2 * lj12 - lj6) * (ir6 * fmin(q4, most));
#pragma unroll
            for (int k = 0; k < D; k++) gi[r][k] = fma(dx[k], f, gi[r][k]);
          }
        }
      }
    }
    if constexpr (WG) {
      double v[R * D];
#pragma unroll
      for (int r = 0; r < R; r++)
#pragma unroll
        for (int k = 0; k < D; k++) v[r * D + k] = (double)gi[r][k];
      block_sum<R * D>(v, lds);
      if (threadIdx.x == 0) {
#pragma unroll
        for (int r = 0; r < R; r++)
#pragma unroll
          for (int k = 0; k < D; k++)
            if (q * R + r < N) g[(size_t)(q * R + r) * D + k] = (T)v[r * D + k];
      }
      __syncthreads();  // the next group's sums reuse lds
    }
  }
  double acc[1] = {ei};
  grid_sum_store<1>(acc, rs);
}

// ---------------------------------------------------------------- cutoff mode
struct BoxArgs {
  double L[3];
  double invL[3];
  double inv_cell[3];
  int nc[3];
  double rlist2;
  double rc2;
  double half_skin2;
};

// Minimum image v - L rint(v / L), with v / L taken as v * (1/L): the two
// can round to different integers only when |v| is within an ulp of L/2,
// where both images are far beyond any cutoff.
template <typename T>
__device__ inline T min_image(T v, T L, T invL) {
  return fma(-L, rint(v * invL), v);
}

template <typename T>
__global__ __launch_bounds__(kBlock) void lj_cell_index_kernel(const T* __restrict__ x, int N, BoxArgs b,
                                                               int* __restrict__ cell, int* __restrict__ count,
                                                               double* __restrict__ xbuild) {
  const int i = blockIdx.x * kBlock + threadIdx.x;
  if (i >= N) return;
  int c[3];
  bool lost = false;
#pragma unroll
  for (int k = 0; k < 3; k++) {
    const double v = (double)x[(size_t)i * 3 + k];
    xbuild[(size_t)i * 3 + k] = v;
    double w = v - b.L[k] * floor(v / b.L[k]);  // wrapped into [0, L)
    lost = lost || !isfinite(w);
    int ci = (int)(w * b.inv_cell[k]);
    if (ci >= b.nc[k]) ci = b.nc[k] - 1;
    if (ci < 0) ci = 0;
    c[k] = ci;
  }
  int id = (c[0] * b.nc[1] + c[1]) * b.nc[2] + c[2];
  // no pair of such a particle is within the list radius: any cell will do, and
  // all of a diverged system in one would be sorted and paired there
  if (lost) id = i % (b.nc[0] * b.nc[1] * b.nc[2]);
  cell[i] = id;
  atomicAdd(&count[id], 1);
}

// Zero cell counts and overflow flag.
__global__ __launch_bounds__(kBlock) void lj_clear_kernel(int* __restrict__ count, int ncell, int* __restrict__ flag) {
  for (int c = blockIdx.x * kBlock + threadIdx.x; c < ncell; c += gridDim.x * kBlock) count[c] = 0;
  if (blockIdx.x == 0 && threadIdx.x == 0) *flag = 0;
}

// Exclusive scan of cell counts by a single block (cell counts are small).
__global__ __launch_bounds__(kBlock) void lj_scan_kernel(const int* __restrict__ count, int* __restrict__ start,
                                                         int* __restrict__ cursor, int ncell) {
  __shared__ int part[kBlock];
  const int per = (ncell + kBlock - 1) / kBlock;
  const int lo = threadIdx.x * per, hi = min(lo + per, ncell);
  int s = 0;
  for (int c = lo; c < hi; c++) s += count[c];
  part[threadIdx.x] = s;
  __syncthreads();
  if (threadIdx.x == 0) {
    int run = 0;
    for (int k = 0; k < kBlock; k++) {
      int v = part[k];
      part[k] = run;
      run += v;
    }
  }
  __syncthreads();
  int run = part[threadIdx.x];
  for (int c = lo; c < hi; c++) {
    start[c] = run;
    cursor[c] = 0;
    run += count[c];
  }
  if (threadIdx.x == kBlock - 1) start[ncell] = run;
}

__global__ __launch_bounds__(kBlock) void lj_fill_kernel(const int* __restrict__ cell, int N,
                                                         const int* __restrict__ start, int* __restrict__ cursor,
                                                         int* __restrict__ order) {
  const int i = blockIdx.x * kBlock + threadIdx.x;
  if (i >= N) return;
  const int c = cell[i];
  const int pos = start[c] + atomicAdd(&cursor[c], 1);
  order[pos] = i;
}

// A coordinate wrapped into [0, L), as the cell index takes it.
__device__ __forceinline__ double wrap_box(double v, double L) { return v - L * floor(v / L); }

// Sort each cell's members by particle id so the neighbour order is
// reproducible: one wavefront per cell; a lane computes the rank of a member by
// comparing it with all others (ids are distinct, so the ranks are a
// permutation), with up to 64 members from registers.  The members' positions go
// out in that order, wrapped into the box, each with its particle id: xc[p] =
// (x, y, z, j) (FP64, the list is built in FP64 in either precision), so that the
// list build reads one contiguous 32-byte entry per candidate instead of an
// index and then three scattered coordinates.
template <typename T>
__global__ __launch_bounds__(kBlock) void lj_sort_cells_kernel(const T* __restrict__ x, BoxArgs b,
                                                               const int* __restrict__ start,
                                                               const int* __restrict__ order, int ncell,
                                                               double4* __restrict__ xc) {
  const int lane = threadIdx.x % kWave;
  const int c = blockIdx.x * (kBlock / kWave) + threadIdx.x / kWave;
  if (c >= ncell) return;  // uniform over the wavefront
  const int lo = start[c], hi = start[c + 1], k = hi - lo;
  auto put = [&](int p, int j) {
    xc[p] = make_double4(wrap_box((double)x[(size_t)j * 3], b.L[0]), wrap_box((double)x[(size_t)j * 3 + 1], b.L[1]),
                         wrap_box((double)x[(size_t)j * 3 + 2], b.L[2]), (double)j);
  };
  if (k <= kWave) {
    const int v = lane < k ? order[lo + lane] : INT_MAX;
    int rank = 0;
    for (int q = 0; q < k; q++) rank += __shfl(v, q, kWave) < v ? 1 : 0;
    if (lane < k) put(lo + rank, v);
  } else {
    for (int a = lane; a < k; a += kWave) {
      const int v = order[lo + a];
      int rank = 0;
      for (int q = 0; q < k; q++) rank += order[lo + q] < v ? 1 : 0;
      put(lo + rank, v);
    }
  }
}

// Verlet list layout: for each group of 64 consecutive particles (one
// wavefront), maxn rows of 64 entries, so that entry k of particle i sits at
// ((i / 64) maxn + k) 64 + i % 64.  A wavefront's lanes read row k of their
// group together (one coalesced 256-byte access in the force pass), and a
// wavefront building its list writes only within its group's maxn x 64
// region, which stays cached until it is complete (with rows of all N
// particles, each lane's k-th entry fell in a different region of a list
// larger than L2).
__host__ __device__ inline size_t nbr_at(int i, int k, int maxn) {
  return ((size_t)(i >> 6) * maxn + k) * 64 + (i & 63);
}
inline size_t nbr_elems(int N, int maxn) { return (size_t)((N + 63) / 64) * 64 * maxn; }

// A list's rows are filled up to a multiple of kListPad (which maxn is too)
// with the particle itself, which the force pass skips: it reads whole chunks.
constexpr int kListPad = 32;
__device__ inline void pad_list(int i, int cnt, int maxn, int* __restrict__ nn, int* __restrict__ nbr) {
  const int n = min(cnt, maxn);
  nn[i] = n;
  for (int k = n; k % kListPad != 0; k++) nbr[nbr_at(i, k, maxn)] = i;
}

// Full Verlet list: neighbour k of particle i at nbr[nbr_at(i, k, maxn)].  The 27
// cells around i's cell are visited in a fixed order and each cell's members
// in particle-id order (lj_sort_cells_kernel), so the list -- and with it the
// order in which the force pass sums pairs -- does not depend on scheduling.
// With at least 3 cells of side >= rc + skin along each axis, the image of a
// neighbour cell that lies within the list radius is the one its index wrap
// implies, so each candidate needs no minimum-image rounding: i's wrapped
// position is shifted once per neighbour cell.  Pairs are kept below the
// list radius widened by 1e-12 of itself, so no pair the minimum-image test
// keeps is lost to rounding; a pair kept in excess lies beyond the cutoff
// (or at it, for skin 0) and the force pass, which tests the cutoff itself,
// skips it.
//
// Q lanes per particle, each testing every Q-th candidate; a ballot gives the
// kept ones consecutive entries in candidate order.  Cells that are neighbours
// in z are neighbours in memory, so away from the z faces the three are one run.
// Particles are taken in cell order (those of xc), so that a wavefront's
// lanes read the same candidates.  Bound by the latency of the candidate loads
// where there are few wavefronts and by the scattered writes of the list where
// there are many (32,768 particles: 60 us, one lane per particle 150).
template <int Q>
__global__ __launch_bounds__(kBlock) void lj_build_list_kernel(int N, BoxArgs b, const int* __restrict__ cell,
                                                               const int* __restrict__ start,
                                                               const double4* __restrict__ xc, int maxn,
                                                               int* __restrict__ nn, int* __restrict__ nbr,
                                                               int* __restrict__ overflow) {
  constexpr int U = 2;  // candidates requested per lane before any is used
  const int pi = (blockIdx.x * kBlock + threadIdx.x) / Q, sub = threadIdx.x % Q;
  if (pi >= N) return;
  const int first = (threadIdx.x % kWave) / Q * Q;  // this particle's lanes in the wavefront
  const double4 vi = xc[pi];
  const int i = (int)vi.w;
  const double xw0 = vi.x, xw1 = vi.y, xw2 = vi.z;
  const double rl2 = b.rlist2 * (1.0 + 1e-12);
  const int c = cell[i];
  const int cz = c % b.nc[2], cy = (c / b.nc[2]) % b.nc[1], cx = c / (b.nc[1] * b.nc[2]);
  const bool inner = cz > 0 && cz < b.nc[2] - 1;
  int cnt = 0;
  for (int dx = -1; dx <= 1; dx++) {
    const int ux = cx + dx;
    const int ax = ux < 0 ? ux + b.nc[0] : (ux >= b.nc[0] ? ux - b.nc[0] : ux);
    // the neighbour cell's image sits at its wrapped position -/+ L
    const double xi0 = ux < 0 ? xw0 + b.L[0] : (ux >= b.nc[0] ? xw0 - b.L[0] : xw0);
    for (int dy = -1; dy <= 1; dy++) {
      const int uy = cy + dy;
      const int ay = uy < 0 ? uy + b.nc[1] : (uy >= b.nc[1] ? uy - b.nc[1] : uy);
      const double xi1 = uy < 0 ? xw1 + b.L[1] : (uy >= b.nc[1] ? xw1 - b.L[1] : xw1);
      const int row = (ax * b.nc[1] + ay) * b.nc[2];
      for (int dz = inner ? 1 : -1; dz <= 1; dz++) {
        const int uz = cz + dz;
        const int az = uz < 0 ? uz + b.nc[2] : (uz >= b.nc[2] ? uz - b.nc[2] : uz);
        const double xi2 = uz < 0 ? xw2 + b.L[2] : (uz >= b.nc[2] ? xw2 - b.L[2] : xw2);
        const int p1 = start[row + az + 1];
        for (int p0 = start[row + (inner ? cz - 1 : az)]; p0 < p1; p0 += U * Q) {
          double4 v[U];
#pragma unroll
          for (int u = 0; u < U; u++) v[u] = xc[min(p0 + u * Q + sub, p1 - 1)];
#pragma unroll
          for (int u = 0; u < U; u++) {
            const int j = (int)v[u].w;
            const double r0 = xi0 - v[u].x, r1 = xi1 - v[u].y, r2 = xi2 - v[u].z;
            const bool keep = p0 + u * Q + sub < p1 && j != i && r0 * r0 + r1 * r1 + r2 * r2 < rl2;
            const unsigned long long all = (__ballot(keep) >> first) & ((1ull << Q) - 1);
            const int at = cnt + __popcll(all & ((1ull << sub) - 1));
            if (keep && at < maxn) nbr[nbr_at(i, at, maxn)] = j;
            cnt += __popcll(all);
          }
        }
      }
    }
  }
  if (sub == 0) {
    pad_list(i, cnt, maxn, nn, nbr);
    if (cnt > maxn) atomicMax(overflow, cnt);
  }
}

// Small boxes (fewer than 3 cells along a side): list by brute force.
template <typename T>
__global__ __launch_bounds__(kBlock) void lj_build_list_brute_kernel(const T* __restrict__ x, int N, BoxArgs b,
                                                                     int maxn, int* __restrict__ nn,
                                                                     int* __restrict__ nbr,
                                                                     int* __restrict__ overflow,
                                                                     double* __restrict__ xbuild) {
  const int i = blockIdx.x * kBlock + threadIdx.x;
  if (i >= N) return;
  double xi[3];
  for (int k = 0; k < 3; k++) {
    xi[k] = (double)x[(size_t)i * 3 + k];
    xbuild[(size_t)i * 3 + k] = xi[k];
  }
  int cnt = 0;
  for (int j = 0; j < N; j++) {
    if (j == i) continue;
    double r2 = 0;
    for (int k = 0; k < 3; k++) {
      const double v = min_image(xi[k] - (double)x[(size_t)j * 3 + k], b.L[k], b.invL[k]);
      r2 += v * v;
    }
    if (r2 < b.rlist2) {
      if (cnt < maxn) nbr[nbr_at(i, cnt, maxn)] = j;
      cnt++;
    }
  }
  pad_list(i, cnt, maxn, nn, nbr);
  if (cnt > maxn) atomicMax(overflow, cnt);
}

// The evaluated point x + t*d, for a line-search trial.
template <typename T>
__global__ __launch_bounds__(kBlock) void lj_point_kernel(const T* __restrict__ x, const T* __restrict__ d, T t,
                                                          size_t n, T* __restrict__ xt) {
  const size_t i = (size_t)blockIdx.x * kBlock + threadIdx.x;
  if (i >= n) return;
  const T s = t * d[i];
  xt[i] = x[i] + s;
}

template <typename T>
struct Pos3 {
  T c[3];
};

// P lanes per particle over its Verlet list, each taking U of every U P
// entries: their indices and then their positions are all requested before any
// is used.  Each lane sums its pairs in list order, and the lanes are added in
// a fixed tree.  The same pass counts the particles that have moved more than
// skin/2 since the list was built (reduction slot 1): when any has, the caller
// rebuilds the list and evaluates again.  Blocks are spread over the XCDs in
// contiguous ranges, so each L2 holds the positions of one spatially coherent
// range of particles.  MODE bit 1 energy, bit 2 gradient, bit 4 (with 2) FIRE's
// sums.  Reduction rows: energy, moved, list overflow; or g.g, v.g, v.v, moved,
// list overflow, largest |g_i|^2.
//
// Bound by VALU issue, about 40 instructions per entry: the reciprocal by
// Newton's iteration, fused products, constant factors and the energy shift
// taken out of the loop, and list rows filled up to whole chunks instead of
// clamped indices (69 before).  Positions are read in place, one 12-byte load
// in FP32 and two loads in FP64.  Force pass at 262,144 particles: 31 us FP32,
// 53 us FP64; with padded copies of the positions and one lane 43 and 69, and at
// 32,768 particles 7.9 and 11.5 against 20 and 23.
template <typename T, int P, int U, int MODE>
__global__ __launch_bounds__(kBlock) void lj_cut_kernel(const T* __restrict__ x, int N, BoxArgs b, T sig2, double eps,
                                                        double eshift, const int* __restrict__ nn,
                                                        const int* __restrict__ nbr, int maxn,
                                                        const double* __restrict__ xbuild,
                                                        const int* __restrict__ overflow, const T* __restrict__ v,
                                                        T* __restrict__ g, RedScratch rs) {
  static_assert(kListPad % (P * U) == 0, "whole chunks");
  constexpr bool WE = MODE & 1, WG = MODE & 2, WS = MODE & 4;
  const int tid = xcd_logical_block(blockIdx.x, gridDim.x) * kBlock + threadIdx.x;
  const int i = tid / P, sub = tid % P;
  auto at = [&](unsigned j) {
    // a 32-bit byte offset from a uniform base
    return *reinterpret_cast<const Pos3<T>*>(reinterpret_cast<const char*>(x) + j * (unsigned)sizeof(Pos3<T>));
  };
  double ei = 0.0, moved = 0.0;
  double gg = 0.0, vg = 0.0, vv = 0.0;
  if (i < N) {
    const Pos3<T> xi = at(i);
    const T L0 = (T)b.L[0], L1 = (T)b.L[1], L2 = (T)b.L[2];
    const T rc2 = (T)b.rc2;
    const T iL0 = (T)b.invL[0], iL1 = (T)b.invL[1], iL2 = (T)b.invL[2];
    T gi[3] = {(T)0, (T)0, (T)0};
    int pairs = 0;
    const int cnt = nn[i];
    const int* row = nbr + nbr_at(i, sub, maxn);
    for (int k0 = 0; k0 < cnt; k0 += U * P, row += U * P * 64) {
      int jj[U];
#pragma unroll
      for (int u = 0; u < U; u++) jj[u] = row[u * P * 64];
      Pos3<T> xj[U];
#pragma unroll
      for (int u = 0; u < U; u++) xj[u] = at(jj[u]);
#pragma unroll
      for (int u = 0; u < U; u++) {
        const T r0 = min_image(xi.c[0] - xj[u].c[0], L0, iL0);
        const T r1 = min_image(xi.c[1] - xj[u].c[1], L1, iL1);
        const T r2v = min_image(xi.c[2] - xj[u].c[2], L2, iL2);
        const T r2 = fma(r0, r0, fma(r1, r1, r2v * r2v));
        const bool in = !(r2 >= rc2) && jj[u] != i;
        const T ir2 = in ? newton_rcp(r2) : (T)0;
        const T s2 = sig2 * ir2;
        const T lj6 = s2 * s2 * s2;
        if (WE) {
          ei += (double)fma(lj6, lj6, -lj6);
          pairs += in;
        }
        if (WG) {
          const T f = fma((T)2 * lj6, lj6, -lj6) * s2;  // in units of epsilon and sigma: in range as lj6^2 is
          gi[0] = fma(r0, f, gi[0]);
          gi[1] = fma(r1, f, gi[1]);
          gi[2] = fma(r2v, f, gi[2]);
        }
      }
    }
    if (WE) ei = 0.5 * (4 * eps * ei - pairs * eshift);
    if (WG) {
#pragma unroll
      for (int off = 1; off < P; off <<= 1)
#pragma unroll
        for (int k = 0; k < 3; k++) gi[k] += __shfl_xor(gi[k], off, kWave);
    }
    if (sub == 0) {
      double dr2 = 0;
#pragma unroll
      for (int k = 0; k < 3; k++) {
        const double v = (double)xi.c[k] - xbuild[(size_t)i * 3 + k];
        dr2 += v * v;
      }
      if (dr2 > b.half_skin2) moved = 1.0;
      if (WG) {
        const T f = (T)(-24 * eps / (double)sig2);
#pragma unroll
        for (int k = 0; k < 3; k++) {
          const T gk = f * gi[k];
          g[(size_t)i * 3 + k] = gk;
          if (WS) {
            const double gd = (double)gk, vd = (double)v[(size_t)i * 3 + k];
            gg += gd * gd;
            vg += vd * gd;
            vv += vd * vd;
          }
        }
      }
    }
  }
  const double over = blockIdx.x == 0 && threadIdx.x == 0 ? (double)*overflow : 0.0;
  if constexpr (WS) {
    __shared__ double lds[kBlock / kWave];
    const double m = block_max(gg, lds);  // a lane holds one particle
    if (threadIdx.x == 0) rs.partials[(size_t)5 * gridDim.x + blockIdx.x] = m;
    double acc[5] = {gg, vg, vv, moved, over};
    grid_sum_store<5>(acc, rs);
  } else {
    double acc[3] = {ei, moved, over};
    grid_sum_store<3>(acc, rs);
  }
}

template <typename T, int D>
int launch_allpairs_d(const T* x, const T* d, T t, int N, T sig6, T eps, T s2, int mode, T* g, RedScratch rs,
                      hipStream_t s) {
  auto go = [&](auto rtag) {
    constexpr int R = decltype(rtag)::value;
    const int nb = grid_blocks((size_t)((N + R - 1) / R) * kBlock);
    switch (mode) {
      case 1: lj_allpairs_kernel<T, D, R, 1><<<nb, kBlock, 0, s>>>(x, d, t, N, sig6, eps, s2, g, rs); break;
      case 2: lj_allpairs_kernel<T, D, R, 2><<<nb, kBlock, 0, s>>>(x, d, t, N, sig6, eps, s2, g, rs); break;
      default: lj_allpairs_kernel<T, D, R, 3><<<nb, kBlock, 0, s>>>(x, d, t, N, sig6, eps, s2, g, rs); break;
    }
    return nb;
  };
  // Four particles per block share each position read and each block's sum;
  // below 2,048 particles that leaves too few blocks for 256 CUs.
  return N < 2048 ? go(std::integral_constant<int, 1>()) : go(std::integral_constant<int, 4>());
}

template <typename T>
void launch_allpairs(int D, const void* x, const void* d, double t, int N, double sigma, double eps, int mode, void* g,
                     RedScratch rs, hipStream_t s, double* eDev = nullptr) {
  if (N < 1) throw std::invalid_argument("LjNd: no particles");
  if ((N + kBlock - 1) / kBlock > kMaxRedBlocks)
    throw std::invalid_argument("LjNd: too many particles for the all-pairs kernel");
  const T* xx = (const T*)x;
  const T* dd = (const T*)d;
  T* gg = (T*)g;
  const int k = sigma != 0 && std::isfinite(sigma) ? std::max(-60, std::min(60, std::ilogb(sigma))) : 0;
  const T sig6 = (T)std::pow(std::ldexp(sigma, -k), 6), s2 = (T)std::ldexp(1.0, -2 * k), tt = (T)t, ee = (T)eps;
  rs = rs.only(0, (mode & 1) ? eDev : nullptr);
  int nb = 0;
  switch (D) {
    case 1: nb = launch_allpairs_d<T, 1>(xx, dd, tt, N, sig6, ee, s2, mode, gg, rs, s); break;
    case 2: nb = launch_allpairs_d<T, 2>(xx, dd, tt, N, sig6, ee, s2, mode, gg, rs, s); break;
    case 3: nb = launch_allpairs_d<T, 3>(xx, dd, tt, N, sig6, ee, s2, mode, gg, rs, s); break;
    case 4: nb = launch_allpairs_d<T, 4>(xx, dd, tt, N, sig6, ee, s2, mode, gg, rs, s); break;
    default: throw std::invalid_argument("LjNd: nDim must be 1..4 on the device path");
  }
  MINIM_HIP_CHECK(hipGetLastError());
  launch_finalize(rs, 1, nb, s);
}

}  // namespace
}  // namespace minim_amd

namespace minim {

using minim_amd::DeviceBuffer;
using minim_amd::kBlock;

struct LjNd::Impl {
  minim_amd::BoxArgs box{};
  bool cellMode = false;
  int maxn = 128;  // a multiple of kListPad
  long builds = 0;
  bool built = false;
  DeviceBuffer cell, count, start, cursor, order, nn, nbr, flag, xbuild, xtrial, xcell;
  int ncell = 0;
};

LjNd::LjNd(const LjNd& o)
    : NewPotential<LjNd>(o), nDim(o.nDim), nParticle(o.nParticle), sigma(o.sigma), epsilon(o.epsilon),
      cutoff(o.cutoff), box(o.box), skin(o.skin) {}

LjNd& LjNd::operator=(const LjNd& o) {
  NewPotential<LjNd>::operator=(o);
  nDim = o.nDim;
  nParticle = o.nParticle;
  sigma = o.sigma;
  epsilon = o.epsilon;
  cutoff = o.cutoff;
  box = o.box;
  skin = o.skin;
  impl_.reset();
  return *this;
}

LjNd::~LjNd() = default;

LjNd& LjNd::setSigma(double s) {
  sigma = s;
  return *this;
}
LjNd& LjNd::setEpsilon(double e) {
  epsilon = e;
  return *this;
}
LjNd& LjNd::setCutoff(double rc, std::array<double, 3> b, double sk) {
  if (rc <= 0 || sk < 0) throw std::invalid_argument("LjNd: cutoff must be positive and skin non-negative.");
  for (double v : b)
    if (v <= 0) throw std::invalid_argument("LjNd: box lengths must be positive.");
  cutoff = rc;
  box = b;
  skin = sk;
  return *this;
}

long LjNd::listBuilds() const { return impl_ ? impl_->builds : 0; }
// The largest list length of the last build, read back from the device (a
// statistic: it waits for the device).
int LjNd::maxNeighbours() const {
  if (!impl_ || !impl_->built) return 0;
  std::vector<int> h(nParticle);
  MINIM_HIP_CHECK(hipMemcpy(h.data(), impl_->nn.get(), sizeof(int) * h.size(), hipMemcpyDeviceToHost));
  int mx = 0;
  for (int v : h) mx = v > mx ? v : mx;
  return mx;
}

// LjNd::init (src/potentials/LjNd.cpp:12-26): nParticle from the coordinate count.
void LjNd::init(const vector<double>& coords) {
  if (nDim < 1) throw std::invalid_argument("LjNd: nDim must be positive.");
  if (coords.size() % nDim != 0)
    throw std::invalid_argument("LjNd: Length of coords must be a multiple of the number of dimensions.");
  nParticle = (int)(coords.size() / nDim);
  uploadFixed(coords.size());
  impl_ = std::make_shared<Impl>();
  if (cutoff > 0) {
    if (nDim != 3) throw std::invalid_argument("LjNd: the cutoff/periodic mode needs nDim = 3.");
    auto& b = impl_->box;
    const double rl = cutoff + skin;
    for (int k = 0; k < 3; k++) {
      if (box[k] < 2 * cutoff) throw std::invalid_argument("LjNd: box must be at least twice the cutoff.");
      b.L[k] = box[k];
      b.nc[k] = (int)std::floor(box[k] / rl);
      if (b.nc[k] < 1) b.nc[k] = 1;
      b.inv_cell[k] = b.nc[k] / box[k];
    }
    b.rlist2 = rl * rl;
    for (int k = 0; k < 3; k++) b.invL[k] = 1.0 / box[k];
    b.rc2 = cutoff * cutoff;
    b.half_skin2 = 0.25 * skin * skin;
    impl_->cellMode = b.nc[0] >= 3 && b.nc[1] >= 3 && b.nc[2] >= 3;
    impl_->ncell = b.nc[0] * b.nc[1] * b.nc[2];
    const size_t N = nParticle;
    impl_->cell.reset(sizeof(int) * N);
    impl_->count.reset(sizeof(int) * impl_->ncell);
    impl_->start.reset(sizeof(int) * (impl_->ncell + 1));
    impl_->cursor.reset(sizeof(int) * impl_->ncell);
    impl_->order.reset(sizeof(int) * N);
    impl_->nn.reset(sizeof(int) * N);
    impl_->nbr.reset(sizeof(int) * minim_amd::nbr_elems(N, impl_->maxn));
    impl_->flag.reset(sizeof(int));
    impl_->xbuild.reset(sizeof(double) * 3 * N);
  }
}

namespace {
// Lanes per particle of the force pass: as many as 512 blocks (two per CU) hold.
// One lane per particle leaves small systems waiting for a chain of 80 list
// entries (4,096 particles, FP64: 15.3 us with one lane, 5.0 with 16); where one
// fills the chip, more lanes only add their sums and unused entries (262,144,
// FP64: 53 us with one, 56 with two).
int cut_lanes(int N) {
  int p = 16;
  while (p > 1 && (size_t)N * p > 512 * (size_t)kBlock) p /= 2;
  return p;
}
int cut_blocks(int N) { return (int)(((size_t)N * cut_lanes(N) + kBlock - 1) / kBlock); }

template <typename T>
void launch_cut_t(LjNd::Impl& I, const T* x, const T* d, T t, int N, double sigma, double eps, double eshift, int mode,
                  T* g, minim_amd::RedScratch rs, hipStream_t s, const T* v) {
  if (d) {
    const size_t n = 3 * (size_t)N;
    if (I.xtrial.bytes() < n * sizeof(double)) I.xtrial.reset(n * sizeof(double));
    T* xt = static_cast<T*>(I.xtrial.get());
    minim_amd::lj_point_kernel<T><<<(int)((n + kBlock - 1) / kBlock), kBlock, 0, s>>>(x, d, t, n, xt);
    x = xt;
  }
  auto go = [&](auto lanes, auto unroll) {
    constexpr int P = decltype(lanes)::value, U = decltype(unroll)::value;
    auto run = [&](auto kernel) {
      kernel<<<cut_blocks(N), kBlock, 0, s>>>(x, N, I.box, (T)(sigma * sigma), eps, eshift, (const int*)I.nn.get(),
                                              (const int*)I.nbr.get(), I.maxn, (const double*)I.xbuild.get(),
                                              (const int*)I.flag.get(), v, g, rs);
    };
    if (v) run(minim_amd::lj_cut_kernel<T, P, U, 6>);
    else if (mode == 1) run(minim_amd::lj_cut_kernel<T, P, U, 1>);
    else if (mode == 2) run(minim_amd::lj_cut_kernel<T, P, U, 2>);
    else run(minim_amd::lj_cut_kernel<T, P, U, 3>);
  };
  using std::integral_constant;
  switch (cut_lanes(N)) {
    case 1: go(integral_constant<int, 1>(), integral_constant<int, 8>()); break;
    case 2: go(integral_constant<int, 2>(), integral_constant<int, 8>()); break;
    case 4: go(integral_constant<int, 4>(), integral_constant<int, 8>()); break;
    case 8: go(integral_constant<int, 8>(), integral_constant<int, 4>()); break;
    default: go(integral_constant<int, 16>(), integral_constant<int, 2>()); break;
  }
}

void launch_cut(LjNd::Impl& I, int prec, const void* x, const void* d, double t, int N, double sigma, double epsilon,
                double eshift, int mode, void* g, minim_amd::RedScratch rs, hipStream_t s, const void* v = nullptr) {
  if (prec == FP64)
    launch_cut_t(I, (const double*)x, (const double*)d, t, N, sigma, epsilon, eshift, mode, (double*)g, rs, s,
                 (const double*)v);
  else
    launch_cut_t(I, (const float*)x, (const float*)d, (float)t, N, sigma, epsilon, eshift, mode, (float*)g, rs, s,
                 (const float*)v);
  MINIM_HIP_CHECK(hipGetLastError());
}

// Lanes per particle of the list build: 16 while one wavefront per four
// particles leaves room, then 8 (whole rebuild with its evaluation at 4,096
// particles: 207 us with one lane, 102 with 8, 88 with 16; at 32,768: 215, 127,
// 131; at 262,144: 429, 385, 423).
int build_lanes(int N) { return N <= 16384 ? 16 : 8; }

// (Re)builds the Verlet list at the evaluated positions x (+ t*d), without
// waiting for it: the force pass reports a list that outgrew its rows (its
// reduction row after the moved particles), and grow_list makes room.
void rebuild_list(LjNd::Impl& I, int prec, const void* x, const void* d, double t, int N, hipStream_t s) {
  const int nb = (N + kBlock - 1) / kBlock;
  // Build at the evaluated positions: materialise x + t*d when needed.
  const void* xb = x;
  if (d) {
    if (I.xtrial.bytes() < 3 * sizeof(double) * (size_t)N) I.xtrial.reset(3 * sizeof(double) * (size_t)N);
    minim_amd::device_copy(I.xtrial.get(), x, 3 * (size_t)N * minim_amd::prec_bytes(prec), s);
    minim_amd::launch_axpy(prec, I.xtrial.get(), d, t, 3 * (size_t)N, s);
    xb = I.xtrial.get();
  }
  int* count = (int*)I.count.get();
  int* flag = (int*)I.flag.get();
  auto go = [&](auto tag) {
    using T = decltype(tag);
    const T* xx = (const T*)xb;
    double* xbuild = (double*)I.xbuild.get();
    if (I.cellMode) {
      constexpr int kCellsPerBlock = kBlock / minim_amd::kWave;  // one wavefront per cell
      const int nbc = (I.ncell + kCellsPerBlock - 1) / kCellsPerBlock;
      if (I.xcell.bytes() < sizeof(double4) * (size_t)N) I.xcell.reset(sizeof(double4) * (size_t)N);
      double4* xc = static_cast<double4*>(I.xcell.get());
      minim_amd::lj_clear_kernel<<<minim_amd::grid_blocks(I.ncell), kBlock, 0, s>>>(count, I.ncell, flag);
      minim_amd::lj_cell_index_kernel<T><<<nb, kBlock, 0, s>>>(xx, N, I.box, (int*)I.cell.get(), count, xbuild);
      minim_amd::lj_scan_kernel<<<1, kBlock, 0, s>>>(count, (int*)I.start.get(), (int*)I.cursor.get(), I.ncell);
      minim_amd::lj_fill_kernel<<<nb, kBlock, 0, s>>>((const int*)I.cell.get(), N, (const int*)I.start.get(),
                                                      (int*)I.cursor.get(), (int*)I.order.get());
      minim_amd::lj_sort_cells_kernel<T><<<nbc, kBlock, 0, s>>>(xx, I.box, (const int*)I.start.get(),
                                                                (const int*)I.order.get(), I.ncell, xc);
      auto build = [&](auto kernel, int lanes) {
        kernel<<<(int)(((size_t)N * lanes + kBlock - 1) / kBlock), kBlock, 0, s>>>(
            N, I.box, (const int*)I.cell.get(), (const int*)I.start.get(), xc, I.maxn, (int*)I.nn.get(),
            (int*)I.nbr.get(), flag);
      };
      if (build_lanes(N) == 16) build(minim_amd::lj_build_list_kernel<16>, 16);
      else build(minim_amd::lj_build_list_kernel<8>, 8);
    } else {
      minim_amd::lj_clear_kernel<<<1, kBlock, 0, s>>>(count, 0, flag);
      minim_amd::lj_build_list_brute_kernel<T><<<nb, kBlock, 0, s>>>(xx, N, I.box, I.maxn, (int*)I.nn.get(),
                                                                     (int*)I.nbr.get(), flag, xbuild);
    }
    MINIM_HIP_CHECK(hipGetLastError());
  };
  if (prec == FP64) go(0.0);
  else go(0.0f);
  I.built = true;
  I.builds++;
}

// Rows for lists of up to longest entries; the list is built again after.  Where
// the memory does not suffice (an exception), there are no rows and no list: the
// next evaluation builds one that outgrows them, and comes here again.
void grow_list(LjNd::Impl& I, int N, int longest) {
  const int maxn = (longest + 2 * minim_amd::kListPad - 1) / minim_amd::kListPad * minim_amd::kListPad;
  I.built = false;
  I.maxn = 0;
  I.nbr.reset(sizeof(int) * minim_amd::nbr_elems(N, maxn));
  I.maxn = maxn;
  I.builds--;
}

// rebuild_list, waiting until it is known that the lists fit.
void rebuild_list_checked(LjNd::Impl& I, int prec, const void* x, int N, hipStream_t s) {
  for (;;) {
    rebuild_list(I, prec, x, nullptr, 0.0, N, s);
    int over = 0;
    MINIM_HIP_CHECK(hipMemcpyAsync(&over, I.flag.get(), sizeof(int), hipMemcpyDeviceToHost, s));
    MINIM_HIP_CHECK(hipStreamSynchronize(s));
    if (over == 0) return;
    grow_list(I, N, over);
  }
}

}  // namespace

// Energy (result slot 0, and eDev when given) and gradient, without waiting for
// them: except in cutoff mode, where the list check is read.
void LjNd::launch(int prec, const void* x, const void* d, double t, bool wantE, double* eDev, void* g,
                  void* stream) const {
  if (!impl_) throw std::runtime_error("LjNd: not initialised (construct a State first).");
  hipStream_t s = static_cast<hipStream_t>(stream);
  auto& ws = minim_amd::Workspace::current();
  const int mode = (wantE ? 1 : 0) | (g ? 2 : 0);
  const int N = nParticle;
  if (cutoff <= 0) {
    if (prec == FP64) minim_amd::launch_allpairs<double>(nDim, x, d, t, N, sigma, epsilon, mode, g, ws.rs(), s, eDev);
    else minim_amd::launch_allpairs<float>(nDim, x, d, t, N, sigma, epsilon, mode, g, ws.rs(), s, eDev);
  } else {
    Impl& I = *impl_;
    if (cut_blocks(N) > minim_amd::kMaxRedBlocks)
      throw std::invalid_argument("LjNd: too many particles for one launch");
    const double src6 = std::pow(sigma / cutoff, 6);
    const double eshift = 4 * epsilon * (src6 * src6 - src6);
    bool build = !I.built;
    for (;;) {
      if (build) rebuild_list(I, prec, x, d, t, N, s);
      const minim_amd::RedScratch rs = ws.rs().copying(0, wantE ? eDev : nullptr);
      launch_cut(I, prec, x, d, t, N, sigma, epsilon, eshift, mode, g, rs, s);
      minim_amd::launch_finalize(rs, 3, cut_blocks(N), s);
      double r[3];  // energy, particles moved more than skin/2 since the list was built, its overflow
      ws.fetch(s, 3, r);
      if (r[1] == 0 && r[2] == 0) break;
      if (r[2] > 0) grow_list(I, N, (int)r[2]);
      build = true;
    }
  }
  if (g) constrainDevice(prec, x, g, (size_t)N * nDim, stream);
}

void LjNd::evaluate(int prec, const void* x, const void* d, double t, double* e, void* g, void* stream) const {
  if (!impl_) throw std::runtime_error("LjNd: not initialised (construct a State first).");
  if (!e && !g) return;
  launch(prec, x, d, t, e != nullptr, nullptr, g, stream);
  if (e) {
    double r[1];
    minim_amd::Workspace::current().fetch(static_cast<hipStream_t>(stream), 1, r);
    *e = r[0];
  }
}

// A class derived from these may have its own evaluate or constraints, which the
// general paths call.
bool LjNd::plain() const {
  return typeid(*this) == typeid(LjNd) || typeid(*this) == typeid(Lj2d) || typeid(*this) == typeid(Lj3d);
}

void LjNd::evaluateAsync(int prec, const void* x, const void* d, double t, bool wantE, double* e_dev, void* g,
                         void* stream) const {
  if (!plain()) return Potential::evaluateAsync(prec, x, d, t, wantE, e_dev, g, stream);
  if (!impl_) throw std::runtime_error("LjNd: not initialised (construct a State first).");
  if (wantE || g) launch(prec, x, d, t, wantE, e_dev, g, stream);
}

// Cutoff mode: the force pass without the host synchronisation of the list
// check; the moved-particle count goes to the result slot returned.
int LjNd::gradientDeferred(int prec, const void* x, void* g, void* stream) const {
  if (!impl_) throw std::runtime_error("LjNd: not initialised (construct a State first).");
  if (cutoff <= 0) return Potential::gradientDeferred(prec, x, g, stream);
  hipStream_t s = static_cast<hipStream_t>(stream);
  auto& ws = minim_amd::Workspace::current();
  Impl& I = *impl_;
  const int N = nParticle;
  if (!I.built) rebuild_list_checked(I, prec, x, N, s);
  const double src6 = std::pow(sigma / cutoff, 6);
  const double eshift = 4 * epsilon * (src6 * src6 - src6);
  minim_amd::RedScratch rs = ws.rs();
  rs = rs.copying(1, rs.mirror + minim_amd::kDeferSlot);
  launch_cut(I, prec, x, nullptr, 0.0, N, sigma, epsilon, eshift, 2, g, rs, s);
  minim_amd::launch_finalize(rs, 3, cut_blocks(N), s);
  constrainDevice(prec, x, g, (size_t)N * nDim, stream);
  return minim_amd::kDeferSlot;
}

void LjNd::redoGradient(int prec, const void* x, void* g, void* stream) const {
  if (!impl_) throw std::runtime_error("LjNd: not initialised (construct a State first).");
  if (cutoff <= 0) return Potential::redoGradient(prec, x, g, stream);
  hipStream_t s = static_cast<hipStream_t>(stream);
  auto& ws = minim_amd::Workspace::current();
  const int N = nParticle;
  rebuild_list_checked(*impl_, prec, x, N, s);
  const double src6 = std::pow(sigma / cutoff, 6);
  const double eshift = 4 * epsilon * (src6 * src6 - src6);
  const minim_amd::RedScratch rs = ws.rs();
  launch_cut(*impl_, prec, x, nullptr, 0.0, N, sigma, epsilon, eshift, 2, g, rs, s);
  minim_amd::launch_finalize(rs, 3, cut_blocks(N), s);
  constrainDevice(prec, x, g, (size_t)N * nDim, stream);
}

// Cutoff mode without constraints: the force pass has each particle's force in
// registers, so that FIRE's dots and largest force need no pass of their own.
bool LjNd::fusesFire(int dim) const {
  return plain() && cutoff > 0 && constraints.empty() && (dim == 0 || dim == 3) &&
         cut_blocks(nParticle) <= minim_amd::kMaxRedBlocks;
}

void LjNd::fireGradient(int prec, const void* x, void* g, const void* v, int, bool again, void* stream) const {
  if (!impl_) throw std::runtime_error("LjNd: not initialised (construct a State first).");
  hipStream_t s = static_cast<hipStream_t>(stream);
  auto& ws = minim_amd::Workspace::current();
  Impl& I = *impl_;
  const int N = nParticle;
  if (again) {
    // a list that was built for the last evaluation may have outgrown its rows
    double r[5];
    ws.fetch(s, 5, r);
    if (r[4] > 0) grow_list(I, N, (int)r[4]);
  }
  if (again || !I.built) rebuild_list(I, prec, x, nullptr, 0.0, N, s);
  const minim_amd::RedScratch rs = ws.rs();
  launch_cut(I, prec, x, nullptr, 0.0, N, sigma, epsilon, 0.0, 2, g, rs, s, v);
  minim_amd::launch_finalize(rs, 6, cut_blocks(N), s, 5);
}

// Average duration (ms) of reps launches of the force kernel (cutoff mode:
// the list is built first when it does not exist yet; all-pairs mode: the
// kernel and its reduction).
double LjNd::componentEnergy(int component, const vector<double>& coords) const {
  return component == 0 ? energy(coords) : 0.0;
}

double LjNd::timeKernel(int prec, const void* x, bool wantE, void* g, int reps, void* stream) const {
  if (!impl_) throw std::runtime_error("LjNd: not initialised (construct a State first).");
  const int mode = (wantE ? 1 : 0) | (g ? 2 : 0);
  if (mode == 0 || reps < 1) throw std::invalid_argument("LjNd: nothing to time");
  hipStream_t s = static_cast<hipStream_t>(stream);
  auto& ws = minim_amd::Workspace::current();
  const int N = nParticle;
  const double src6 = cutoff > 0 ? std::pow(sigma / cutoff, 6) : 0.0;
  const double eshift = 4 * epsilon * (src6 * src6 - src6);
  auto launch = [&]() {
    if (cutoff > 0) {
      launch_cut(*impl_, prec, x, nullptr, 0.0, N, sigma, epsilon, eshift, mode, g, ws.rs(), s);
    } else if (prec == FP64) {
      minim_amd::launch_allpairs<double>(nDim, x, nullptr, 0.0, N, sigma, epsilon, mode, g, ws.rs(), s);
    } else {
      minim_amd::launch_allpairs<float>(nDim, x, nullptr, 0.0, N, sigma, epsilon, mode, g, ws.rs(), s);
    }
  };
  if (cutoff > 0 && !impl_->built) rebuild_list_checked(*impl_, prec, x, N, s);
  launch();
  hipEvent_t e0, e1;
  MINIM_HIP_CHECK(hipEventCreate(&e0));
  MINIM_HIP_CHECK(hipEventCreate(&e1));
  MINIM_HIP_CHECK(hipEventRecord(e0, s));
  for (int i = 0; i < reps; i++) launch();
  MINIM_HIP_CHECK(hipEventRecord(e1, s));
  MINIM_HIP_CHECK(hipEventSynchronize(e1));
  float ms = 0;
  MINIM_HIP_CHECK(hipEventElapsedTime(&ms, e0, e1));
  MINIM_HIP_CHECK(hipEventDestroy(e0));
  MINIM_HIP_CHECK(hipEventDestroy(e1));
  return (double)ms / reps;
}

}  // namespace minim
