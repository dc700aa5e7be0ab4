// pfu.hip -- the element form of the phase field (PhaseFieldUnstructured,
// src/potentials/PhaseFieldUnstructured.cpp) on MI355X (gfx950).
//
// The reference evaluates a list of elements one after another
// (State::elementEG, src/State.cpp:58-79): a seven-site gradient element per
// site and fluid (or per site for the "fixed" density mode, whose last fluid
// is implicit), one-DOF pressure, surface, force and confinement elements and
// a soft-density element per site, then the volume term over the whole field
// (blockEnergyGradient, :280-308).  Two forms here, chosen by init:
//
//  * gathered per site (pfu_site_kernel) when the list holds nothing but fluid,
//    pressure and three-fluid soft-density elements: one thread per site adds
//    the seven-site elements that its site is part of, so nothing is read but
//    the concentrations (and a 4-byte code per site next to solid nodes);
//  * the list itself (pfu_chunk_kernel) otherwise: the host groups the elements
//    into chunks of nearby sites; a block takes one chunk at a time, one thread
//    per element, accumulates the energy in FP64 for a deterministic two-stage
//    reduction and the gradient contributions in an FP64 LDS accumulator
//    (ds_add_f64), then stores the gradient of every site only its chunk touches
//    and writes the partial sums of the sites other chunks also touch to a
//    scratch slot; a second pass sums those partials per site in chunk order.
//    No global atomics; the LDS adds of one chunk land in the order its threads
//    reach them, so the gradient's last bits may vary from launch to launch.
//
// Each element keeps the reference's formula, including its choices.
#include "common.hpp"
#include "pf_tile.hpp"
#include "pfu.hpp"

namespace minim_amd {

namespace {

template <typename T, typename TV, bool DIR>
struct Coords {
  const T* __restrict__ x;
  const TV* __restrict__ d;
  T t;
  __device__ __forceinline__ T operator()(int i) const {
    T c = x[i];
    if constexpr (DIR) {
      const T s = t * (T)d[i];
      c = c + s;
    }
    return c;
  }
};

// The gradient term of one seven-site element (phaseGradient,
// PhaseFieldUnstructured.cpp:311-515): node 0 is the site, nodes (1,6), (2,5),
// (3,4) its x, y, z neighbours; self[i] marks a neighbour that is the site
// itself (the reference's stand-in for a solid neighbour).  Contributions to
// the nodes' gradients go to gl.
template <typename T, bool WE, bool WG>
__device__ __forceinline__ void phase7(const T (&c)[kPFUNodes], const bool (&self)[kPFUNodes], T factor, T& e,
                                       T (&gl)[kPFUNodes]) {
  const int mp[3][2] = {{1, 6}, {2, 5}, {3, 4}};
  T grad2 = (T)0;
#pragma unroll
  for (int d = 0; d < 3; d++) {
    const int m = mp[d][0], p = mp[d][1];
    if (!self[m] && !self[p]) {
      const T gm = c[0] - c[m], gp = c[0] - c[p];
      if (WE) grad2 = grad2 + (T)0.5 * (gm * gm + gp * gp);
      if (WG) {
        gl[0] = gl[0] + factor * (gm + gp);
        gl[m] = gl[m] - factor * gm;
        gl[p] = gl[p] - factor * gp;
      }
    } else if (!self[p]) {
      const T gp = c[0] - c[p];
      if (WE) grad2 = grad2 + gp * gp;
      if (WG) {
        gl[0] = gl[0] + (factor * (T)2) * gp;
        gl[p] = gl[p] - (factor * (T)2) * gp;
      }
    } else if (!self[m]) {
      const T gm = c[0] - c[m];
      if (WE) grad2 = grad2 + gm * gm;
      if (WG) {
        gl[0] = gl[0] + (factor * (T)2) * gm;
        gl[m] = gl[m] - (factor * (T)2) * gm;
      }
    }
  }
  if (WE) e = e + factor * grad2;
}

// MODE bits: 1 = energy, 2 = gradient, 4 = at x + t*d.  NF: the fluid count
// when it is 1..4 (index arithmetic with constants), 0 for u.nf.
template <typename T, typename TV, int MODE, int NF>
__global__ __launch_bounds__(kBlock) void pfu_chunk_kernel(PFUArgs u, const T* __restrict__ x,
                                                           const TV* __restrict__ d, T t, TV* __restrict__ g,
                                                           RedScratch rs) {
  constexpr bool WE = MODE & 1, WG = MODE & 2, DIR = MODE & 4;
  __shared__ uint32_t ssite[kPFUChunkDofs];
  __shared__ double sacc[WG ? kPFUChunkDofs : 1];
  const Coords<T, TV, DIR> cx{x, d, t};
  const int nf = NF > 0 ? NF : u.nf;
  // gradient contribution v to fluid k of local site l
  auto add = [&](int l, int k, T v) {
    if (WG && v != (T)0) unsafeAtomicAdd(&sacc[l * nf + k], (double)v);
  };
  auto gsite = [&](int l) { return (int)(ssite[l] & ~kPFUShared); };
  double acc[2] = {0.0, 0.0};
  for (int c = blockIdx.x; c < u.nchunk; c += gridDim.x) {
    const uint32_t s0 = u.chunk_site[c];
    const int ns = (int)(u.chunk_site[c + 1] - s0);
    for (int i = threadIdx.x; i < ns; i += kBlock) ssite[i] = u.sites[s0 + i];
    if (WG)
      for (int i = threadIdx.x; i < ns * nf; i += kBlock) sacc[i] = 0.0;
    __syncthreads();
    const uint32_t e1 = u.chunk_el[c + 1];
    for (uint32_t ie = u.chunk_el[c] + threadIdx.x; ie < e1; ie += kBlock) {
      const uint4 r = u.rec[ie];
      const int loc[kPFUNodes] = {(int)(r.x & 0xffffu), (int)(r.x >> 16), (int)(r.y & 0xffffu), (int)(r.y >> 16),
                                  (int)(r.z & 0xffffu), (int)(r.z >> 16), (int)(r.w & 0xffffu)};
      const int type = (int)((r.w >> 16) & 0xffu), f = (int)(r.w >> 24);
      const int site0 = gsite(loc[0]);
      T e = (T)0;
      switch (type) {
        case kPFUFluid: {  // fluidEnergy (:518-538)
          const T vol = (T)u.node_vol[site0];
          T c[kPFUNodes], gl[kPFUNodes];
          bool self[kPFUNodes];
#pragma unroll
          for (int i = 0; i < kPFUNodes; i++) {
            c[i] = cx(gsite(loc[i]) * nf + f);
            gl[i] = (T)0;
            self[i] = (i > 0) && loc[i] == loc[0];
          }
          const T c0 = c[0];
          if (nf == 1) {
            const T factor = ((T)u.kappa[0] / (T)16) * vol;
            if (WE) e = e + (factor * ((c0 + (T)1) * (c0 + (T)1))) * ((c0 - (T)1) * (c0 - (T)1));
            if (WG) gl[0] = gl[0] + ((factor * (T)4) * c0) * (c0 * c0 - (T)1);
          } else {
            const T factor = ((T)0.5 * (T)u.kappa[f]) * vol;
            if (WE) e = e + (factor * (c0 * c0)) * ((c0 - (T)1) * (c0 - (T)1));
            if (WG) gl[0] = gl[0] + (((factor * (T)2) * c0) * (c0 - (T)1)) * ((T)2 * c0 - (T)1);
          }
          T gfac = (nf == 1) ? ((T)0.25 * (T)u.kappaP[0]) * vol : ((T)0.5 * (T)u.kappaP[f]) * vol;
          gfac = gfac / (T)u.res2;
          phase7<T, WE, WG>(c, self, gfac, e, gl);
#pragma unroll
          for (int i = 0; i < kPFUNodes; i++) add(loc[i], f, gl[i]);
          break;
        }
        case kPFUFluidAll: {  // fluidEnergyAll (:541-586): the last fluid is 1 - the others
          const T vol = (T)u.node_vol[site0];
          int sn[kPFUNodes];
          T cN[kPFUNodes], gN[kPFUNodes];
          bool none[kPFUNodes];
#pragma unroll
          for (int i = 0; i < kPFUNodes; i++) {
            sn[i] = gsite(loc[i]) * nf;
            cN[i] = (T)1;
            gN[i] = (T)0;
            none[i] = false;  // the reference passes distinct indices here: no node counts as solid
          }
          for (int k = 0; k < nf - 1; k++)
#pragma unroll
            for (int i = 0; i < kPFUNodes; i++) cN[i] = cN[i] - cx(sn[i] + k);
          const T bfN = ((T)0.5 * (T)u.kappa[nf - 1]) * vol;
          const T gfN = ((T)0.5 * (T)u.kappaP[nf - 1]) * vol;  // not divided by res^2 (:555)
          if (WE) e = e + (bfN * (cN[0] * cN[0])) * ((cN[0] - (T)1) * (cN[0] - (T)1));
          if (WG) gN[0] = gN[0] + (((bfN * (T)2) * cN[0]) * (cN[0] - (T)1)) * ((T)2 * cN[0] - (T)1);
          phase7<T, WE, WG>(cN, none, gfN, e, gN);
          for (int k = 0; k < nf - 1; k++) {
            T c[kPFUNodes], gl[kPFUNodes];
            bool self[kPFUNodes];
#pragma unroll
            for (int i = 0; i < kPFUNodes; i++) {
              c[i] = cx(sn[i] + k);
              gl[i] = (T)0;
              self[i] = (i > 0) && loc[i] == loc[0];
            }
            const T c0 = c[0];
            const T bf = ((T)0.5 * (T)u.kappa[k]) * vol;
            if (WE) e = e + (bf * (c0 * c0)) * ((c0 - (T)1) * (c0 - (T)1));
            if (WG) gl[0] = gl[0] + (((bf * (T)2) * c0) * (c0 - (T)1)) * ((T)2 * c0 - (T)1);
            T gf = ((T)0.5 * (T)u.kappaP[k]) * vol;
            gf = gf / (T)u.res2;
            phase7<T, WE, WG>(c, self, gf, e, gl);
#pragma unroll
            for (int i = 0; i < kPFUNodes; i++) add(loc[i], k, gl[i] - gN[i]);
          }
          break;
        }
        case kPFUPressure: {  // pressureEnergy (:613-628)
          const T pr = (T)u.pressure[f];
          const T v = (T)u.node_vol[site0];
          const T c = cx(site0 * nf + f);
          if (nf == 1) {
            if (WE) e = e - pr * (((T)0.5 * (c + (T)1)) * v);
            add(loc[0], f, -(((T)0.5 * pr) * v));
          } else {
            if (WE) e = e - pr * (c * v);
            add(loc[0], f, -(pr * v));
          }
          break;
        }
        case kPFUDensity: {  // densityConstraintEnergy (:631-642): three DOFs of the site
          if (nf == 1) break;
          const T coef = (T)u.coef_density;
          const T rho = ((cx(site0 * nf) + cx(site0 * nf + 1)) + cx(site0 * nf + 2)) - (T)1;
          if (WE) e = e + coef * (rho * rho);
          const T gr = ((T)2 * coef) * rho;
          add(loc[0], 0, gr);
          add(loc[0], 1, gr);
          add(loc[0], 2, gr);
          break;
        }
        case kPFUSurface: {  // surfaceEnergy (:645-654): binary fluids only
          if (nf != 1) break;
          const double* p = u.par + 3 * (size_t)u.pidx[ie];
          const T area = (T)p[0], w = (T)p[1];
          const T phi = cx(site0 * nf + f);
          if (WE) e = e + (w * ((((phi * phi) * phi) / (T)3 - phi) - (T)2 / (T)3)) * area;
          add(loc[0], f, (w * (phi * phi - (T)1)) * area);
          break;
        }
        case kPFUForce: {  // forceEnergy (:657-676)
          const T c = (nf == 1) ? (T)0.5 * ((T)1 + cx(site0 * nf + f)) : cx(site0 * nf + f);
          if (c < (T)0.01) break;
          const double* p = u.par + 3 * (size_t)u.pidx[ie];
          const T vol = (T)p[0], fm = (T)p[1], h = (T)p[2];
          if (WE) e = e + ((c * vol) * fm) * h;
          add(loc[0], f, (nf == 1) ? ((((T)0.5 * vol) * fm) * h) : ((vol * fm) * h));
          break;
        }
        case kPFUConfinement: {  // ffConfinementEnergy (:679-692)
          const T c = cx(site0 * nf + f);
          const double* p = u.par + 3 * (size_t)u.pidx[ie];
          const T coef = ((T)p[0] * (T)u.st_mean) * (T)u.res2;
          const T c0 = (T)p[1];
          if ((c0 - (T)0.5) * (c - (T)0.5) < (T)0) {
            if (WE) e = e + coef * ((c - (T)0.5) * (c - (T)0.5));
            add(loc[0], f, (coef * (T)2) * (c - (T)0.5));
          }
          break;
        }
        default:
          break;
      }
      if (WE) acc[0] += (double)e;
    }
    __syncthreads();
    if (WG) {
      // sites only this chunk touches: the gradient; the others: partials
      TV* __restrict__ part = static_cast<TV*>(u.scratch) + (size_t)s0 * nf;
      for (int i = threadIdx.x; i < ns * nf; i += kBlock) {
        const int l = i / nf;
        const uint32_t en = ssite[l];
        const TV v = (TV)sacc[i];
        if (en & kPFUShared)
          part[i] = v;
        else
          g[(size_t)(en & ~kPFUShared) * nf + (i - l * nf)] = v;
      }
      __syncthreads();
    }
  }
  grid_sum_store<2>(acc, rs);
}

// The gradient of the sites that are not exclusive to one chunk: the sum of
// their partials in chunk order (zero for a site no element touches).
template <typename T>
__global__ __launch_bounds__(kBlock) void pfu_gather_kernel(PFUArgs u, T* __restrict__ g) {
  const int nf = u.nf;
  const T* __restrict__ part = static_cast<const T*>(u.scratch);
  const size_t n = u.ngather * nf;
  for (size_t i = (size_t)blockIdx.x * kBlock + threadIdx.x; i < n; i += (size_t)gridDim.x * kBlock) {
    const size_t j = i / nf;
    const int k = (int)(i - j * nf);
    const uint32_t p0 = u.gpos_off[j], p1 = u.gpos_off[j + 1];
    double sum = 0.0;
    for (uint32_t p = p0; p < p1; p++) sum += (double)part[(size_t)u.gpos[p] * nf + k];
    g[(size_t)u.gsite[j] * nf + k] = (T)sum;
  }
}

// ---------------------------------------------------------------- per-site form
template <typename T, int N>
struct SiteVec {
  T v[N];
};

// Concentrations (x, or x + t*d) and codes of the R own rows and the halo site
// of one x plane.
template <typename T, int NF, int R, bool SOLID>
struct SitePlane {
  T x[R][NF];
  T hx[NF];
  unsigned q[SOLID ? R : 1];
  unsigned hq;
};

template <typename T, int NF, int R, bool SOLID, bool DIR>
__device__ __forceinline__ void load_site_plane(const PFUArgs& u, size_t pl, const T* __restrict__ x,
                                                const T* __restrict__ d, T t, const TileThread& th,
                                                SitePlane<T, NF, R, SOLID>& p) {
  auto one = [&](unsigned site, T(&v)[NF]) {
    const unsigned off = site * (unsigned)(NF * sizeof(T));
    const char* xb = reinterpret_cast<const char*>(x + pl * NF);
    const SiteVec<T, NF> xv = *reinterpret_cast<const SiteVec<T, NF>*>(xb + off);
#pragma unroll
    for (int k = 0; k < NF; k++) v[k] = xv.v[k];
    if constexpr (DIR) {
      const char* db = reinterpret_cast<const char*>(d + pl * NF);
      const SiteVec<T, NF> dv = *reinterpret_cast<const SiteVec<T, NF>*>(db + off);
#pragma unroll
      for (int k = 0; k < NF; k++) {
        const T st = t * dv.v[k];
        v[k] = v[k] + st;
      }
    }
  };
#pragma unroll
  for (int r = 0; r < R; r++) one(th.site[r], p.x[r]);
  one(th.hsite, p.hx);
  if constexpr (SOLID) {
    const uint32_t* qp = u.wcode + pl;
#pragma unroll
    for (int r = 0; r < R; r++) p.q[r] = qp[th.site[r]];
    p.hq = qp[th.hsite];
  }
}

// Weight of the bond to the plus neighbour along canonical dimension j.
template <typename T>
__device__ __forceinline__ T bond_w(unsigned q, int j) {
  return (T)((q >> (kPFWeightShift + kPFWeightBits * j)) & ((1u << kPFWeightBits) - 1u)) * (T)0.0625;
}

// One site: the energy of its own elements (each bond's two halves counted at
// its minus end), and its gradient, to which every seven-site element that
// contains it contributes: for a bond (i, j) the elements of both ends give
// 2 f w (c_i - c_j), with w = (v_i h_i->j + v_j h_j->i) / res^3 (1 away from
// solid nodes).  The contributions are added in FP64 in either precision, as
// the list form's accumulator does, and the projection is applied before the
// one rounding.  Bonds of weight zero do not read the other site's value (a
// solid site may hold anything).
template <typename T, int NF, bool WE, bool WG, bool SOLID>
__device__ __forceinline__ void site_elements(const PFUArgs& u, const PFArgs& con, const T (&c)[NF],
                                              const T (&xm)[NF], const T (&xp)[NF], const T (&ym)[NF],
                                              const T (&yp)[NF], const T (&zm)[NF], const T (&zp)[NF], unsigned qc,
                                              unsigned qxm, unsigned qym, unsigned qzm, double& ea,
                                              double (&g)[NF]) {
  const int kind = (int)(qc & 15u);
  const T vc = !SOLID ? (T)1 : kind >= 2 ? (T)(kind - 1) * (T)0.125 : (T)kind;
  const bool fluid = !SOLID || kind != 0;
  const T wf[3] = {SOLID ? bond_w<T>(qc, 0) : (T)1, SOLID ? bond_w<T>(qc, 1) : (T)1,
                   SOLID ? bond_w<T>(qc, 2) : (T)1};
  const T wb[3] = {SOLID ? bond_w<T>(qxm, 0) : (T)1, SOLID ? bond_w<T>(qym, 1) : (T)1,
                   SOLID ? bond_w<T>(qzm, 2) : (T)1};
#pragma unroll
  for (int k = 0; k < NF; k++) {
    const T ck = c[k];
    T dm[3] = {ck - xm[k], ck - ym[k], ck - zm[k]};
    T dp[3] = {ck - xp[k], ck - yp[k], ck - zp[k]};
    if constexpr (SOLID) {
#pragma unroll
      for (int j = 0; j < 3; j++) {
        dm[j] = wb[j] == (T)0 ? (T)0 : dm[j];
        dp[j] = wf[j] == (T)0 ? (T)0 : dp[j];
      }
    }
    const T a2 = ck - (T)1;
    if (WE && fluid) {
      // fluidEnergy (:518-538) and the halves of phaseGradient's squares
      T sq = (T)0;
#pragma unroll
      for (int j = 0; j < 3; j++) sq = fma(SOLID ? wf[j] * dp[j] : dp[j], dp[j], sq);
      T e;
      if (NF == 1) {
        const T a1 = ck + (T)1;
        e = ((T)u.fb[k] * vc) * ((a1 * a1) * (a2 * a2));
      } else {
        e = ((T)u.fb[k] * vc) * ((ck * ck) * (a2 * a2));
      }
      e = fma((T)u.fg[k], sq, e);
      const T pr = (T)u.pressure[k];  // pressureEnergy (:613-628)
      if (pr != (T)0) e = e - pr * ((NF == 1 ? (T)0.5 * (ck + (T)1) : ck) * (vc * (T)u.v1));
      ea += (double)e;
    }
    if (WG) {
      double lap = 0.0;
#pragma unroll
      for (int j = 0; j < 3; j++) {
        lap = SOLID ? fma((double)wb[j], (double)dm[j], lap) : lap + (double)dm[j];
        lap = SOLID ? fma((double)wf[j], (double)dp[j], lap) : lap + (double)dp[j];
      }
      T bg;
      if (NF == 1) bg = (((T)4 * (T)u.fb[k]) * vc) * (ck * fma(ck, ck, (T)-1));
      else bg = (((T)2 * (T)u.fb[k]) * vc) * ((ck * a2) * fma((T)2, ck, (T)-1));
      double gk = fma(2.0 * u.fg[k], lap, (double)bg);
      const double pr = u.pressure[k];
      if (pr != 0.0) gk -= (NF == 1 ? 0.5 * pr : pr) * ((double)vc * u.v1);
      g[k] = fluid ? gk : 0.0;
    }
  }
  if constexpr (NF == 3) {
    if (u.soft && fluid) {  // densityConstraintEnergy (:631-642)
      const T rho = ((c[0] + c[1]) + c[2]) - (T)1;
      const T coef = (T)u.coef_density;
      if (WE) ea += (double)(coef * (rho * rho));
      if (WG) {
        const T gr = ((T)2 * coef) * rho;
#pragma unroll
        for (int k = 0; k < NF; k++) g[k] += (double)gr;
      }
    }
  }
  if (WG) {
    // fixed fluids zeroed, then the mean of the variable ones removed
    if (con.fixmask) {
#pragma unroll
      for (int k = 0; k < NF; k++)
        if (con.fixmask & (1u << k)) g[k] = 0.0;
    }
    if (NF > 1 && con.density == kDensityHard && con.nvar > 0) {
      double comp = g[0];
#pragma unroll
      for (int k = 1; k < NF; k++) comp += g[k];
      comp *= con.inv_nvar;
#pragma unroll
      for (int k = 0; k < NF; k++)
        if (!(con.fixmask & (1u << k))) g[k] -= comp;
    }
  }
}

// The grid form's decomposition (pf_tile.hpp): a block streams the x planes of
// a 64 x 4R (z, y) tile through a two-plane LDS ring, the loads of plane i+2
// in flight while plane i is computed; own columns and x neighbours stay in
// registers.  Bound by memory: 128x112x120x3, energy and gradient with the
// reduction, FP64 21.1 us = 3.9 TB/s of concentrations in and gradient out,
// FP32 16.4 us; the list form, which reads 16 bytes and issues some 200
// instructions per element, took 156 and 130 us there.  Gradient error against
// 64 bits 1.53e-16 (list 1.59e-16) and 2.8e-8 in FP32 (list 5.5e-8).
// MODE bits: 1 = energy, 2 = gradient, 4 = at x + t*d.
template <typename T, int NF, int MODE, int R, bool SOLID>
__global__ __launch_bounds__(kBlock) void pfu_site_kernel(PFUArgs u, PFArgs con, TileGeom G,
                                                          const T* __restrict__ x, const T* __restrict__ d, T t,
                                                          T* __restrict__ g, RedScratch rs) {
  constexpr bool WE = MODE & 1, WG = MODE & 2, DIR = MODE & 4;
  constexpr int LH = kTileWaves * R + 2, LW = kTileZ + 2;
  using Plane = SitePlane<T, NF, R, SOLID>;
  __shared__ T lds[2][LH][LW][NF];
  __shared__ unsigned lq[SOLID ? 2 : 1][SOLID ? LH : 1][SOLID ? LW : 1];

  TileThread th;
  tile_thread(G, xcd_logical_block(blockIdx.x, gridDim.x), threadIdx.x, th);
  const size_t YZ = (size_t)G.Y * G.Z;
  const int X = G.X, x0 = th.x0, x1 = th.x1;
  const bool halo = th.hrow >= 0;
  auto load = [&](int plane, Plane& p) {
    load_site_plane<T, NF, R, SOLID, DIR>(u, (size_t)tile_plane(plane, X) * YZ, x, d, t, th, p);
  };
  auto fill = [&](int b, const Plane& p) {
#pragma unroll
    for (int r = 0; r < R; r++) {
#pragma unroll
      for (int k = 0; k < NF; k++) lds[b][th.lrow0 + r][th.lcol][k] = p.x[r][k];
      if constexpr (SOLID) lq[b][th.lrow0 + r][th.lcol] = p.q[r];
    }
    if (halo) {
#pragma unroll
      for (int k = 0; k < NF; k++) lds[b][th.hrow][th.hcol][k] = p.hx[k];
      if constexpr (SOLID) lq[b][th.hrow][th.hcol] = p.hq;
    }
  };

  T A[R][NF], B[R][NF], Cn[R][NF];  // planes i-1, i, i+1 of the own rows
  unsigned qA[R], qB[R], qC[R];
#pragma unroll
  for (int r = 0; r < R; r++) qA[r] = qB[r] = qC[r] = 0;
  {
    Plane pm, p0, p1;
    load(x0 - 1, pm);
    load(x0, p0);
    load(x0 + 1, p1);
#pragma unroll
    for (int r = 0; r < R; r++) {
#pragma unroll
      for (int k = 0; k < NF; k++) {
        A[r][k] = pm.x[r][k];
        B[r][k] = p0.x[r][k];
        Cn[r][k] = p1.x[r][k];
      }
      if constexpr (SOLID) {
        qA[r] = pm.q[r];
        qB[r] = p0.q[r];
        qC[r] = p1.q[r];
      }
    }
    fill(0, p0);
    fill(1, p1);
  }
  __syncthreads();

  double acc[1] = {0.0};
#pragma nounroll
  for (int i = x0; i < x1; i++) {
    const int b = (i - x0) & 1;
    const bool more = i + 1 < x1;  // the chunk's last plane needs no further one
    Plane q;
    if (more) load(i + 2, q);
    T* gp = g + (size_t)i * YZ * NF;
#pragma unroll
    for (int r = 0; r < R; r++) {
      T ym[NF], yp[NF], zm[NF], zp[NF];
#pragma unroll
      for (int k = 0; k < NF; k++) {
        ym[k] = (r > 0) ? B[r > 0 ? r - 1 : 0][k] : lds[b][th.lrow0 + r - 1][th.lcol][k];
        yp[k] = (r < R - 1) ? B[r < R - 1 ? r + 1 : 0][k] : lds[b][th.lrow0 + r + 1][th.lcol][k];
        zm[k] = lds[b][th.lrow0 + r][th.lcol - 1][k];
        zp[k] = lds[b][th.lrow0 + r][th.lcol + 1][k];
      }
      unsigned qym = 0, qzm = 0;
      if constexpr (SOLID) {
        qym = (r > 0) ? qB[r > 0 ? r - 1 : 0] : lq[b][th.lrow0 + r - 1][th.lcol];
        qzm = lq[b][th.lrow0 + r][th.lcol - 1];
      }
      double es = 0.0, gv[NF];
      site_elements<T, NF, WE, WG, SOLID>(u, con, B[r], A[r], Cn[r], ym, yp, zm, zp, qB[r], qA[r], qym, qzm, es, gv);
      if (th.own & (1u << r)) {
        if (WE) acc[0] += es;
        if (WG) {
          T* gs = gp + (size_t)th.site[r] * NF;  // streaming stores: not re-read here
#pragma unroll
          for (int k = 0; k < NF; k++) __builtin_nontemporal_store((T)gv[k], gs + k);
        }
      }
    }
    if (!more) break;
    lds_barrier();  // every wave is done reading buffer b
    fill(b, q);
#pragma unroll
    for (int r = 0; r < R; r++) {
#pragma unroll
      for (int k = 0; k < NF; k++) {
        A[r][k] = B[r][k];
        B[r][k] = Cn[r][k];
        Cn[r][k] = q.x[r][k];
      }
      if constexpr (SOLID) {
        qA[r] = qB[r];
        qB[r] = qC[r];
        qC[r] = q.q[r];
      }
    }
  }
  grid_sum_store<1>(acc, rs);
}

// Rows per thread: three plane copies of the own rows and the plane in flight
// stay in registers.
template <typename T, int NF, bool SOLID>
constexpr int site_rows() {
  return sizeof(T) * NF <= (SOLID ? 12 : 24) ? 4 : 2;
}

constexpr int kSiteTargetBlocks = 512;  // two blocks of 4 waves per CU

template <typename T, int NF, int MODE, bool SOLID>
int launch_site_solid(const PFUArgs& u, const PFArgs& con, const T* x, const T* d, T t, T* g, RedScratch rs,
                      hipStream_t s) {
  constexpr int R = site_rows<T, NF, SOLID>();
  TileGeom G;
  if (!tile_geom(u.X, u.Y, u.Z, R, 0, kSiteTargetBlocks, kMaxRedBlocks, G, 0, march_busy(NF * sizeof(T))))
    throw std::invalid_argument("PhaseFieldUnstructured: grid too large for one launch");
  pfu_site_kernel<T, NF, MODE, R, SOLID><<<G.nblocks, kBlock, 0, s>>>(u, con, G, x, d, t, g, rs);
  return G.nblocks;
}

template <typename T, int NF, int MODE>
int launch_site_nf(const PFUArgs& u, const PFArgs& con, const T* x, const T* d, T t, T* g, RedScratch rs,
                   hipStream_t s) {
  return u.wcode ? launch_site_solid<T, NF, MODE, true>(u, con, x, d, t, g, rs, s)
                 : launch_site_solid<T, NF, MODE, false>(u, con, x, d, t, g, rs, s);
}

template <typename T, int MODE>
int launch_site(const PFUArgs& u, const PFArgs& con, const T* x, const T* d, T t, T* g, RedScratch rs,
                hipStream_t s) {
  switch (u.nf) {
    case 1: return launch_site_nf<T, 1, MODE>(u, con, x, d, t, g, rs, s);
    case 2: return launch_site_nf<T, 2, MODE>(u, con, x, d, t, g, rs, s);
    case 3: return launch_site_nf<T, 3, MODE>(u, con, x, d, t, g, rs, s);
    default: return launch_site_nf<T, 4, MODE>(u, con, x, d, t, g, rs, s);
  }
}

// Fluid volumes for the volume term (:284-293).
template <typename T, typename TV, bool DIR>
__global__ __launch_bounds__(kBlock) void pfu_volumes_kernel(PFUArgs u, const T* __restrict__ x,
                                                             const TV* __restrict__ d, T t, RedScratch rs) {
  const Coords<T, TV, DIR> cx{x, d, t};
  const int nf = u.nf;
  double acc[kPFMaxFluid];
#pragma unroll
  for (int k = 0; k < kPFMaxFluid; k++) acc[k] = 0.0;
  for (size_t s = (size_t)blockIdx.x * kBlock + threadIdx.x; s < u.ngrid; s += (size_t)gridDim.x * kBlock) {
    const double v = u.node_vol[s];
#pragma unroll
    for (int k = 0; k < kPFMaxFluid; k++) {
      if (k >= nf) continue;
      const double c = (double)cx((int)(s * nf + k));
      acc[k] += (nf == 1) ? (0.5 * (c + 1)) * v : c * v;
    }
  }
  grid_sum_store<kPFMaxFluid>(acc, rs);
}

// volCoef * volDiff per fluid, and (with the energy) the term's energy added to
// the elements' (:295-300).  One thread.
__global__ void pfu_volfix_kernel(PFUArgs u, const double* __restrict__ vol, double* __restrict__ energy,
                                  double* mirror, int want_energy, double* eOut) {
  if (threadIdx.x != 0 || blockIdx.x != 0) return;
  double e = want_energy ? energy[0] : 0.0;
  for (int k = 0; k < u.nf; k++) {
    const double diff = vol[k] - u.volume[k];
    e += u.vol_coef * (diff * diff) / 1;
    u.volg[k] = u.vol_coef * diff;
  }
  if (want_energy) energy[0] = e;
  if (want_energy && mirror) mirror[0] = e;
  if (eOut) *eOut = e;
}

// The volume term's gradient, weighted towards interfaces (:301-306).
template <typename T, typename TV, bool DIR>
__global__ __launch_bounds__(kBlock) void pfu_volgrad_kernel(PFUArgs u, const T* __restrict__ x,
                                                             const TV* __restrict__ d, T t, TV* __restrict__ g) {
  const Coords<T, TV, DIR> cx{x, d, t};
  const size_t nd = u.ngrid * u.nf;
  for (size_t i = (size_t)blockIdx.x * kBlock + threadIdx.x; i < nd; i += (size_t)gridDim.x * kBlock) {
    const int k = (int)(i % u.nf);
    const T c = cx((int)i);
    T w = ((T)4 * c) * ((T)1 - c);
    if (w < (T)0) w = (T)0;
    const T add = (((T)u.volg[k] * (T)u.node_vol[i / u.nf]) * w);
    g[i] = (TV)((T)g[i] + add);
  }
}

template <typename T, int MODE>
void launch_chunk(const PFUArgs& u, int nb, const T* x, const T* d, T t, T* g, RedScratch rs, hipStream_t s) {
  switch (u.nf) {
    case 1: pfu_chunk_kernel<T, T, MODE, 1><<<nb, kBlock, 0, s>>>(u, x, d, t, g, rs); break;
    case 2: pfu_chunk_kernel<T, T, MODE, 2><<<nb, kBlock, 0, s>>>(u, x, d, t, g, rs); break;
    case 3: pfu_chunk_kernel<T, T, MODE, 3><<<nb, kBlock, 0, s>>>(u, x, d, t, g, rs); break;
    case 4: pfu_chunk_kernel<T, T, MODE, 4><<<nb, kBlock, 0, s>>>(u, x, d, t, g, rs); break;
    default: pfu_chunk_kernel<T, T, MODE, 0><<<nb, kBlock, 0, s>>>(u, x, d, t, g, rs); break;
  }
}

// Blocks of a chunk-kernel launch: each loops over chunks (at most
// kMaxRedBlocks blocks write reduction partials).
int chunk_blocks(const PFUArgs& u) { return u.nchunk < 1 ? 1 : (u.nchunk < 2048 ? u.nchunk : 2048); }

// The elements' energies (reduction value 0 of the block count returned) and
// gradient: constrained when gathered per site, else not.
template <typename T>
int launch_elements(const PFUArgs& u, const PFArgs& con, int mode, const T* x, const T* d, T t, T* g, RedScratch rs,
                    hipStream_t s) {
  if (u.gather) {
    switch (mode) {
      case 1: return launch_site<T, 1>(u, con, x, d, t, g, rs, s);
      case 2: return launch_site<T, 2>(u, con, x, d, t, g, rs, s);
      case 3: return launch_site<T, 3>(u, con, x, d, t, g, rs, s);
      case 5: return launch_site<T, 5>(u, con, x, d, t, g, rs, s);
      default: throw std::invalid_argument("pfu: unsupported evaluation mode");
    }
  }
  const int nb = chunk_blocks(u);
  switch (mode) {
    case 1: launch_chunk<T, 1>(u, nb, x, d, t, g, rs, s); break;
    case 2: launch_chunk<T, 2>(u, nb, x, d, t, g, rs, s); break;
    case 3: launch_chunk<T, 3>(u, nb, x, d, t, g, rs, s); break;
    case 5: launch_chunk<T, 5>(u, nb, x, d, t, g, rs, s); break;
    default: throw std::invalid_argument("pfu: unsupported evaluation mode");
  }
  if ((mode & 2) && u.ngather)
    pfu_gather_kernel<T><<<grid_blocks(u.ngather * u.nf, 1, 8192), kBlock, 0, s>>>(u, g);
  return nb;
}

template <typename T>
void eval_t(const PFUArgs& u, const PFArgs& con, int mode, const void* x, const void* d, double t, void* g,
            RedScratch rs, hipStream_t s, double* eOut) {
  const T* xx = static_cast<const T*>(x);
  const T* dd = static_cast<const T*>((mode & 4) ? d : x);
  T* gg = static_cast<T*>(g);
  const T tt = (T)t;
  const size_t nd = u.ngrid * u.nf;
  const RedScratch re = rs.only(0, (mode & 1) && !u.volfix ? eOut : nullptr);
  const int nb = launch_elements<T>(u, con, mode, xx, dd, tt, gg, re, s);
  MINIM_HIP_CHECK(hipGetLastError());
  launch_finalize(re, 1, nb, s);
  if (u.volfix) {
    const RedScratch slot = rs.from(kPFVolSlot);
    const int nbv = grid_blocks(u.ngrid, 4, 2048);
    if (mode & 4)
      pfu_volumes_kernel<T, T, true><<<nbv, kBlock, 0, s>>>(u, xx, dd, tt, slot);
    else
      pfu_volumes_kernel<T, T, false><<<nbv, kBlock, 0, s>>>(u, xx, dd, tt, slot);
    launch_finalize(slot, kPFMaxFluid, nbv, s);
    pfu_volfix_kernel<<<1, 64, 0, s>>>(u, rs.result + kPFVolSlot, rs.result, rs.mirror, (mode & 1) ? 1 : 0,
                                       (mode & 1) ? eOut : nullptr);
    if (mode & 2) pfu_volgrad_kernel<T, T, false><<<grid_blocks(nd, 4, 4096), kBlock, 0, s>>>(u, xx, dd, tt, gg);
    MINIM_HIP_CHECK(hipGetLastError());
  }
  // the site kernel has projected the elements' gradient; the projection of
  // what the volume term adds to it gives the projection of the sum
  if ((mode & 2) && (!u.gather || u.volfix)) pf_launch_constrain(con, sizeof(T) == 8 ? F64 : F32, gg, u.ngrid, rs, s);
}

// The fewest rows per thread (so the most tiles) of the two precisions.
template <int NF>
constexpr int least_rows(bool solid) {
  constexpr int a = std::min(site_rows<double, NF, true>(), site_rows<float, NF, true>());
  constexpr int b = std::min(site_rows<double, NF, false>(), site_rows<float, NF, false>());
  return solid ? a : b;
}

}  // namespace

bool pfu_site_fits(const int canon[3], int nf, bool solid) {
  if ((double)canon[1] * canon[2] * nf * sizeof(double) >= 4294967296.0) return false;
  int R;
  switch (nf) {
    case 1: R = least_rows<1>(solid); break;
    case 2: R = least_rows<2>(solid); break;
    case 3: R = least_rows<3>(solid); break;
    case 4: R = least_rows<4>(solid); break;
    default: return false;
  }
  TileGeom G;
  return tile_geom(canon[0], canon[1], canon[2], R, 0, kSiteTargetBlocks, kMaxRedBlocks, G);
}

void pfu_launch_eval(const PFUArgs& u, const PFArgs& con, int prec, int mode, const void* x, const void* d, double t,
                     void* g, RedScratch rs, hipStream_t s, double* eOut) {
  if ((mode & 4) && (mode & 2)) throw std::invalid_argument("pfu: gradients at a trial point are not supported");
  if (u.ngrid * (size_t)u.nf >= (size_t)1 << 31) throw std::invalid_argument("pfu: more than 2^31 DOFs");
  if (prec == F64) eval_t<double>(u, con, mode, x, d, t, g, rs, s, eOut);
  else eval_t<float>(u, con, mode, x, d, t, g, rs, s, eOut);
}

double pfu_time_elements(const PFUArgs& u, const PFArgs& con, int prec, int mode, const void* x, void* g, int reps,
                         RedScratch rs, hipStream_t s) {
  auto launch = [&]() {
    if (prec == F64) {
      const double* xx = static_cast<const double*>(x);
      launch_elements<double>(u, con, mode == 1 ? 1 : 3, xx, xx, 0.0, (double*)g, rs, s);
    } else {
      const float* xx = static_cast<const float*>(x);
      launch_elements<float>(u, con, mode == 1 ? 1 : 3, xx, xx, 0.0f, (float*)g, rs, s);
    }
  };
  launch();
  MINIM_HIP_CHECK(hipGetLastError());
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

}  // namespace minim_amd
