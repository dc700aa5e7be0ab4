// bah.hip -- bar-and-hinge elastic sheet on MI355X.
//
// Element kernels follow BarAndHinge::stretching (src/potentials/BarAndHinge.cpp:269-290,
// including its gradient factor 2*k*dl/l, twice the derivative of its
// 0.5*k*dl^2 energy), bending (:293-356) and forceEnergy (:359-369); element
// order and the all-DOFs-fixed skip follow BarAndHinge::init (:16-67).
//
// The reference loops over heap elements and scatters into g.  Here a block
// takes clusters of up to kBaHNodes nodes (bah_mesh.hpp), stages the positions
// that their elements need in LDS, evaluates each hinge that touches a cluster
// once and each bar at each of its ends there, leaves the hinges' forces in LDS,
// and then two threads per own node add its elements' forces in the order of the
// element lists.  Energy and gradient come from the same pass, every
// gradient entry is written once, and there are no atomics and no per-element
// stores: bitwise reproducible.  At 1024^2 nodes, energy and gradient: 116 us in
// FP64 and 72 in FP32; an energy pass that stored each hinge's angle, then a
// gather per node that recomputed four hinges per hinge, took 240 and 150.
//
// Rigidities, rest lengths and rest angles that are the same for every
// element are passed as scalars instead of per-element streams.
//
// Bending angle: the FP64 path uses the reference's acos form (bit-level
// parity); the FP32 path uses atan2(|b2| n1.b3, n1.n2), the same angle without
// acos's loss of precision near 0 and pi.
#include <algorithm>
#include <cmath>
#include <stdexcept>
#include <typeinfo>

#include "bah_mesh.hpp"
#include "common.hpp"
#include "minim/BarAndHinge.h"
#include "runtime.hpp"
#include "vec.hpp"

namespace minim_amd {
namespace {

struct BaHArgs {
  int nnode, ncluster, nchunk;
  const BaHChunk* chunk;
  const int* cluster;    // first chunk of each cluster
  const int* node;       // node tables
  const double* bk;      // per bar code, or null: every bar has bkU
  const double* bl0;     // ... bl0U
  const ushort4* hinge;
  const double* hk;      // per hinge record, or null: hkU
  const double* ht0;     // ... ht0U
  double bkU, bl0U, hkU, ht0U;
  const ushort4* bcode;  // BaHCodes, four codes each
  const ushort4* hcode;
  const double* fz;      // per node (cluster order) z force or nullptr
  const unsigned char* flags;  // per node (cluster order): bits 0-2 the fixed components, bit 3 the force exists
};

// flags
constexpr unsigned char kForced = 8;

// Parts of the energy (componentEnergy asks for one of them).
enum BaHParts : int { kBars = 1, kHinges = 2, kForces = 4, kAllParts = 7 };

template <typename T>
__device__ inline void cross(const T (&a)[3], const T (&b)[3], T (&c)[3]) {
  c[0] = a[1] * b[2] - a[2] * b[1];
  c[1] = a[2] * b[0] - a[0] * b[2];
  c[2] = a[0] * b[1] - a[1] * b[0];
}

template <typename T>
__device__ inline T dot3(const T (&a)[3], const T (&b)[3]) {
  return a[0] * b[0] + a[1] * b[1] + a[2] * b[2];
}

// Correctly rounded FP64 quotients and roots as the compiler's, without its
// scaling of operands near the ends of the exponent range (12 and 22
// instructions become 8 and 13).  The operands here are lengths to the powers
// 1 to 4; the angle's cosine already takes one to the power 8.  A reciprocal by
// Newton's iteration, then one correction by the exact remainder (Markstein,
// IA-64 and Elementary Functions, 2000, ch. 8 and 9).
__device__ inline double reciprocal(double b) { return newton_rcp(b); }
__device__ inline float reciprocal(float b) { return b; }
// a / b, with r = reciprocal(b)
__device__ inline double quotient(double a, double b, double r) {
  const double q = a * r;
  return __builtin_fma(__builtin_fma(-b, q, a), r, q);
}
__device__ inline float quotient(float a, float b, float) { return a / b; }
template <typename T>
__device__ inline T quotient(T a, T b) {
  return quotient(a, b, reciprocal(b));
}
__device__ inline double root(double x) {
  const double y = __builtin_amdgcn_rsq(x);
  double g = x * y, h = 0.5 * y;
  const double e = __builtin_fma(-h, g, 0.5);
  g = __builtin_fma(g, e, g);
  h = __builtin_fma(h, e, h);
  g = __builtin_fma(__builtin_fma(-g, g, x), h, g);
  g = __builtin_fma(__builtin_fma(-g, g, x), h, g);
  return x == 0.0 || x == __builtin_inf() ? x : g;
}
__device__ inline float root(float x) { return sqrt(x); }

// Hinge geometry shared by energy and gradient.
template <typename T>
struct HingeGeo {
  T b1[3], b2[3], b3[3], n1[3], n2[3];
  T b2m, n1sq, n2sq, dtheta;
};

// Hinge geometry from the four node positions, without the angle.
template <typename T>
__device__ inline void hinge_geo_vec(const T (&x1)[3], const T (&x2)[3], const T (&x3)[3], const T (&x4)[3],
                                     HingeGeo<T>& G) {
#pragma unroll
  for (int k = 0; k < 3; k++) {
    G.b1[k] = x2[k] - x1[k];
    G.b2[k] = x3[k] - x2[k];
    G.b3[k] = x4[k] - x3[k];
  }
  G.b2m = root(dot3(G.b2, G.b2));
  cross(G.b1, G.b2, G.n1);
  cross(G.b2, G.b3, G.n2);
  G.n1sq = dot3(G.n1, G.n1);
  G.n2sq = dot3(G.n2, G.n2);
}

// The bending angle's deviation from the rest angle t0.
template <typename T>
__device__ inline void hinge_dtheta(HingeGeo<T>& G, T t0) {
  const T n1b3 = dot3(G.n1, G.b3);
  const T pi = (T)3.14159265358979323846;
  T theta;
  if (sizeof(T) == 8) {
    T c = quotient(dot3(G.n1, G.n2), root(G.n1sq * G.n2sq));
    c = c < (T)-1 ? (T)-1 : c;
    c = c > (T)1 ? (T)1 : c;
    theta = (n1b3 >= 0) ? acos(c) : (T)2 * pi - acos(c);
  } else {
    const T yv = G.b2m * n1b3;
    const T at = atan2(yv, dot3(G.n1, G.n2));
    theta = (yv >= 0) ? at : (T)2 * pi + at;
  }
  // dtheta = fmod(theta - t0 + pi, 2 pi) - pi (BarAndHinge.cpp:324).  With
  // |a| < 2b, fmod(a, b) is a, a - b or a + b, each exact (Sterbenz), so the
  // library call is needed only for rest angles far outside [0, 2 pi].
  const T a = (theta - t0) + pi, b2 = (T)2 * pi;
  T r;
  if (a < (T)2 * b2 && a > -(T)2 * b2) r = a >= b2 ? a - b2 : (a <= -b2 ? a + b2 : a);
  else r = fmod(a, b2);
  G.dtheta = r - pi;
}

// A hinge's gradient at its four nodes (BarAndHinge.cpp:336-354).  With
// A = k dtheta |b2| n1 / |n1|^2, B = k dtheta |b2| n2 / |n2|^2,
// skew1 = -b1.b2 / |b2|^2, skew2 = -b3.b2 / |b2|^2: node 0 gets -A, node 1
// (1 - skew1) A - skew2 B, node 2 skew1 A - (1 - skew2) B, node 3 B.
template <typename T>
__device__ inline void hinge_gradient(const HingeGeo<T>& G, T k, T (&f)[4][3]) {
  const T gf = k * (G.dtheta);
  const T f1 = quotient(G.b2m, G.n1sq), f2 = quotient(G.b2m, G.n2sq);
  const T bb = G.b2m * G.b2m, rb = reciprocal(bb);
  const T s1 = quotient(-dot3(G.b1, G.b2), bb, rb);
  const T s2 = quotient(-dot3(G.b3, G.b2), bb, rb);
#pragma unroll
  for (int c = 0; c < 3; c++) {
    const T A = gf * (f1 * G.n1[c]);
    const T B = gf * (f2 * G.n2[c]);
    f[0][c] = -A;
    f[1][c] = ((T)1 - s1) * A - s2 * B;
    f[2][c] = s1 * A - ((T)1 - s2) * B;
    f[3][c] = B;
  }
}

// What a thread reads for a chunk: one node of the table, two hinge records,
// and the first codes of the node that it adds up.
template <typename T, typename TV>
struct ChunkIn {
  T x[3];
  TV d[3];
  int node;
  ushort4 hinge[2], bcode, hcode[2];
};

// The neighbouring lane's value (lanes 2 i and 2 i + 1 exchange).
__device__ inline int swap_pair(int v) { return __builtin_amdgcn_mov_dpp(v, 0xB1, 0xF, 0xF, true); }
__device__ inline float swap_pair(float v) { return __int_as_float(swap_pair(__float_as_int(v))); }
__device__ inline double swap_pair(double v) {
  return __hiloint2double(swap_pair(__double2hiint(v)), swap_pair(__double2loint(v)));
}

// Adds the four terms of this lane, then the four of its neighbour: in the even
// lane of a pair, the order of the codes.
template <typename T>
__device__ inline void add_pair(T (&sum)[3], const T (&f)[4][3]) {
#pragma unroll
  for (int v = 0; v < 4; v++)
#pragma unroll
    for (int m = 0; m < 3; m++) sum[m] += f[v][m];
#pragma unroll
  for (int v = 0; v < 4; v++)
#pragma unroll
    for (int m = 0; m < 3; m++) sum[m] += swap_pair(f[v][m]);
}

// Blocks of a launch: as many as are resident at once (LDS and registers let
// three FP64 and five FP32 blocks share a CU), each with an equal run of clusters.
template <typename T>
constexpr int kBaHBlocks = 256 * (sizeof(T) == 8 ? 3 : 5);

// The whole evaluation: a block works through its run of clusters (runs are
// contiguous per XCD: neighbours share nodes in one L2).  E, G: the energy, the
// gradient.  d: evaluate at x + t*d (as axpy forms it), which also goes to xout
// when given.  TV: the storage of d and g (FP32 for FP64 arithmetic in the
// mixed schedule).  mask: fixed components of the gradient are zero.
//
// Per chunk: positions to LDS, barrier, bars (at each end: two threads per
// node, every other entry of its codes) and hinges (two per thread), whose
// forces on their four nodes go to LDS component by component, barrier, then a
// node's two threads fetch its hinges' forces, and the even one adds them up,
// bars and hinges in the order of the lists.  The next chunk's reads are in
// flight during all of it, two barriers per chunk.
//
// Bound by VALU issue: 1,190 instructions per wave and chunk in FP64, 74 % of
// the time of the three blocks per CU (one chunk per block without the reads
// ahead, with bars in LDS and four barriers: 54 %, 155 us at 1024^2 nodes; eight
// terms per hinge in LDS that each node combined itself: 160 us).  FP64 blocks
// stand three to a CU by their 52 KB of LDS and 150 registers.
template <typename T, typename TV, bool E, bool G>
__global__ __launch_bounds__(kBlock, sizeof(T) == 8 ? 3 : 5) void bah_kernel(
    BaHArgs a, const BaHChunk* __restrict__ chunks, const int* __restrict__ nodes, const T* __restrict__ x,
    const TV* __restrict__ d, T t, T* __restrict__ xout, TV* __restrict__ g, bool mask, int parts, RedScratch rs) {
  static_assert(kBaHTable == kBlock && kBaHHinges <= 2 * kBlock && 2 * kBaHNodes <= kBlock, "threads");
  __shared__ T sx[3][kBaHTable];
  __shared__ int sn[G ? kBaHNodes : 1];
  __shared__ T st[G ? 12 * kBaHCol : 1];
  const int tid = threadIdx.x, own = tid >> 1, half = tid & 1;
  if (G && tid < 12) st[tid * kBaHCol + kBaHHinges] = (T)0;
  double acc[1] = {0.0};
  const int b = xcd_logical_block(blockIdx.x, gridDim.x);
  const int k0 = (int)((long long)a.ncluster * b / gridDim.x);
  const int k1 = (int)((long long)a.ncluster * (b + 1) / gridDim.x);
  const int c0 = k0 < a.ncluster ? a.cluster[k0] : a.nchunk;
  const int c1 = k1 < a.ncluster ? a.cluster[k1] : a.nchunk;

  // entry 2 q + half of this thread's node
  auto codes = [&](const ushort4* from, uint32_t at, int nCode, int nOwn, int q, unsigned short pad) {
    ushort4 w = make_ushort4(pad, pad, pad, pad);
    if (own < nOwn && 2 * q + half < nCode) w = from[at + (size_t)(2 * q + half) * nOwn + own];
    return w;
  };
  auto node_of = [&](const BaHChunk& c) { return tid < c.nNode ? nodes[c.node0 + tid] : 0; };
  auto read = [&](const BaHChunk& c, int node, ChunkIn<T, TV>& in) {
    in.node = node;
    if (tid < c.nNode) {
#pragma unroll
      for (int q = 0; q < 3; q++) {
        in.x[q] = x[(size_t)node * 3 + q];
        if (d) in.d[q] = d[(size_t)node * 3 + q];
      }
    }
    const int nHinge = G ? c.nHinge : c.nHingeOwn;
#pragma unroll
    for (int u = 0; u < 2; u++)
      if (tid + u * kBlock < nHinge) in.hinge[u] = a.hinge[c.hinge0 + tid + u * kBlock];
    in.bcode = codes(a.bcode, c.bcode0, c.nBarCode, c.nOwn, 0, kBaHNoBar);
    if (G) {
#pragma unroll
      for (int q = 0; q < 2; q++) in.hcode[q] = codes(a.hcode, c.hcode0, c.nHingeCode, c.nOwn, q, kBaHNoHinge);
    }
  };

  if (c0 < c1) {
    BaHChunk c = chunks[c0], next = chunks[min(c0 + 1, c1 - 1)];
    ChunkIn<T, TV> in;
    read(c, node_of(c), in);
    int nextNode = node_of(next);
    T gn[3] = {(T)0, (T)0, (T)0};
    for (int ci = c0; ci < c1; ci++) {
      if (tid < c.nNode) {
#pragma unroll
        for (int q = 0; q < 3; q++) {
          T p = in.x[q];
          if (d) {
            const T s = t * (T)in.d[q];
            p = p + s;
          }
          sx[q][tid] = p;
          if (xout && tid < c.nOwn) xout[(size_t)in.node * 3 + q] = p;
        }
        if (G && tid < c.nOwn) sn[tid] = in.node;
      }
      const ChunkIn<T, TV> now = in;
      const BaHChunk after = chunks[min(ci + 2, c1 - 1)];
      lds_barrier();
      read(next, nextNode, in);
      nextNode = node_of(after);

      const bool mine = own < c.nOwn;
      const int me = mine ? own : 0;
      T p[3];
#pragma unroll
      for (int q = 0; q < 3; q++) p[q] = sx[q][me];
      const int gnode = G ? sn[me] : 0;
      if (G || (parts & kBars)) {
        auto bars = [&](const ushort4& w, int q) {
          const int cs[4] = {w.x, w.y, w.z, w.w};
          T f[4][3];
#pragma unroll
          for (int v = 0; v < 4; v++) {
            f[v][0] = f[v][1] = f[v][2] = (T)0;
            if (cs[v] == kBaHNoBar || (!G && (cs[v] & 1))) continue;
            const size_t at = 4 * (c.bcode0 + (size_t)(2 * q + half) * c.nOwn + own) + v;
            const T kb = (T)(a.bk ? a.bk[at] : a.bkU), l0 = (T)(a.bl0 ? a.bl0[at] : a.bl0U);
            T dx[3];
#pragma unroll
            for (int m = 0; m < 3; m++) dx[m] = p[m] - sx[m][cs[v] >> 1];
            const T l = root(dot3(dx, dx));
            const T dl = l - l0;
            if (E && (cs[v] & 1) == 0) acc[0] += (double)((T)0.5 * kb * (dl * dl));
            // stretching gradient 2 k (l - l0) / l * dx (BarAndHinge.cpp:282)
            const T gf = quotient((T)2 * kb * dl, l);
#pragma unroll
            for (int m = 0; m < 3; m++) f[v][m] = gf * dx[m];
          }
          if constexpr (G) add_pair(gn, f);
        };
        bars(now.bcode, 0);
        for (int q = 1; 2 * q < c.nBarCode; q++)
          bars(codes(a.bcode, c.bcode0, c.nBarCode, c.nOwn, q, kBaHNoBar), q);
      }
      if (G || (parts & kHinges)) {
        const int nHinge = G ? c.nHinge : c.nHingeOwn;
#pragma unroll
        for (int u = 0; u < 2; u++) {
          const int i = tid + u * kBlock;
          if (i >= nHinge) break;
          const T kh = (T)(a.hk ? a.hk[c.hinge0 + i] : a.hkU), t0 = (T)(a.ht0 ? a.ht0[c.hinge0 + i] : a.ht0U);
          T x1[3], x2[3], x3[3], x4[3];
#pragma unroll
          for (int q = 0; q < 3; q++) {
            x1[q] = sx[q][now.hinge[u].x];
            x2[q] = sx[q][now.hinge[u].y];
            x3[q] = sx[q][now.hinge[u].z];
            x4[q] = sx[q][now.hinge[u].w];
          }
          HingeGeo<T> geo;
          hinge_geo_vec(x1, x2, x3, x4, geo);
          hinge_dtheta(geo, t0);
          if (E && i < c.nHingeOwn) acc[0] += (double)((T)0.5 * kh * (geo.dtheta * geo.dtheta));
          if constexpr (G) {
            T f[4][3];
            hinge_gradient(geo, kh, f);
#pragma unroll
            for (int v = 0; v < 4; v++)
#pragma unroll
              for (int q = 0; q < 3; q++) st[bah_slot(i, v) + q * kBaHCol] = f[v][q];
          }
        }
      }
      if (a.fz && !c.more && mine && half == 0 && (a.flags[c.own0 + own] & kForced)) {
        const double f = a.fz[c.own0 + own];
        if (E && (parts & kForces)) acc[0] -= f * (double)p[2];
        gn[2] -= (T)f;
      }
      lds_barrier();
      if constexpr (G) {
        auto add = [&](const ushort4& w) {
          const int cs[4] = {w.x, w.y, w.z, w.w};
          T f[4][3];
#pragma unroll
          for (int v = 0; v < 4; v++)
#pragma unroll
            for (int m = 0; m < 3; m++) f[v][m] = st[cs[v] + m * kBaHCol];
          add_pair(gn, f);
        };
        add(now.hcode[0]);
        if (c.nHingeCode > 2) add(now.hcode[1]);
        for (int q = 2; 2 * q < c.nHingeCode; q++)
          add(codes(a.hcode, c.hcode0, c.nHingeCode, c.nOwn, q, kBaHNoHinge));
        if (!c.more) {
          const int fl = mask && mine ? a.flags[c.own0 + own] : 0;
#pragma unroll
          for (int q = 0; q < 3; q++) {
            if (mine && half == 0) g[(size_t)gnode * 3 + q] = fl >> q & 1 ? (TV)0 : (TV)gn[q];
            gn[q] = (T)0;
          }
        }
      }
      c = next;
      next = after;
    }
  }
  if constexpr (E) {
    __syncthreads();
    grid_sum_store<1>(acc, rs);
  }
}

}  // namespace
}  // namespace minim_amd

namespace minim {

using minim_amd::DeviceBuffer;
using minim_amd::kBlock;

struct BarAndHinge::Dev {
  minim_amd::BaHArgs args{};
  std::shared_ptr<DeviceBuffer> mem, ht0;  // the tables; rest angles that were set one by one
  std::vector<int> hinge;                  // the hinge of each record
  std::vector<int> fixed;                  // the single-DOF constraints that the tables are for
  size_t nFixed = 0;                       // constraints that the node flags hold
};

BarAndHinge& BarAndHinge::setTriangulation(const vector2d<int>& triList) {
  tri_ = triList;
  tablesStale_ = true;
  return *this;
}
BarAndHinge& BarAndHinge::setBondList(const vector2d<int>& b) {
  bonds_ = b;
  tablesStale_ = true;
  return *this;
}
BarAndHinge& BarAndHinge::setHingeList(const vector2d<int>& h) {
  hinges_ = h;
  tablesStale_ = true;
  return *this;
}
BarAndHinge& BarAndHinge::setRigidity(double kb, double kh) {
  kBond_ = {kb};
  kHinge_ = {kh};
  tablesStale_ = true;
  return *this;
}
BarAndHinge& BarAndHinge::setRigidity(const vector<double>& kb, const vector<double>& kh) {
  if (!kb.empty()) kBond_ = kb;
  if (!kh.empty()) kHinge_ = kh;
  tablesStale_ = true;
  return *this;
}
BarAndHinge& BarAndHinge::setLength0(double l) {
  length0_ = {l};
  tablesStale_ = true;
  return *this;
}
BarAndHinge& BarAndHinge::setLength0(const vector<double>& l) {
  length0_ = l;
  tablesStale_ = true;
  return *this;
}
BarAndHinge& BarAndHinge::setTheta0(double t) {
  theta0_ = {t};
  tablesStale_ = true;
  return *this;
}
BarAndHinge& BarAndHinge::setTheta0(const vector<double>& t) {
  theta0_ = t;
  tablesStale_ = true;
  return *this;
}
BarAndHinge& BarAndHinge::setForce(const vector<double>& f) {
  force_ = f;
  tablesStale_ = true;
  return *this;
}

namespace {

// The edges of all triangles, sorted by (lower node, upper node, triangle):
// edge k of triangle t joins its nodes k and k + 1.
struct Edges {
  struct Edge {
    int lo, hi, id;  // id: 3 t + k
  };
  std::vector<Edge> e;
  std::vector<int> first;  // per id: the first of the edges that join the same nodes
  explicit Edges(const vector2d<int>& tris) : e(3 * tris.size()), first(3 * tris.size()) {
    int least = 0, most = -1;
    for (size_t t = 0; t < tris.size(); t++) {
      if (tris[t].size() != 3) throw std::invalid_argument("BarAndHinge: triangles need three nodes.");
      for (int k = 0; k < 3; k++) {
        const int a = tris[t][k], b = tris[t][(k + 1) % 3];
        e[3 * t + k] = {std::min(a, b), std::max(a, b), (int)(3 * t + k)};
        least = std::min(least, e[3 * t + k].lo);
        most = std::max(most, e[3 * t + k].hi);
      }
    }
    auto before = [](const Edge& u, const Edge& v) {
      return u.lo != v.lo ? u.lo < v.lo : u.hi != v.hi ? u.hi < v.hi : u.id < v.id;
    };
    if (least >= 0 && (size_t)most < 4 * e.size()) {
      // by lower node first (a count per node), then each node's few edges
      std::vector<size_t> at(most + 2, 0);
      for (const auto& x : e) at[x.lo + 1]++;
      for (int n = 0; n <= most; n++) at[n + 1] += at[n];
      std::vector<Edge> s(e.size());
      auto next = at;
      for (const auto& x : e) s[next[x.lo]++] = x;
      e.swap(s);
      for (int n = 0; n <= most; n++) std::sort(e.begin() + at[n], e.begin() + at[n + 1], before);
    } else {
      std::sort(e.begin(), e.end(), before);
    }
    for (size_t i = 0; i < e.size(); i++)
      first[e[i].id] = i > 0 && same(i - 1, i) ? first[e[i - 1].id] : (int)i;
  }
  bool same(size_t i, size_t j) const { return e[i].lo == e[j].lo && e[i].hi == e[j].hi; }
};

// Bond list of BarAndHinge::computeBondList (BarAndHinge.cpp:70-93): sorted
// node pairs of every triangle, lexicographically sorted and unique.
vector2d<int> bonds_from_tris(const vector2d<int>& tris) {
  const Edges g(tris);
  vector2d<int> out;
  out.reserve(g.e.size() / 2 + 1);
  for (size_t i = 0; i < g.e.size(); i++)
    if (i == 0 || !g.same(i - 1, i)) out.push_back({g.e[i].lo, g.e[i].hi});
  return out;
}

// Hinge list of BarAndHinge::computeHingeList (BarAndHinge.cpp:96-147) in
// the same order, built from the triangles of each edge instead of the
// reference's all-pairs triangle loop: for each triangle it1 and each later
// triangle it2 sharing exactly two nodes, nodes = [unshared of it1, the next
// two of it1 in cyclic order, unshared of it2].
vector2d<int> hinges_from_tris(const vector2d<int>& tris) {
  const Edges g(tris);
  vector2d<int> out;
  out.reserve(g.e.size() / 2 + 1);
  std::vector<int> cand;
  for (int it1 = 0; it1 < (int)tris.size(); it1++) {
    cand.clear();
    for (int k = 0; k < 3; k++) {
      const size_t i0 = g.first[3 * (size_t)it1 + k];
      for (size_t i = i0; i < g.e.size() && g.same(i0, i); i++)
        if (g.e[i].id / 3 > it1) cand.push_back(g.e[i].id / 3);
    }
    std::sort(cand.begin(), cand.end());
    cand.erase(std::unique(cand.begin(), cand.end()), cand.end());
    for (int it2 : cand) {
      bool s1[3] = {false, false, false}, s2[3] = {false, false, false};
      int nShared = 0;
      for (int a = 0; a < 3; a++)
        for (int b = 0; b < 3; b++)
          if (tris[it1][a] == tris[it2][b]) {
            nShared++;
            s1[a] = true;
            s2[b] = true;
          }
      if (nShared != 2) continue;
      std::vector<int> nodes(4);
      for (int a = 0; a < 3; a++)
        if (!s1[a]) {
          nodes[0] = tris[it1][a];
          nodes[1] = tris[it1][(a + 1) % 3];
          nodes[2] = tris[it1][(a + 2) % 3];
        }
      for (int b = 0; b < 3; b++)
        if (!s2[b]) nodes[3] = tris[it2][b];
      out.push_back(std::move(nodes));
    }
  }
  return out;
}

double pi() { return 4 * std::atan(1.0); }

}  // namespace

// BarAndHinge::init (BarAndHinge.cpp:16-67)
void BarAndHinge::init(const vector<double>& coords) {
  if (coords.size() % 3 != 0) throw std::invalid_argument("BarAndHinge: coordinates must be 3 per node.");
  const int nnode = (int)(coords.size() / 3);
  if (bonds_.empty()) {
    if (tri_.empty()) throw std::invalid_argument("BarAndHinge: The triangulation has not been set.");
    bonds_ = bonds_from_tris(tri_);
  }
  if (hinges_.empty()) {
    if (tri_.empty()) throw std::invalid_argument("BarAndHinge: The triangulation has not been set.");
    hinges_ = hinges_from_tris(tri_);
  }
  for (auto& b : bonds_)
    if (b.size() < 2 || b[0] < 0 || b[1] < 0 || b[0] >= nnode || b[1] >= nnode)
      throw std::invalid_argument("BarAndHinge: bond references a node outside the coordinates.");
  for (auto& h : hinges_) {
    if (h.size() < 4) throw std::invalid_argument("BarAndHinge: hinges need four nodes.");
    for (int k = 0; k < 4; k++)
      if (h[k] < 0 || h[k] >= nnode) throw std::invalid_argument("BarAndHinge: hinge references a node outside the coordinates.");
  }
  // computeRigidities (:150-160), computeLength0 (:213-226), computeTheta0 (:229-248)
  if (kBond_.empty() || kHinge_.empty())
    throw std::invalid_argument("BarAndHinge requires the rigidities to be set (thickness-derived rigidities are not supported)");
  if (kBond_.size() == 1) kBond_ = vector<double>(bonds_.size(), kBond_[0]);
  if (kHinge_.size() == 1) kHinge_ = vector<double>(hinges_.size(), kHinge_[0]);
  if (kBond_.size() != bonds_.size() || kHinge_.size() != hinges_.size())
    throw std::invalid_argument("BarAndHinge: rigidity arrays do not match the element lists.");
  auto X = [&](int n, int k) { return coords[3 * (size_t)n + k]; };
  if (length0_.empty()) {
    length0_.resize(bonds_.size());
    for (size_t i = 0; i < bonds_.size(); i++) {
      double s = 0;
      for (int k = 0; k < 3; k++) {
        double v = X(bonds_[i][0], k) - X(bonds_[i][1], k);
        s += v * v;
      }
      length0_[i] = std::sqrt(s);
    }
  } else if (length0_.size() == 1) {
    length0_ = vector<double>(bonds_.size(), length0_[0]);
  }
  if (theta0_.empty()) {
    theta0_.resize(hinges_.size());
    for (size_t i = 0; i < hinges_.size(); i++) {
      const auto& h = hinges_[i];
      double b1[3], b2[3], b3[3];
      for (int k = 0; k < 3; k++) {
        b1[k] = X(h[1], k) - X(h[0], k);
        b2[k] = X(h[2], k) - X(h[1], k);
        b3[k] = X(h[3], k) - X(h[2], k);
      }
      double n1[3] = {b1[1] * b2[2] - b1[2] * b2[1], b1[2] * b2[0] - b1[0] * b2[2], b1[0] * b2[1] - b1[1] * b2[0]};
      double n2[3] = {b2[1] * b3[2] - b2[2] * b3[1], b2[2] * b3[0] - b2[0] * b3[2], b2[0] * b3[1] - b2[1] * b3[0]};
      double nn1 = std::sqrt(n1[0] * n1[0] + n1[1] * n1[1] + n1[2] * n1[2]);
      double nn2 = std::sqrt(n2[0] * n2[0] + n2[1] * n2[1] + n2[2] * n2[2]);
      double c = (n1[0] * n2[0] + n1[1] * n2[1] + n1[2] * n2[2]) / (nn1 * nn2);
      double n1b3 = n1[0] * b3[0] + n1[1] * b3[1] + n1[2] * b3[2];
      theta0_[i] = (n1b3 >= 0) ? std::acos(c) : 2 * pi() - std::acos(c);
    }
  } else if (theta0_.size() == 1) {
    theta0_ = vector<double>(hinges_.size(), theta0_[0]);
  }
  if (length0_.size() != bonds_.size() || theta0_.size() != hinges_.size())
    throw std::invalid_argument("BarAndHinge: rest length/angle arrays do not match the element lists.");
  if (!force_.empty() && force_.size() != 3 && force_.size() != coords.size())
    throw std::invalid_argument("BarAndHinge: force must have 3 or 3*nNode entries.");
  uploadFixed(coords.size());
  nNodeHint = nnode;
  order_ = std::make_shared<const vector<int>>(minim_amd::bah_mesh::order(coords, minim_amd::bah_mesh::parts(nnode)));
  upload();
}

// With tables on the device that are for these lists and constraints, only the
// angle's records change, in a copy of the angles (a copy of this potential may
// share them): at 150^2 nodes 0.1 ms, all tables anew 11.
void BarAndHinge::setHingeTheta0(int iHinge, double t0) {
  theta0_.at(iHinge) = t0;
  if (!dev_) return;
  if (tablesStale_ || dev_->fixed != fixedDofs() || dev_->nFixed != constraints.size()) {
    upload();
    return;
  }
  const size_t n = dev_->hinge.size();
  if (n == 0) return;
  auto dev = std::make_shared<Dev>(*dev_);
  dev->ht0 = std::make_shared<DeviceBuffer>(sizeof(double) * n);
  double* to = static_cast<double*>(dev->ht0->get());
  if (dev_->args.ht0) {
    MINIM_HIP_CHECK(hipMemcpy(to, dev_->args.ht0, sizeof(double) * n, hipMemcpyDeviceToDevice));
  } else {
    const std::vector<double> all(n, dev_->args.ht0U);
    MINIM_HIP_CHECK(hipMemcpy(to, all.data(), sizeof(double) * n, hipMemcpyHostToDevice));
  }
  for (size_t r = 0; r < n; r++)
    if (dev->hinge[r] == iHinge)
      MINIM_HIP_CHECK(hipMemcpy(to + r, &t0, sizeof(double), hipMemcpyHostToDevice));
  MINIM_HIP_CHECK(hipStreamSynchronize(nullptr));  // other streams read the angles next
  dev->args.ht0 = to;
  dev_ = dev;
}

void BarAndHinge::upload() {
  const int nnode = nNodeHint;
  std::vector<char> fixed(3 * (size_t)nnode, 0);
  for (int i : fixedDofs())
    if (i >= 0 && (size_t)i < fixed.size()) fixed[i] = 1;
  auto allFixed = [&](const int* nd, int k) {
    for (int q = 0; q < k; q++)
      for (int c = 0; c < 3; c++)
        if (!fixed[3 * (size_t)nd[q] + c]) return false;
    return true;
  };
  auto dev = std::make_shared<Dev>();
  std::vector<int> bar, hin, hinId;
  std::vector<double> bk, bl, hk, ht;
  bar.reserve(2 * bonds_.size());
  hin.reserve(4 * hinges_.size());
  for (size_t i = 0; i < bonds_.size(); i++) {
    int nd[2] = {bonds_[i][0], bonds_[i][1]};
    if (allFixed(nd, 2)) continue;
    bar.insert(bar.end(), nd, nd + 2);
    bk.push_back(kBond_[i]);
    bl.push_back(length0_[i]);
  }
  for (size_t i = 0; i < hinges_.size(); i++) {
    int nd[4] = {hinges_[i][0], hinges_[i][1], hinges_[i][2], hinges_[i][3]};
    if (allFixed(nd, 4)) continue;
    hin.insert(hin.end(), nd, nd + 4);
    hinId.push_back((int)i);
    hk.push_back(kHinge_[i]);
    ht.push_back(theta0_[i]);
  }
  minim_amd::BaHLists lists;
  lists.nnode = nnode;
  lists.bar = &bar;
  lists.hinge = &hin;
  const auto mesh = minim_amd::bah_mesh::build(lists, *order_, minim_amd::bah_mesh::parts(nnode));
  std::vector<double> fz;
  std::vector<unsigned char> flags(nnode, 0);
  if (!force_.empty()) fz.resize(nnode);
  for (int o = 0; o < nnode; o++) {
    const int n = (*order_)[o];
    for (int k = 0; k < 3; k++) flags[o] |= fixed[3 * (size_t)n + k] << k;
    if (force_.empty()) continue;
    fz[o] = force_.size() == 3 ? force_[2] : force_[3 * (size_t)n + 2];
    if (!allFixed(&n, 1)) flags[o] |= minim_amd::kForced;
  }
  dev->nFixed = constraints.size();
  dev->fixed = fixedDofs();
  dev->hinge.reserve(mesh.hingeId.size());
  for (int h : mesh.hingeId) dev->hinge.push_back(hinId[h]);
  // parameters shared by every element go as scalars, others per bar code and hinge record
  auto uniform = [](const std::vector<double>& v) {
    for (double x : v)
      if (!(x == v[0]) || std::signbit(x) != std::signbit(v[0])) return false;
    return true;
  };
  auto records = [&](const std::vector<double>& v, const std::vector<int>& id) {
    std::vector<double> r;
    if (uniform(v)) return r;
    r.reserve(id.size());
    for (int i : id) r.push_back(v[i]);
    return r;
  };
  const auto bkR = records(bk, mesh.barId), blR = records(bl, mesh.barId), hkR = records(hk, mesh.hingeId),
             htR = records(ht, mesh.hingeId);
  // one allocation, 256-byte aligned sub-buffers
  std::vector<std::pair<const void*, size_t>> src;
  std::vector<size_t> at;
  size_t off = 0;
  auto reserve = [&](const auto& v) {
    src.push_back({v.data(), v.size() * sizeof(v[0])});
    at.push_back(off);
    off += (src.back().second + 255) / 256 * 256;
    return at.size() - 1;
  };
  const size_t i_chunk = reserve(mesh.chunk), i_cluster = reserve(mesh.cluster), i_node = reserve(mesh.node),
               i_hinge = reserve(mesh.hinge), i_bcode = reserve(mesh.bcode),
               i_hcode = reserve(mesh.hcode), i_bk = reserve(bkR), i_bl = reserve(blR), i_hk = reserve(hkR),
               i_ht = reserve(htR), i_fz = reserve(fz), i_flags = reserve(flags);
  dev->mem = std::make_shared<DeviceBuffer>(off + 256);
  char* base = static_cast<char*>(dev->mem->get());
  for (size_t i = 0; i < src.size(); i++)
    if (src[i].second) MINIM_HIP_CHECK(hipMemcpy(base + at[i], src[i].first, src[i].second, hipMemcpyHostToDevice));
  auto dptr = [&](size_t i) { return (const double*)(src[i].second ? base + at[i] : nullptr); };
  auto& a = dev->args;
  a.nnode = nnode;
  a.ncluster = (int)mesh.cluster.size();
  a.nchunk = (int)mesh.chunk.size();
  a.chunk = (const minim_amd::BaHChunk*)(base + at[i_chunk]);
  a.cluster = (const int*)(base + at[i_cluster]);
  a.node = (const int*)(base + at[i_node]);
  a.bk = dptr(i_bk);
  a.bl0 = dptr(i_bl);
  a.hinge = (const ushort4*)(base + at[i_hinge]);
  a.hk = dptr(i_hk);
  a.ht0 = dptr(i_ht);
  a.bkU = bk.empty() ? 0.0 : bk[0];
  a.bl0U = bl.empty() ? 0.0 : bl[0];
  a.hkU = hk.empty() ? 0.0 : hk[0];
  a.ht0U = ht.empty() ? 0.0 : ht[0];
  a.bcode = (const ushort4*)(base + at[i_bcode]);
  a.hcode = (const ushort4*)(base + at[i_hcode]);
  a.fz = dptr(i_fz);
  a.flags = (const unsigned char*)(base + at[i_flags]);
  dev_ = dev;
  tablesStale_ = false;
}

namespace {
// One evaluation: energy (into rs.result[0], and to eDev when given) when
// wantE, gradient when g; at x + t*d when d, which also goes to xout when
// given.  prec: the coordinates and the arithmetic; pv: d and g (FP32 against
// FP64 coordinates in the mixed schedule).  mask: the gradient of single-DOF
// constraints comes out zero.
void launch_bah(const BarAndHinge::Dev& dv, int prec, int pv, const void* x, const void* d, double t, void* xout,
                bool wantE, void* g, bool mask, minim_amd::RedScratch rs, hipStream_t s, double* eDev = nullptr,
                int parts = minim_amd::kAllParts) {
  const auto& a = dv.args;
  rs = rs.only(0, eDev);
  if (pv != prec && !(prec == FP64 && pv == FP32))
    throw std::invalid_argument("BarAndHinge: FP32 coordinates with FP64 vectors are not supported.");
  // the same blocks with and without the gradient: the energy is the same bit for bit
  const int most = prec == FP64 ? minim_amd::kBaHBlocks<double> : minim_amd::kBaHBlocks<float>;
  const int nb = std::max(1, std::min(a.ncluster, most));
  auto go = [&](auto tag, auto vtag) {
    using T = decltype(tag);
    using TV = decltype(vtag);
    auto run = [&](auto kernel) {
      kernel<<<nb, kBlock, 0, s>>>(a, a.chunk, a.node, (const T*)x, (const TV*)d, (T)t, (T*)xout, (TV*)g, mask, parts, rs);
      MINIM_HIP_CHECK(hipGetLastError());
    };
    if (wantE && g) run(minim_amd::bah_kernel<T, TV, true, true>);
    else if (wantE) run(minim_amd::bah_kernel<T, TV, true, false>);
    else if (g) run(minim_amd::bah_kernel<T, TV, false, true>);
  };
  if (prec == FP64 && pv == FP64) go(0.0, 0.0);
  else if (prec == FP64) go(0.0, 0.0f);
  else go(0.0f, 0.0f);
  if (wantE) minim_amd::launch_finalize(rs, 1, nb, s);
}
}  // namespace

// The node flags hold every constraint (none was added since the upload, none
// reads the coordinates, and no derived class has its own): the kernel zeroes the
// fixed components itself.
bool BarAndHinge::maskHolds() const {
  return constraints.size() == dev_->nFixed && !hasNormalConstraints() && typeid(*this) == typeid(BarAndHinge);
}

void BarAndHinge::evaluate(int prec, const void* x, const void* d, double t, double* e, void* g,
                           void* stream) const {
  BarAndHinge::evaluateAsync(prec, x, d, t, e != nullptr, nullptr, g, stream);
  if (e) {
    double r[1];
    minim_amd::Workspace::current().fetch(static_cast<hipStream_t>(stream), 1, r);
    *e = r[0];
  }
}

// evaluate without the host synchronisation: the energy stays on the device
// (e_dev, or the calling thread's reduction result slot 0).
void BarAndHinge::evaluateAsync(int prec, const void* x, const void* d, double t, bool wantE, double* e_dev, void* g,
                                void* stream) const {
  if (!dev_) throw std::runtime_error("BarAndHinge: not initialised (construct a State first).");
  if (g && d) throw std::invalid_argument("BarAndHinge: gradients at a trial point are not supported.");
  if (!wantE && !g) return;
  const bool mask = maskHolds();
  launch_bah(*dev_, prec, prec, x, d, t, nullptr, wantE, g, mask, minim_amd::Workspace::current().rs(),
             static_cast<hipStream_t>(stream), wantE ? e_dev : nullptr);
  if (g && !mask) constrainDevice(prec, x, g, 3 * (size_t)dev_->args.nnode, stream);
}

// The mixed schedule's second phase: FP64 coordinates and arithmetic, the
// direction and the gradient in FP32.  Only single-DOF constraints (their
// projection does not read the coordinates).
bool BarAndHinge::supportsMixed() const { return !hasNormalConstraints(); }

void BarAndHinge::evaluateMixedAsync(const void* x, const void* d, double t, bool wantE, double* e_dev, void* g,
                                     void* stream) const {
  if (!dev_) throw std::runtime_error("BarAndHinge: not initialised (construct a State first).");
  if (g && d) throw std::invalid_argument("BarAndHinge: gradients at a trial point are not supported.");
  if (!supportsMixed()) throw std::invalid_argument("BarAndHinge: no mixed evaluation with normal constraints.");
  if (!wantE && !g) return;
  const bool mask = maskHolds();
  launch_bah(*dev_, FP64, FP32, x, d, t, nullptr, wantE, g, mask, minim_amd::Workspace::current().rs(),
             static_cast<hipStream_t>(stream), wantE ? e_dev : nullptr);
  if (g && !mask) constrainDevice(FP32, nullptr, g, 3 * (size_t)dev_->args.nnode, stream);
}

// x + t*d, formed exactly as the in-place update x += t*d would, goes to xout
// from the pass that evaluates there.  With g null only the energy is
// evaluated (the gradient is deferred until the trial is accepted).
bool BarAndHinge::supportsStep() const { return dev_ != nullptr; }
bool BarAndHinge::stepDefersGradient() const { return true; }

void BarAndHinge::evaluateStepAsync(int px, int pv, const void* x, const void* d, double t, void* xout, void* g,
                                    void* stream) const {
  if (!dev_) throw std::runtime_error("BarAndHinge: not initialised (construct a State first).");
  if (pv != px && !supportsMixed())
    throw std::invalid_argument("BarAndHinge: no mixed evaluation with normal constraints.");
  const bool mask = maskHolds();
  hipStream_t s = static_cast<hipStream_t>(stream);
  const size_t n3 = 3 * (size_t)dev_->args.nnode, bx = px == FP64 ? 8 : 4, bv = pv == FP64 ? 8 : 4;
  auto overlap = [n3](const void* p, size_t bp, const void* q, size_t bq) {
    const auto a = reinterpret_cast<uintptr_t>(p), b = reinterpret_cast<uintptr_t>(q);
    return p && q && a < b + n3 * bq && b < a + n3 * bp;
  };
  const bool scales = xout == x && d == x && px == pv;  // x = x + t*x
  if ((overlap(xout, bx, d, bv) && !scales) || overlap(xout, bx, g, bv) || (xout != x && overlap(xout, bx, x, bx)))
    throw std::invalid_argument("BarAndHinge: x + t*d must go to x or to memory of its own.");
  if (xout == x || overlap(g, bv, x, bx) || overlap(g, bv, d, bv)) {
    // a cluster reads x and d at its neighbours' nodes too: with an output over
    // an input, the point is formed first
    if (xout != x) minim_amd::device_copy(xout, x, n3 * bx, s);
    minim_amd::launch_axpy_mixed(px, xout, pv, d, t, n3, s);
    x = xout;
    d = nullptr;
    xout = nullptr;
  }
  launch_bah(*dev_, px, pv, x, d, t, xout, true, g, mask, minim_amd::Workspace::current().rs(), s);
  if (g && !mask) constrainDevice(pv, pv == px ? (xout ? xout : x) : nullptr, g, n3, stream);
}

void BarAndHinge::evaluateMixed(const void* x, const void* d, double t, double* e, void* g, void* stream) const {
  evaluateMixedAsync(x, d, t, e != nullptr, nullptr, g, stream);
  if (e) {
    double r[1];
    minim_amd::Workspace::current().fetch(static_cast<hipStream_t>(stream), 1, r);
    *e = r[0];
  }
}

// The energy of one element type (State::componentEnergy, src/State.cpp:307-312):
// the energy pass over bars (type 0), hinges (1) or the external force on the
// nodes (2) alone, in FP64 at the host coordinates.
double BarAndHinge::componentEnergy(int component, const vector<double>& coords) const {
  if (!dev_) throw std::runtime_error("BarAndHinge: not initialised (construct a State first).");
  const auto& a = dev_->args;
  if ((size_t)coords.size() != 3 * (size_t)a.nnode)
    throw std::invalid_argument("BarAndHinge: coordinates have the wrong size.");
  if (component < 0 || component > 2 || (component == 2 && !a.fz)) return 0.0;
  hipStream_t s = nullptr;
  auto& ws = minim_amd::Workspace::current();
  void* xd = minim_amd::Staging::current().device(0, coords.size() * sizeof(double));
  minim_amd::upload_raw(coords.data(), coords.size(), FP64, xd, s);
  launch_bah(*dev_, FP64, FP64, xd, nullptr, 0.0, nullptr, true, nullptr, false, ws.rs(), s, nullptr, 1 << component);
  double r[1];
  ws.fetch(s, 1, r);
  return r[0];
}

// Average duration (ms) of reps evaluations on the device (with the energy's
// reduction; no constraints, no host copy).
double BarAndHinge::timeKernel(int prec, const void* x, bool wantE, void* g, int reps, void* stream) const {
  if (!dev_) throw std::runtime_error("BarAndHinge: not initialised (construct a State first).");
  if ((!wantE && !g) || reps < 1) throw std::invalid_argument("BarAndHinge: nothing to time");
  hipStream_t s = static_cast<hipStream_t>(stream);
  auto& ws = minim_amd::Workspace::current();
  launch_bah(*dev_, prec, prec, x, nullptr, 0.0, nullptr, wantE, g, false, ws.rs(), s);
  hipEvent_t e0, e1;
  MINIM_HIP_CHECK(hipEventCreate(&e0));
  MINIM_HIP_CHECK(hipEventCreate(&e1));
  MINIM_HIP_CHECK(hipEventRecord(e0, s));
  for (int i = 0; i < reps; i++) launch_bah(*dev_, prec, prec, x, nullptr, 0.0, nullptr, wantE, g, false, ws.rs(), s);
  MINIM_HIP_CHECK(hipEventRecord(e1, s));
  MINIM_HIP_CHECK(hipEventSynchronize(e1));
  float ms = 0;
  MINIM_HIP_CHECK(hipEventElapsedTime(&ms, e0, e1));
  MINIM_HIP_CHECK(hipEventDestroy(e0));
  MINIM_HIP_CHECK(hipEventDestroy(e1));
  return (double)ms / reps;
}

}  // namespace minim
