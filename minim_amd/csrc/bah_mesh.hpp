// bah_mesh.hpp -- how a bar-and-hinge mesh is cut into clusters of nodes.
//
// Plain C++ (no HIP), so that the tables can be checked on the CPU.
//
// A cluster is up to kBaHNodes nodes that lie close together.  A block of the
// kernel evaluates the hinges that touch a cluster's own nodes once each, from
// node positions staged in LDS, and each own node then adds the hinges it is
// part of; bars are evaluated at each of their ends.  A hinge that touches
// several clusters is evaluated in each of them (a patch of 11 x 11 nodes of a
// triangulated sheet touches 1.25 hinges per hinge of its own); its energy
// counts in the cluster of its first node, a bar's at its first end.
//
// Nodes are ordered by recursive bisection of their initial positions along
// the longest side of their box.  The positions set only how many elements
// are shared: any order gives the same results.
//
// Tables per chunk (usually one per cluster; more when a single node has more
// elements than a chunk holds): the node ids, own nodes first; the hinges as
// 16-bit positions in that table, those whose energy counts here first, each
// part in list order; and for each own node, in list order, a code per bar (the
// other end's position << 1 | the node's end) and per hinge (where the kernel
// leaves the force on this corner, bah_slot), four codes per entry.
#pragma once

#include <algorithm>
#include <cmath>
#include <cstddef>
#include <cstdint>
#include <future>
#include <stdexcept>
#include <system_error>
#include <type_traits>
#include <utility>
#include <vector>

namespace minim_amd {

constexpr int kBaHNodes = 120;   // own nodes of a cluster, at most
constexpr int kBaHTable = 256;   // nodes of a chunk, at most
constexpr int kBaHHinges = 480;  // hinges of a chunk, at most

// The forces of a chunk's hinges: component m of corner k of hinge i at
// bah_slot(i, k) + m * kBaHCol.  Column kBaHHinges is zero: padding reads it.
constexpr int kBaHCol = kBaHHinges + 1;
constexpr int bah_slot(int i, int k) { return 3 * k * kBaHCol + i; }

constexpr uint16_t kBaHNoBar = 0xFFFF;                 // padding of the bar codes
constexpr uint16_t kBaHNoHinge = bah_slot(kBaHHinges, 0);  // ... and of the hinge codes

struct BaHCodes {  // four codes of one node
  uint16_t c[4];
};

struct alignas(64) BaHChunk {
  uint32_t node0;           // first entry in the node table
  uint32_t hinge0;          // first hinge record
  uint32_t bcode0, hcode0;  // first BaHCodes; entry (q, i) at q * nOwn + i
  int own0;                 // first own node in the order of all clusters
  int nOwn, nNode;          // own nodes, nodes in the table
  int nHinge, nHingeOwn;
  int nBarCode, nHingeCode;  // entries per own node
  int more;                  // the next chunk belongs to the same cluster
};

// Input lists: nodes of each bar (2) and hinge (4).
struct BaHLists {
  int nnode = 0;
  const std::vector<int>* bar = nullptr;
  const std::vector<int>* hinge = nullptr;
};

struct BaHMesh {
  std::vector<BaHChunk> chunk;
  std::vector<int> cluster;       // first chunk of each cluster
  std::vector<int> node;          // node tables
  std::vector<uint16_t> hinge;    // 4 per record
  std::vector<int> hingeId;       // list position of each record
  std::vector<BaHCodes> bcode, hcode;
  std::vector<int> barId;         // list position of each bar code (0 for padding)
};

namespace bah_mesh {

// f() on a thread of its own, or where there is none to be had when it is waited for.
template <typename F>
inline std::future<void> start(F f) {
  try {
    return std::async(std::launch::async, f);
  } catch (const std::system_error&) {
    return std::async(std::launch::deferred, f);
  }
}

// f(range) on contiguous ranges of [0, n), in parallel.
template <typename F>
inline void ranges(int n, int parts, F f) {
  std::vector<std::future<void>> job;
  for (int p = 1; p < parts; p++) {
    const int a = (int)((long long)n * p / parts), b = (int)((long long)n * (p + 1) / parts);
    job.push_back(start([=] { f(p, a, b); }));
  }
  f(0, 0, (int)((long long)n / parts));
  for (auto& j : job) j.get();
}

// Threads for the tables of n nodes: one takes about 0.3 us a node, and starting
// one some 30 us.
constexpr int kPerThread = 512;
inline int threads_for(int n) { return std::max(1, std::min(8, n / kPerThread)); }

struct Point {
  float c[3];
  int id;
};

// Parts [m0, m1) of m hold the points [n m0 / m, n m1 / m): bisect the longest
// side of the box at the middle part's border.
inline void bisect(Point* p, long long n, int m, int m0, int m1, int threads) {
  if (m1 - m0 < 2) return;
  Point *a = p + n * m0 / m, *b = p + n * m1 / m;
  if (b - a < 2) return;
  float lo[3], hi[3];
  for (int k = 0; k < 3; k++) lo[k] = hi[k] = a->c[k];
  for (Point* q = a; q != b; q++)
    for (int k = 0; k < 3; k++) {
      lo[k] = std::min(lo[k], q->c[k]);
      hi[k] = std::max(hi[k], q->c[k]);
    }
  int ax = 0;
  for (int k = 1; k < 3; k++)
    if (hi[k] - lo[k] > hi[ax] - lo[ax]) ax = k;
  const int mid = m0 + (m1 - m0) / 2;
  Point* c = p + n * mid / m;
  if (c != a && c != b)
    std::nth_element(a, c, b, [ax](const Point& u, const Point& v) {
      return u.c[ax] != v.c[ax] ? u.c[ax] < v.c[ax] : u.id < v.id;
    });
  if (threads > 1 && b - a > 2 * kPerThread) {
    auto left = start([=] { bisect(p, n, m, m0, mid, threads / 2); });
    bisect(p, n, m, mid, m1, threads - threads / 2);
    left.get();
  } else {
    bisect(p, n, m, m0, mid, 1);
    bisect(p, n, m, mid, m1, 1);
  }
}

// Nodes in cluster order; part k of m holds [n k / m, n (k + 1) / m).
inline std::vector<int> order(const std::vector<double>& coords, int m) {
  const int n = (int)(coords.size() / 3);
  std::vector<Point> p(n);
  for (int i = 0; i < n; i++) {
    for (int k = 0; k < 3; k++) {
      const float v = (float)coords[3 * (size_t)i + k];
      p[i].c[k] = std::isfinite(v) ? v : 0.0f;
    }
    p[i].id = i;
  }
  bisect(p.data(), n, m, 0, m, threads_for(n));
  std::vector<int> o(n);
  for (int i = 0; i < n; i++) o[i] = p[i].id;
  return o;
}

// Clusters of a mesh of n nodes: full ones for large meshes; smaller ones, down
// to 32 nodes, while there are fewer than 768 (three blocks per CU).
inline int parts(int n) {
  const int full = (n + kBaHNodes - 1) / kBaHNodes, least = (n + 31) / 32;
  return std::max(1, std::max(full, std::min(least, 768)));
}

// node -> places in the element list (element * corners + corner), ascending
struct Csr {
  std::vector<int> ptr, idx;
  Csr(int nnode, const std::vector<int>& e) : ptr(nnode + 1, 0), idx(e.size()) {
    for (int n : e) ptr[n + 1]++;
    for (int n = 0; n < nnode; n++) ptr[n + 1] += ptr[n];
    std::vector<int> at(ptr.begin(), ptr.end() - 1);
    for (size_t q = 0; q < e.size(); q++) idx[at[e[q]]++] = (int)q;
  }
};

// Builds the chunks of the clusters [c0, c1) into out (offsets from zero).
class Builder {
 public:
  Builder(const BaHLists& l, const Csr& bars, const Csr& hinges, const std::vector<int>& order,
          const std::vector<int>& rank, BaHMesh& out)
      : l_(l), bars_(bars), hinges_(hinges), order_(order), rank_(rank), out_(out), seen_(l.nnode, -1),
        place_(l.nnode) {}

  // The nodes order[a, b) as one cluster, or as several if they do not fit.
  void add(int a, int b) {
    a_ = a;
    b_ = b;
    collect(bars_, *l_.bar, 2, be_);
    collect(hinges_, *l_.hinge, 4, he_);
    if ((int)he_.size() <= kBaHHinges && table(be_.data(), be_.size(), he_.data(), he_.size())) {
      out_.cluster.push_back((int)out_.chunk.size());
      emit(be_.data(), be_.size(), he_.data(), he_.size(), 0);
      return;
    }
    if (b - a > 1) {
      add(a, a + (b - a) / 2);
      add(a + (b - a) / 2, b);
      return;
    }
    // one node with many elements: bars, then hinges, in pieces.  An element
    // adds at most three nodes besides the node itself.
    out_.cluster.push_back((int)out_.chunk.size());
    constexpr size_t kPiece = (kBaHTable - 1) / 3;
    for (size_t q = 0; q < be_.size(); q += kPiece) {
      const size_t k = std::min(kPiece, be_.size() - q);
      table(be_.data() + q, k, nullptr, 0);
      emit(be_.data() + q, k, nullptr, 0, q + k < be_.size() || !he_.empty());
    }
    for (size_t q = 0; q < he_.size(); q += kPiece) {
      const size_t k = std::min(kPiece, he_.size() - q);
      table(nullptr, 0, he_.data() + q, k);
      emit(nullptr, 0, he_.data() + q, k, q + k < he_.size());
    }
  }

 private:
  const BaHLists& l_;
  const Csr &bars_, &hinges_;
  const std::vector<int>&order_, &rank_;  // rank: position of each node in order
  BaHMesh& out_;
  int a_ = 0, b_ = 0;
  std::vector<int> be_, he_, halo_;
  std::vector<int> seen_, place_;  // per node: the last table that took it as halo, and its position there
  int tables_ = 0;
  std::vector<std::vector<int>> code_, id_;  // per own node

  bool own(int n) const { return rank_[n] >= a_ && rank_[n] < b_; }

  // Elements that touch an own node, ascending.
  void collect(const Csr& c, const std::vector<int>& e, int K, std::vector<int>& out) {
    out.clear();
    for (int i = a_; i < b_; i++) {
      const int n = order_[i];
      for (int q = c.ptr[n]; q < c.ptr[n + 1]; q++) {
        const int el = c.idx[q] / K, corner = c.idx[q] % K;
        bool first = true;  // from its first own corner only
        for (int k = 0; k < corner; k++) first = first && !own(e[(size_t)el * K + k]);
        if (first) out.push_back(el);
      }
    }
    std::sort(out.begin(), out.end());
  }

  // The other nodes of the elements (halo_); false if the table would be too long.
  bool table(const int* be, size_t nb, const int* he, size_t nh) {
    halo_.clear();
    tables_++;
    auto take = [&](const std::vector<int>& e, int K, const int* el, size_t n) {
      for (size_t q = 0; q < n; q++)
        for (int k = 0; k < K; k++) {
          const int nd = e[(size_t)el[q] * K + k];
          if (own(nd) || seen_[nd] == tables_) continue;
          seen_[nd] = tables_;
          halo_.push_back(nd);
        }
    };
    take(*l_.bar, 2, be, nb);
    take(*l_.hinge, 4, he, nh);
    std::sort(halo_.begin(), halo_.end());
    for (size_t i = 0; i < halo_.size(); i++) place_[halo_[i]] = (b_ - a_) + (int)i;
    return (b_ - a_) + halo_.size() <= (size_t)kBaHTable;
  }

  int position(int n) const { return own(n) ? rank_[n] - a_ : place_[n]; }

  // The codes collected per own node, as entries; returns the entries per node.
  int entries(std::vector<BaHCodes>& codes, uint16_t pad) const {
    const int nOwn = b_ - a_;
    size_t most = 0;
    for (int i = 0; i < nOwn; i++) most = std::max(most, code_[i].size());
    const size_t n = (most + 3) / 4, k0 = codes.size();
    codes.resize(k0 + n * nOwn, BaHCodes{{pad, pad, pad, pad}});
    for (int i = 0; i < nOwn; i++)
      for (size_t q = 0; q < code_[i].size(); q++) codes[k0 + (q / 4) * nOwn + i].c[q % 4] = (uint16_t)code_[i][q];
    return (int)n;
  }

  void clear() {
    code_.resize(b_ - a_);
    id_.resize(b_ - a_);
    for (auto& c : code_) c.clear();
    for (auto& c : id_) c.clear();
  }

  void bars(const int* el, size_t n, BaHChunk& c) {
    clear();
    for (size_t q = 0; q < n; q++) {
      const int* nd = &(*l_.bar)[(size_t)el[q] * 2];
      const int pos[2] = {position(nd[0]), position(nd[1])};
      for (int k = 0; k < 2; k++)
        if (pos[k] < c.nOwn) {
          code_[pos[k]].push_back(pos[1 - k] << 1 | k);
          id_[pos[k]].push_back(el[q]);
        }
    }
    const size_t k0 = out_.bcode.size();
    c.nBarCode = entries(out_.bcode, kBaHNoBar);
    out_.barId.resize(4 * out_.bcode.size(), 0);
    for (int i = 0; i < c.nOwn; i++)
      for (size_t q = 0; q < id_[i].size(); q++) out_.barId[4 * (k0 + (q / 4) * c.nOwn + i) + q % 4] = id_[i][q];
  }

  void hinges(const int* el, size_t n, BaHChunk& c) {
    clear();
    c.nHinge = (int)n;
    c.nHingeOwn = 0;
    for (size_t q = 0; q < n; q++) c.nHingeOwn += own((*l_.hinge)[(size_t)el[q] * 4]);
    const size_t r0 = out_.hingeId.size();
    out_.hingeId.resize(r0 + n);
    out_.hinge.resize((r0 + n) * 4);
    int at[2] = {0, c.nHingeOwn};  // next counted and next other record
    for (size_t q = 0; q < n; q++) {
      const int* nd = &(*l_.hinge)[(size_t)el[q] * 4];
      const int p = at[own(nd[0]) ? 0 : 1]++;
      out_.hingeId[r0 + p] = el[q];
      for (int k = 0; k < 4; k++) {
        const int pos = position(nd[k]);
        out_.hinge[(r0 + p) * 4 + k] = (uint16_t)pos;
        if (pos < c.nOwn) code_[pos].push_back(bah_slot(p, k));
      }
    }
    c.nHingeCode = entries(out_.hcode, kBaHNoHinge);
  }

  void emit(const int* be, size_t nb, const int* he, size_t nh, int more) {
    BaHChunk c{};
    c.node0 = (uint32_t)out_.node.size();
    c.hinge0 = (uint32_t)out_.hingeId.size();
    c.bcode0 = (uint32_t)out_.bcode.size();
    c.hcode0 = (uint32_t)out_.hcode.size();
    c.own0 = a_;
    c.nOwn = b_ - a_;
    c.nNode = c.nOwn + (int)halo_.size();
    c.more = more;
    out_.node.insert(out_.node.end(), order_.begin() + a_, order_.begin() + b_);
    out_.node.insert(out_.node.end(), halo_.begin(), halo_.end());
    bars(be, nb, c);
    hinges(he, nh, c);
    out_.chunk.push_back(c);
  }
};

// The tables of all clusters; ord from order(coords, m).
inline BaHMesh build(const BaHLists& l, const std::vector<int>& ord, int m) {
  const int n = l.nnode;
  const Csr bars(n, *l.bar), hinges(n, *l.hinge);
  std::vector<int> rank(n);
  for (int i = 0; i < n; i++) rank[ord[i]] = i;
  const int np = std::max(1, std::min(m, threads_for(n)));
  std::vector<BaHMesh> part(np);
  ranges(m, np, [&](int p, int m0, int m1) {
    Builder b(l, bars, hinges, ord, rank, part[p]);
    for (int k = m0; k < m1; k++) {
      const int a = (int)((long long)n * k / m), e = (int)((long long)n * (k + 1) / m);
      if (e > a) b.add(a, e);
    }
  });
  size_t most = 0;  // longest table: offsets have 32 bits
  for (auto& p : part) most += std::max({p.node.size(), p.hingeId.size(), p.bcode.size(), p.hcode.size()});
  if (most > UINT32_MAX) throw std::invalid_argument("BarAndHinge: the mesh has too many elements.");
  if (np == 1) return std::move(part[0]);
  BaHMesh out;
  for (auto& p : part) {
    const int chunk0 = (int)out.chunk.size();
    for (auto c : p.chunk) {
      c.node0 += (uint32_t)out.node.size();
      c.hinge0 += (uint32_t)out.hingeId.size();
      c.bcode0 += (uint32_t)out.bcode.size();
      c.hcode0 += (uint32_t)out.hcode.size();
      out.chunk.push_back(c);
    }
    for (int c : p.cluster) out.cluster.push_back(chunk0 + c);
    auto join = [](auto& to, auto& from) {
      to.insert(to.end(), from.begin(), from.end());
      std::remove_reference_t<decltype(from)>().swap(from);
    };
    join(out.node, p.node);
    join(out.hinge, p.hinge);
    join(out.barId, p.barId);
    join(out.hingeId, p.hingeId);
    join(out.bcode, p.bcode);
    join(out.hcode, p.hcode);
  }
  return out;
}

}  // namespace bah_mesh
}  // namespace minim_amd
