// common.hpp -- shared device/host helpers for the minim_amd HIP library.
//
// Conventions used by every kernel in this library:
//  * vectors are flat arrays of T (double or float) resident in HBM; the
//    PhaseField layout is AoS, index = site * nFluid + fluid, site = (x*Ny+y)*Nz+z;
//  * every reduction accumulates in FP64, per thread, then per wavefront
//    (64 lanes, shuffles), then per block (LDS), then across blocks in a fixed
//    order by a second, small kernel (or, for small launches of the tiled
//    PhaseField kernel, by the last block) -- results are bitwise reproducible;
//  * kernels are compiled with -ffp-contract=off: every product is rounded
//    before it is added, as in the reference's element-wise vector operators.
#pragma once

#include <hip/hip_runtime.h>

#include <cstddef>
#include <cstdint>
#include <stdexcept>
#include <string>

#include "arrival.hpp"

namespace minim_amd {

constexpr int kBlock = 256;          // threads per block (4 wavefronts of 64)
constexpr int kWave = 64;
constexpr int kMaxRedBlocks = 8192;  // upper bound on blocks of any reducing launch
constexpr int kMaxDots = 96;         // upper bound on values reduced by one launch
constexpr int kSelfBlocks = kWave;    // largest launch that finishes its own reduction
static_assert(kSelfBlocks <= (int)kArrivals, "one lane and one arrival per block");
// Result slot of a deferred validity flag (Potential::gradientDeferred): the
// last one, written by that launch and read by the caller's next fetch.
constexpr int kDeferSlot = kMaxDots - 1;

enum Prec : int { F64 = 0, F32 = 1 };

inline size_t prec_bytes(int p) { return p == F64 ? 8 : 4; }

struct HipError : std::runtime_error {
  explicit HipError(const std::string& s) : std::runtime_error(s) {}
};

#define MINIM_HIP_CHECK(expr)                                                                  \
  do {                                                                                         \
    hipError_t _e = (expr);                                                                    \
    if (_e != hipSuccess) {                                                                    \
      (void)hipGetLastError(); /* reported here, not by the next launch's check */             \
      throw ::minim_amd::HipError(std::string("HIP error ") + hipGetErrorString(_e) + " at " + \
                                  __FILE__ + ":" + std::to_string(__LINE__) + " (" #expr ")"); \
    }                                                                                          \
  } while (0)

// Barrier that orders LDS traffic only: waits for this wave's LDS operations,
// not for its outstanding global loads and stores.
__device__ __forceinline__ void lds_barrier() { asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory"); }

// 1 / v by the hardware's estimate and Newton's iteration: within an ulp.
__device__ __forceinline__ float newton_rcp(float v) {
  const float r = __builtin_amdgcn_rcpf(v);
  return __builtin_fmaf(__builtin_fmaf(-v, r, 1.0f), r, r);
}
__device__ __forceinline__ double newton_rcp(double v) {
  double r = __builtin_amdgcn_rcp(v);
  r = __builtin_fma(__builtin_fma(-v, r, 1.0), r, r);
  return __builtin_fma(__builtin_fma(-v, r, 1.0), r, r);
}

// ---------------------------------------------------------------- reductions
// Sum K doubles over the 64 lanes of a wavefront.
template <int K>
__device__ inline void wave_sum(double (&v)[K]) {
#pragma unroll
  for (int off = kWave / 2; off > 0; off >>= 1) {
#pragma unroll
    for (int k = 0; k < K; k++) v[k] += __shfl_xor(v[k], off, kWave);
  }
}

// Block-wide sum of K doubles; the result is valid in thread 0 only.
// lds must hold (kBlock/kWave)*K doubles.
template <int K>
__device__ inline void block_sum(double (&v)[K], double* lds) {
  wave_sum<K>(v);
  const int lane = threadIdx.x % kWave, wid = threadIdx.x / kWave;
  if (lane == 0) {
#pragma unroll
    for (int k = 0; k < K; k++) lds[wid * K + k] = v[k];
  }
  __syncthreads();
  if (threadIdx.x == 0) {
#pragma unroll
    for (int k = 0; k < K; k++) {
      double s = lds[k];
      for (int w = 1; w < kBlock / kWave; w++) s += lds[w * K + k];
      v[k] = s;
    }
  }
}

// Scratch for cross-block reductions: K rows of per-block partials and the
// final result (device).
//
// Many blocks: two stages, no fences and no atomics.  Each block of the
// producing kernel writes its K partial sums (grid_sum_store), then a small
// kernel with one block per value sums the partials in block order
// (launch_finalize).  A "last block finishes the sum" scheme with a device-scope
// fence in every block writes back the whole L2 each time on CDNA3/4.
//
// Kernels compiled with grid_sum_store<K, true>, for up to kSelfBlocks blocks: the
// last block to arrive does finish the sum, in the same order, in place of
// launch_finalize.  It needs no fence, because the partials themselves bypass the
// L2 (relaxed device-scope atomics): a block waits for its own partials to be
// stored, then counts itself.  It saves a launch (128 x 128 field, 16 blocks:
// energy and gradient 9.4 -> 7.2 us), but the blocks are counted one after the
// other (at 512 blocks an evaluation took 1.5 to 2 us longer than with the second
// launch), and the 23 sums of a Gram pass take as long as the launch they save.
struct RedScratch {
  double* partials;  // [kMaxDots][kMaxRedBlocks], value k of block b at k * gridDim + b
  double* result;    // [kMaxDots]
  double* mirror = nullptr;   // the same values in pinned host memory, for Workspace::fetch
  unsigned* ticket = nullptr; // this launch's arrival counter (arrival.hpp), or null: two stages only
  double* few = nullptr;      // its partials, [kMaxDots][kSelfBlocks]
  double* copy = nullptr;     // value copyK goes there too (a caller's device slot)
  int copyK = -1;
  // The same scratch with results from slot k on.
  RedScratch from(int k) const {
    RedScratch r = *this;
    r.result += k;
    if (mirror) r.mirror += k;
    return r;
  }
  // ... with value k also written to dst (none if null).
  RedScratch copying(int k, double* dst) const {
    RedScratch r = *this;
    r.copy = dst;
    r.copyK = dst ? k : -1;
    return r;
  }
  // ... to dst alone: nothing fetches it (a store to host memory holds the end of
  // the kernel up by about 0.5 us).
  RedScratch only(int k, double* dst) const {
    RedScratch r = copying(k, dst);
    if (dst) r.mirror = nullptr;
    return r;
  }
};

// The last block's part: v (thread 0) are this block's partial sums.
template <int K>
__device__ inline void finish_in_kernel(double (&v)[K], const RedScratch& rs) {
  __shared__ bool last;
  const int nb = gridDim.x;
  if (threadIdx.x == 0) {
#pragma unroll
    for (int k = 0; k < K; k++)
      __hip_atomic_store(&rs.few[(size_t)k * nb + blockIdx.x], v[k], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
    const unsigned w = arrival_weight(nb, blockIdx.x);
    last = arrival_last(__hip_atomic_fetch_add(rs.ticket, w, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT), w);
  }
  __syncthreads();
  if (!last) return;
  // one lane per partial, as finalize_kernel; each wave takes every fourth value
  constexpr int W = kBlock / kWave, J = (K + W - 1) / W;
  const int lane = threadIdx.x % kWave, wid = threadIdx.x / kWave;
  double s[J];
#pragma unroll
  for (int j = 0; j < J; j++) {
    const int k = wid + j * W;
    s[j] = k < K && lane < nb ? __hip_atomic_load(&rs.few[(size_t)k * nb + lane], __ATOMIC_RELAXED,
                                                  __HIP_MEMORY_SCOPE_AGENT)
                              : 0.0;
  }
  wave_sum(s);
  if (lane == 0) {
#pragma unroll
    for (int j = 0; j < J; j++) {
      const int k = wid + j * W;
      if (k >= K) break;
      rs.result[k] = s[j];
      if (rs.mirror) rs.mirror[k] = s[j];
      if (k == rs.copyK) *rs.copy = s[j];
    }
  }
}

// All threads of the (1-D) grid must call this; v is each thread's contribution.
// RS: RedScratch, or Partials for kernels that need no more of it.
struct Partials {
  double* partials;
};
template <int K, bool SELF = false, typename RS>
__device__ inline void grid_sum_store(double (&v)[K], const RS& rs) {
  __shared__ double lds[(kBlock / kWave) * (K > 0 ? K : 1)];
  block_sum<K>(v, lds);
  if constexpr (SELF) {
    finish_in_kernel(v, rs);
  } else if (threadIdx.x == 0) {
    const size_t nb = gridDim.x;
#pragma unroll
    for (int k = 0; k < K; k++) rs.partials[(size_t)k * nb + blockIdx.x] = v[k];
  }
}

// Second stage: result[k] = sum over the nb partials of value k, in a fixed
// order (stream-ordered after the producing kernel).  Value maxK, if any, is the
// square root of the largest partial instead (a NaN wins).
void launch_finalize(RedScratch rs, int K, int nb, hipStream_t s, int maxK = -1);

// NaN-propagating maximum
__device__ inline double nan_max(double a, double b) { return (b > a || b != b) ? b : a; }
// Block-wide nan_max; valid in thread 0.  lds must hold kBlock/kWave doubles.
__device__ inline double block_max(double m, double* lds) {
  for (int off = kWave / 2; off > 0; off >>= 1) m = nan_max(m, __shfl_xor(m, off, kWave));
  if (threadIdx.x % kWave == 0) lds[threadIdx.x / kWave] = m;
  __syncthreads();
  for (int w = 0; w < kBlock / kWave; w++) m = nan_max(m, lds[w]);
  return m;
}

// MI355X dispatches consecutive workgroups round-robin over its 8 XCDs, each
// with a private L2.  Remap the hardware block id so that every XCD receives a
// contiguous range of logical blocks: neighbouring tiles (which share halo
// rows) then run on the same XCD and hit the same L2.  A bijection for any nb.
constexpr int kXcd = 8;
__device__ inline int xcd_logical_block(int b, int nb) {
  const int q = nb / kXcd, r = nb % kXcd;
  const int k = b % kXcd, i = b / kXcd;
  return (k < r) ? k * (q + 1) + i : r * (q + 1) + (k - r) * q + i;
}

// Number of blocks for a grid-stride launch over n work items.
inline int grid_blocks(size_t n, int per_thread = 1, int max_blocks = kMaxRedBlocks) {
  size_t threads = (n + per_thread - 1) / per_thread;
  size_t b = (threads + kBlock - 1) / kBlock;
  if (b < 1) b = 1;
  if (b > (size_t)max_blocks) b = max_blocks;
  return (int)b;
}

}  // namespace minim_amd
