// arrival.hpp -- how the blocks of a small launch count themselves, so that the
// last to arrive finishes the launch's sums (common.hpp).  Plain C++ apart from
// the qualifiers, so that it can be checked on the CPU.
//
// Every launch adds kArrivals to its counter in all, whatever its number of
// blocks: block 0 makes up the difference.  The counter is never set back, so a
// launch that finds it at a multiple of kArrivals leaves it at one, also when
// another launch counted on it at the same time (which spoils the sums of those
// two, but no later ones).
#pragma once

#ifndef MINIM_HD
#if defined(__HIPCC__) || defined(__HIP__)
#define MINIM_HD __host__ __device__
#else
#define MINIM_HD
#endif
#endif

namespace minim_amd {

constexpr unsigned kArrivals = 64;  // blocks of a launch, at most

// What block b of nb adds.
MINIM_HD inline unsigned arrival_weight(int nb, int b) { return b == 0 ? kArrivals - (unsigned)(nb - 1) : 1u; }

// The block that adds weight to a count of before is the last of its launch.
MINIM_HD inline bool arrival_last(unsigned before, unsigned weight) { return (before + weight) % kArrivals == 0; }

}  // namespace minim_amd
