// The pull step of a 2D cell from global memory, shared by the two kernels
// that keep the following steps in LDS (lbm_tb2d.hip, lbm_tile2d.hip): the
// class ids of the cell and its sources in a first round of loads, the
// populations its rules select in a second.
#pragma once

#include "lbm_step_impl.h"

namespace lbm {
namespace {

// the class ids of a cell and of its pull sources x - e_q (the first load
// round of a masked pull step); cell offsets are in-plane (2D: the grid)
template <class S>
struct PullIds {
  uint32_t c0;
  uint32_t src[S::Q];
};

// (a grid without a class map: every cell is class 0, a plain collision)
template <class S, bool MASK>
__device__ __forceinline__ void load_pull_ids(const KParams& p, int cell, const int (&a1)[3],
                                              const int (&a2)[3], PullIds<S>& ids) {
  if constexpr (!MASK) {
#pragma unroll
    for (int q = 0; q < S::Q; ++q) ids.src[q] = 0;
    ids.c0 = 0;
    return;
  }
  ids.c0 = elem(p.cls, (uint32_t)cell);
#pragma unroll
  for (int q = 1; q < S::Q; ++q) ids.src[q] = elem(p.cls, (uint32_t)nb_in_plane<S>(q, -1, a1, a2));
  ids.src[0] = ids.c0;
}

// The classes' fields the kernel reads per cell, in LDS: flags, op and
// no-stream bits by class id
struct ClassLds {
  uint8_t flags[256];
  uint8_t op[256];
  uint32_t nsm[256];
};

// the second round: the stored value the pull step takes for each
// population (halfway bounce-back: the cell's own opposite population where
// the fluid cell's source is solid; a no-stream bit: the cell's own value).
// Element offsets are 32-bit (the host checks that the array fits).
template <class S, class ST>
__device__ __forceinline__ void load_pull_pops(const KParams& p, int cell, const int (&a1)[3],
                                               const int (&a2)[3], const PullIds<S>& ids,
                                               const ClassLds& cl, typename ST::T (&raw)[S::Q]) {
  using T = typename ST::T;
  const T* fin = (const T*)p.fin;
  const uint32_t flags = cl.flags[ids.c0], nsm = cl.nsm[ids.c0];
  const bool near = (flags & (LBM_CLASS_NEAR_SOLID | LBM_CLASS_SOLID)) == LBM_CLASS_NEAR_SOLID;
  const uint32_t sq = (uint32_t)p.sq;
  if (!__any(near || nsm != 0)) {
    // a wavefront away from boundaries: the plain pull
#pragma unroll
    for (int q = 0; q < S::Q; ++q)
      raw[q] = elem(fin, (uint32_t)q * sq + (uint32_t)nb_in_plane<S>(q, -1, a1, a2));
    return;
  }
  // selects, not branches: every lane reads its sources' flags
#pragma unroll
  for (int q = 0; q < S::Q; ++q) {
    const bool bounce = near & (q != 0) & ((cl.flags[ids.src[q]] & LBM_CLASS_SOLID) != 0);
    const bool own = bounce | (((nsm >> q) & 1u) != 0);
    const uint32_t pop = (uint32_t)(bounce ? S::opp[q] : q) * sq;
    raw[q] = elem(fin, pop + (uint32_t)(own ? cell : nb_in_plane<S>(q, -1, a1, a2)));
  }
}

__device__ __forceinline__ int wrap(int i, int n) { return i < 0 ? i + n : (i >= n ? i - n : i); }

}  // namespace
}  // namespace lbm
