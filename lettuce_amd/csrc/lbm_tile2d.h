// Declarations of the several-step kernel for 2D grids (lbm_tile2d.hip).
#pragma once

#include "lbm_step_impl.h"

namespace lbm {

struct Tile2dParams {
  KParams k;
  int t1, t2;  // the cells a block owns along i1 and i2
  int nt2;     // tiles along i2
  int steps;   // steps of this launch (its stages, with lead or trail)
  int lead;    // the first stage collides without streaming
  int trail;   // the last stage streams without colliding
  int reach;   // cells per step that a cell's value depends on (1, or 2 with
               // a class map)
};
using Tile2dFn = void (*)(const Tile2dParams);

// kernel for (storage codec, collision, with a class map), or nullptr
Tile2dFn pick_tile2d_kernel(int codec, int coll, bool mask);
// dynamic LDS bytes of a block, and the kernel's static ones
int64_t tile2d_lds_bytes(int t1, int t2, int steps, int reach, int storage_bytes, bool mask);
int64_t tile2d_static_lds_bytes();

}  // namespace lbm
