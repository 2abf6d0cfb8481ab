// Kernel instantiations of the fused step for D3Q27.
#include "lbm_step_impl.h"

namespace lbm {
KernelFn pick_kernel_d3q27(int storage, int coll, bool mask, int mode, bool flat) {
  return pick_kernel<D3Q27>(storage, coll, mask, mode, flat);
}
}  // namespace lbm
