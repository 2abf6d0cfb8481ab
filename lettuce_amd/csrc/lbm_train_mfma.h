// Launchers of the FP32 training kernels on matrix instructions
// (lbm_train_mfma.hip).
#pragma once

#include "lbm_train_cell.h"

namespace lbm {

// blocks of a launch over `cells` cells, each of which writes one vector of
// NPARAM partial sums
int train_mfma_blocks(int64_t cells);
void launch_train_forward_mfma(int32_t stencil, const KParams& p, const TrainArgs& t, hipStream_t s);
void launch_train_backward_mfma(int32_t stencil, const KParams& p, const TrainArgs& t, const float* lam,
                                int gathered, float* mu, float* part, hipStream_t s);

}  // namespace lbm
