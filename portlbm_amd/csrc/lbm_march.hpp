// Several time steps in one launch: the marching kernel's parameters and its
// host entry (lbm_march.hip).
#pragma once

#include "lbm_device.hpp"

namespace lbm_dev
{

constexpr uint32_t kMarchMaxSteps = 4;

struct MarchParams
{
    StepParams p;                  // uy_in / uy_out: the outlet history before the first and after the last step
    uint32_t sr[kMarchMaxSteps];   // stochastic-rounding seeds of the steps (0: round to nearest)
    uint32_t strips, segs, rows;   // column strips, row segments, rows per segment
};

// Enqueues `steps` fused time steps from p.src to p.dst (lattices of the same
// placement, boundary data equal in both).
void march_launch(int layout, int storage, uint32_t steps, const MarchParams &m, int cus, hipStream_t stream);

}  // namespace lbm_dev
