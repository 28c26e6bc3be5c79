// Several time steps in one launch: the parameters and host entries of the
// marching kernel (lbm_march.hip) and of the LDS tile kernel (lbm_tile.hip).
#pragma once

#include "lbm_device.hpp"

namespace lbm_dev
{

constexpr uint32_t kMarchMaxSteps = 4;
constexpr uint32_t kFusedMaxSteps = 8;

struct MarchParams
{
    StepParams p;                  // uy_in / uy_out: the outlet history before the first and after the last step
    uint32_t sr[kFusedMaxSteps];   // stochastic-rounding seeds of the steps (0: round to nearest)
    uint32_t strips, segs, rows;   // column strips, row segments, rows per segment
};

// Enqueues `steps` fused time steps from p.src to p.dst (lattices of the same
// placement, boundary data equal in both).
void march_launch(int layout, int storage, uint32_t steps, const MarchParams &m, int cus, hipStream_t stream);

// The region of nodes of a k_tile_steps block (columns x rows).
enum class TileShape
{
    k16x16,
    k32x16,
    k32x32
};

// The same through k_tile_steps: 2 (steps - 1) less than either extent of the shape.
void tile_launch(int layout, int storage, uint32_t steps, TileShape shape, const MarchParams &m, hipStream_t stream);

}  // namespace lbm_dev
