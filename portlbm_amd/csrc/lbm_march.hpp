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

// How several steps go into one launch: by marching waves, or in LDS tiles of
// a region of columns x rows.
enum class TileShape
{
    k16x16,
    k32x16,
    k32x32
};
struct FusePlan
{
    uint32_t steps = 1;  // per launch, at most
    bool tiles = false;
    TileShape shape = TileShape::k32x32;
};

// Small lattices are bound by the launch itself and then by the latency of a
// step: blocks hold a region of nodes in LDS for several steps
// (k_tile_steps), the region small enough that every compute unit gets one.
// Large lattices are bound by HBM: marching waves read each row once
// (k_march).  us per step on porous channels (FP64 stream / FP32 stream /
// FP16 collision), one step per launch, then the shapes around the choice:
//   256 x 64     3.8 / 3.6 / 4.6     16x16 T 5: 1.25 / 1.23 / 1.45    32x16 T 6: 1.42 / 1.30 / 1.44
//   512 x 128    4.5 / 3.8 / 5.0     32x32 T 6: 2.12 / 1.75 / 1.73    16x16 T 5: 2.41 / 2.04 / 1.99
//   1024 x 256   10.2 / 6.1 / 6.3    32x32 T 5: 4.69 / 3.73 / 3.65    32x16 T 4: 4.38 / 3.82 / 3.90
//   2048 x 512   29.5 / 16.1 / 16.3  32x16 T 4: 12.6 / 10.7 / 11.1    march:     14.6 / 13.0 / 20.3
//   4096 x 1024  112 / 55.8 / 48.9   32x16 T 4: 59.0 / 42.9 / 38.7    march:     45.4 / 32.7 / 37.5
// and at the lines between the shapes (bundle layout, FP64 / FP32 / BF16;
// "1.8e5": inner nodes):
//   1.8e5  32x32 T 6: 3.77 / 3.18 / 3.27   T 5: 4.06 / 3.38 / 3.42
//   2.6e5  32x32 T 6: 5.06 / 4.20 / 4.16   T 5: 4.52 / 3.59 / 3.74
//   3.9e5  32x32 T 5: 6.39 / 4.96 / 5.00   32x16 T 4: 5.81 / 4.98 / 5.12 (FP64 collision 7.12, 6.90)
//   1.0e6  32x16 T 3: 11.7 / 10.1 / 10.4   32x16 T 4: 12.2 / 10.7 / 11.1   march: 14.8 / 13.9 / 18.0
//   2.0e6  32x16 T 3: 23.2 / 18.5 / 19.1   32x16 T 4: 22.9 / 19.8 / 20.5   march: 24.8 / 19.8 / 24.1
//   3.0e6  32x16 T 3: 39.0 / 27.2 / 28.0   march: 35.1 / 27.2 / 27.5 (3001 x 997 for nsol, FP32: 31.0, 28.4)
// FP64 marches from 1.5e6: at 2.0e6 the collision layout takes 24.7 marched
// and 27.3 in tiles.
inline FusePlan plan_fusion(size_t elem, uint64_t nodes)
{
    if (nodes >= (elem == 8 ? 1500000u : (elem == 4 ? 2500000u : 3500000u)))
        return FusePlan{kMarchMaxSteps, false, TileShape::k32x32};
    if (nodes <= 36000u)
        return FusePlan{5u, true, TileShape::k16x16};
    if (nodes <= (elem == 8 ? 300000u : 500000u))
        return FusePlan{nodes <= 200000u ? 6u : 5u, true, TileShape::k32x32};
    return FusePlan{elem == 8 ? 4u : 3u, true, TileShape::k32x16};
}

// The first launch of n steps: as few launches as there can be, of nearly the same length.
inline uint32_t first_chunk(const FusePlan &plan, uint32_t n)
{
    const uint32_t launches = (n + plan.steps - 1u) / plan.steps;
    return (n + launches - 1u) / launches;
}

// Enqueues `steps` fused time steps from p.src to p.dst (lattices of the same
// placement, boundary data equal in both).
void march_launch(int layout, int storage, uint32_t steps, const MarchParams &m, int cus, hipStream_t stream);

// The same through k_tile_steps: 2 (steps - 1) less than either extent of the shape.
void tile_launch(int layout, int storage, uint32_t steps, TileShape shape, const MarchParams &m, hipStream_t stream);

// ---- batched domains --------------------------------------------------------
constexpr uint32_t kBatchX0 = 15;  // x = 1 starts a 16-node (64 B in FP32) segment

struct BatchDom
{
    uint64_t lat;   // element offset of the domain's lattice in each arena
    uint32_t code;  // node offset in the code arena
    uint32_t res;   // offset in the result arena (4 * D doubles)
    uint32_t uy;    // offset in the outlet-history arena (2 * V doubles)
    uint32_t H, V, P, S, D;
    uint32_t tile_w;
    double omega, rho_out;
};

// A wave's strip x and rows y0 .. y1 - 1 (k_batch_march), or the first node
// (x, y0) that a block stores (k_batch_tiles).
struct BatchPart
{
    uint32_t dom, x, y0, y1;
};

struct BatchFused
{
    const BatchDom *doms;
    const BatchPart *parts;
    const void *src;
    void *dst;
    const uint16_t *codes;
    double *res;
    double *uy;
    int parity;  // half of the outlet history that is read
    uint32_t write_macros;
    uint32_t nan_protection;
    const float *ones;  // rho_ref of the 16-bit forms: 1 in every column
};

// The lattice of domain d, unexpanded, in the stream layout.
template <int S>
__device__ __forceinline__ StepParams batch_params(const BatchFused &a, uint32_t d)
{
    using T = typename Storage<S>::T;
    const BatchDom dm = a.doms[d];
    StepParams p{};
    p.src = static_cast<const T *>(a.src) + dm.lat;
    p.dst = static_cast<T *>(a.dst) + dm.lat;
    p.code = a.codes + dm.code;
    p.rho = a.res + dm.res;
    p.jx = p.rho + dm.D;
    p.jy = p.rho + 2u * size_t(dm.D);
    p.jabs = p.rho + 3u * size_t(dm.D);
    p.uy_in = a.uy + dm.uy + uint32_t(a.parity) * dm.V;
    p.uy_out = a.uy + dm.uy + uint32_t(1 - a.parity) * dm.V;
    p.omega = dm.omega;
    p.rho_out = dm.rho_out;
    p.H = p.Hx = dm.H;
    p.V = p.Vx = dm.V;
    p.P = dm.P;
    p.X0 = kBatchX0;
    p.S = dm.S;
    p.write_macros = a.write_macros;
    p.nan_protection = a.nan_protection;
    p.ref_in = p.ref_out = a.ones;
    return p;
}

// Column strips of a domain, the cost model behind the rows of a wave, and
// the launches: `steps` <= kMarchMaxSteps from a.src to a.dst; tiles store
// what stays correct for `halo` + 1 steps (steps <= halo + 1).
uint32_t march_strips(int storage, uint32_t inner_width);
double march_cost(uint64_t waves, double rows, uint32_t steps, int cus);
void batch_march_launch(int storage, uint32_t steps, const BatchFused &a, uint32_t waves, hipStream_t stream);
void batch_tile_launch(int storage, uint32_t steps, uint32_t halo, TileShape shape, const BatchFused &a,
                       uint32_t blocks, hipStream_t stream);

}  // namespace lbm_dev
