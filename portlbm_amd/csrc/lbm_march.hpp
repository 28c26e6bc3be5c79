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
// and at the lines between the shapes (FP64 / FP32 / BF16, bundle layout;
// "1.8e5": inner nodes):
//   1.8e5  32x32 T 6: 3.77 / 3.18 / 3.27   T 5: 4.06 / 3.38 / 3.42
//   2.6e5  32x32 T 6: 5.06 / 4.20 / 4.16   T 5: 4.52 / 3.59 / 3.74
//   3.9e5  32x32 T 5: 6.39 / 4.96 / 5.00   32x16 T 4: 5.81 / 4.98 / 5.12 (FP64 collision 7.12, 6.90)
//   1.05e6 32x16 T 3: 14.7 / 11.5 / 11.6   32x16 T 4: 13.7 / 11.6 / 11.9 (FP64 collision 22.0, 18.7)
//   1.5e6  32x16 T 3: 19.3 / 15.3 / 15.4   32x16 T 4: 19.0 / 16.2 / 16.4   march: 20.8 / 16.9 / 21.2
// (FP64 collision at 1.5e6: 29.6, 25.8, march 20.9).  March against the better
// of T 3 and T 4 (stream, collision, bundle):
//   FP64   2.0e6  25.4 25.5 25.4 : 29.3 34.8 27.7     3.0e6  33.8 35.7 35.5 : 39.4 51.7 40.1
//   FP32   2.25e6 21.7 23.3 23.2 : 21.1 27.0 23.1     2.5e6  23.6 24.9 24.9 : 23.4 29.7 24.6
//          2.75e6 24.7 26.4 25.8 : 26.0 32.5 27.1     3.0e6  26.4 28.1 27.8 : 28.1 35.4 30.0
//   FP16   2.5e6  23.3 24.7 24.2 : 20.9 24.8 23.7     3.0e6  24.5 25.9 25.9 : 25.0 29.2 28.6
//          3.5e6  26.8 29.1 28.8 : 29.0 33.3 32.8     4.2e6  32.4 34.0 33.7 : 34.3 39.9 38.0
//
// All of that is for lattices of some width and height.  A marching wave owns
// 56, 112 or 224 columns (FP64, FP32, 16-bit), a block 22 to 28 columns by 10
// to 26 rows, and what of them lies past the lattice is work for nothing:
// * FP64 and FP32 march where the lattice takes at least half of the waves'
//   columns (1.9e6 nodes 64 wide, 0.57: FP64 36.4, tiles 38.0, FP32 at 3.8e6
//   55.5, 56.8; batches of 16 x 16 domains, 0.14 in FP32).
// * 16-bit lattices compare the us that 1e6 nodes take: marching, 5.7 over the
//   share of the columns and 8 / nodes for a launch's ramp, never below a share
//   of 0.6; tiles, 9.9 over the share of the regions; in the stream layout also
//   one step per launch, 8.2 where the columns fill that kernel's blocks of 256
//   to 0.85 (up to 11 where they do not).  58 x 65000: march 94.6, 32x32 T 5
//   47.7, 32x16 T 3 55.0, one step 58.7; 226 x 65000: 169, 145, 161, 124; 450 x
//   65000: 264, 269, 286, 228; 280 x 65000: 167, 173, 170, 195; 976 domains of
//   64 x 64: 90.2, 48.0, 53.6, 94.4.  Their tiles are 32x16 with T 3 unless T
//   4's rows (65000 x 26: 17.4 : 18.6) or 32x32's columns (113 x 30000: 34.1 :
//   38.6) fit clearly better; where no shape has a share of 0.6 the stream
//   layout takes one step per launch (65000 x 13: 9.6, T 4 11.5, T 3 11.7).
// * Lattices of at most 10 rows take 32x16 tiles with T 4 (10 own rows), of 11
//   or 12 with T 3: 65000 x 6 5.6 / 5.1 / 5.5 us in the stream layout, with the
//   shape for 3.9e5 nodes otherwise 5.7 / 9.4 / 8.9; 40000 x 11 6.3 / 5.3 / 5.5
//   against 7.9 / 6.9 / 7.2.
//   One or two rows between walls in the stream layout leave a step nothing to
//   share: one step per launch (65000 x 3: 3.7 / 3.2 / 3.8, T 4 5.1 / 4.7 / 4.8).
struct FuseExtent
{
    uint32_t w, h;  // inner columns and rows
};

// The plan for one lattice, or for the domains of a batch together.
FusePlan plan_fusion(size_t elem, int layout, const FuseExtent *domains, size_t count);

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
