// Several time steps of the two-lattice algorithms in one launch, for lattices
// that the launch and the latency of one step bound rather than HBM: a
// 256 x 64 channel took 3.6 to 5.3 us per step with one step per launch.
//
// A block holds a region of W x H nodes, one per thread.  The first step pulls
// from the source lattice; every further step pulls from the LDS copy of the
// step before (two copies in turn, one barrier per step) and is correct one
// node further in, so T steps yield the region without T - 1 nodes at each
// edge.  The fields equal the one-step kernels' bit for bit.
//
// The region's size trades recomputed edges against blocks: 16 x 16 at T = 5
// keeps 8 x 8 of 256 nodes, but gives a 256 x 64 lattice 256 blocks, one per
// compute unit, and a step then takes the latency of one node's pulls and
// collision.  Measured us per step, one step per launch -> here: 256 x 64
// FP64 stream 3.82 -> 1.25, collision 5.24 -> 1.30; 512 x 128 4.53 -> 2.12;
// 1024 x 256 10.2 -> 4.7, collision 9.3 -> 5.0; 2048 x 512 29.5 -> 12.6.  The
// marching kernel takes over where HBM bounds a step (plan_fusion).
//
// What bounds it (rocprofv3): at 1024 x 256 in FP64 the 473 blocks of 147 KB of
// LDS, one per compute unit, go in two rounds; compute units are busy 0.60 of
// the time, vector instructions take 0.27 of the SIMDs' cycles, waves wait 0.47
// of theirs.  At 1999 x 501 in BF16 vector instructions take 0.69.

#include "lbm_march.hpp"

namespace lbm_dev
{

// One block: stores the nodes from (x0, y0) on that lie at least `halo` nodes
// inside its region (steps <= halo + 1).
template <int L, int S, int W, int H>
__device__ __forceinline__ void tile_block(const StepParams &p, const uint32_t (&sr)[kFusedMaxSteps], uint32_t steps,
                                           int halo, int x0, int y0)
{
    using E = typename Storage<S>::T;
    using C = typename Storage<S>::C;
    constexpr int NT = W * H;
    __shared__ E pop[2][9][NT];
    __shared__ C uy[2][H];
    __shared__ uint16_t codes[NT];
    const E *src = static_cast<const E *>(p.src);
    const int tid = int(threadIdx.x), tx = tid % W, ty = tid / W;
    const int x = x0 - halo + tx, y = y0 - halo + ty;
    const bool inside = x >= 0 && y >= 0 && x < int(p.Hx) && y < int(p.Vx);
    const bool inner = x >= 1 && y >= 1 && x <= int(p.Hx) - 2 && y <= int(p.Vx) - 2;
    const uint32_t pn = inside ? place(uint32_t(x), uint32_t(y), p.P, p.X0) : 0u;
    const uint32_t code = inside ? p.code[pn] : uint32_t(LBM_CODE_SOLID);
    const bool fluid = inner && (code & LBM_CODE_FLUID);
    const int depth = min(min(tx, W - 1 - tx), min(ty, H - 1 - ty));  // steps that stay correct here: depth + 1
    codes[tid] = uint16_t(fluid ? code : 0u);
    const Rt3 r3 = rt3_of<S>(p.ref_in, inside ? uint32_t(x) : 0u);
    if (inside && !fluid && !(code & LBM_CODE_SOLID))
    {
        // neither fluid nor solid: constant populations
#pragma unroll
        for (int d = 0; d < 9; ++d)
            pop[0][d][tid] = pop[1][d][tid] = src[at<L>(pn, uint32_t(d), p.S)];
    }
    C fs[1][9];
    C(&f)[9] = fs[0];
    if (fluid)
        pull<L, S>(src, pn, code, p.P, p.S, f, r3);
    for (uint32_t k = 1;; ++k)
    {
        const uint32_t b = k & 1u;  // step k leaves its populations in pop[b]
        if (fluid && depth >= (k < steps ? int(k) - 1 : halo))
        {
            if (k > 1u)
            {
#pragma unroll
                for (int d = 0; d < 9; ++d)
                {
                    const bool bb = (code >> d) & 1u;
                    const int dd = bb ? 8 - d : d;
                    const int n = bb ? tid : tid - cx_of(d) - cy_of(d) * W;
                    f[d] = Storage<S>::load(&pop[b ^ 1u][0][0], uint32_t(dd * NT + n), dd, bb ? 0.f : r3.rel(cx_of(d)));
                }
            }
            if (code & LBM_CODE_OUTLET)
            {
                const C u = k > 1u && (codes[max(tid - 1, 0)] & LBM_CODE_UY_SOURCE) ? uy[b ^ 1u][ty] : C(p.uy_in[y]);
                if constexpr (shifted_storage<S>())
                    zou_he_outlet<C>(f, C(p.rho_out) - r3.own(), u);
                else
                    zou_he_outlet<C, Storage<S>::kPromote>(f, C(p.rho_out), u);
            }
            C rhos[1], jxs[1], jys[1], usqs[1];
            collide_nodes<C, Storage<S>::kPromote, Storage<S>::kFull, 1>(fs, C(p.omega), rhos, jxs, jys, usqs);
            const C rho = rhos[0], jx = jxs[0], jy = jys[0], usq = usqs[0];
            E t[9];
            node_bits<S>(f, pn, sr[k - 1u], t, 0.f);
            if (k < steps)
            {
                if (code & LBM_CODE_UY_SOURCE)
                    uy[b][ty] = clamp_output(jy, p.nan_protection);
#pragma unroll
                for (int d = 0; d < 9; ++d)
                    pop[b][d][tid] = t[d];
            }
            else
            {
                if constexpr (shifted_storage<S>())
                    write_moments<C, double>(p, code, uint32_t(x), uint32_t(y), double(r3.own()) + double(rho), jx, jy,
                                             usq);
                else
                    write_moments<C>(p, code, uint32_t(x), uint32_t(y), rho, jx, jy, usq);
                E *dst = static_cast<E *>(p.dst);
#pragma unroll
                for (int d = 0; d < 9; ++d)
                    dst[at<L>(pn, uint32_t(d), p.S)] = t[d];
            }
        }
        if (k == steps)
            break;
        __syncthreads();
    }
}

template <int L, int S, int W, int H>
__global__ __launch_bounds__(W * H) void k_tile_steps(MarchParams a, uint32_t steps)
{
    const int halo = int(steps) - 1;
    tile_block<L, S, W, H>(a.p, a.sr, steps, halo, 1 + int(blockIdx.x) * (W - 2 * halo),
                           1 + int(blockIdx.y) * (H - 2 * halo));
}

// The same for the domains of a batch: each block has its own domain and first node.
template <int S, int W, int H>
__global__ __launch_bounds__(W * H) void k_batch_tiles(BatchFused a, uint32_t steps, int halo)
{
    const BatchPart part = a.parts[blockIdx.x];
    const StepParams p = batch_params<S>(a, part.dom);
    constexpr uint32_t sr[kFusedMaxSteps] = {};
    tile_block<LBM_LAYOUT_STREAM, S, W, H>(p, sr, steps, halo, int(part.x), int(part.y0));
}

template <int L, int S, int W, int H>
static void launch_shape(uint32_t steps, const MarchParams &m, hipStream_t stream)
{
    const uint32_t ow = W - 2u * (steps - 1u), oh = H - 2u * (steps - 1u);
    hipLaunchKernelGGL((k_tile_steps<L, S, W, H>), dim3((m.p.Hx - 2u + ow - 1u) / ow, (m.p.Vx - 2u + oh - 1u) / oh),
                       dim3(W * H), 0, stream, m, steps);
}

template <int L, int S>
static void launch(uint32_t steps, TileShape shape, const MarchParams &m, hipStream_t stream)
{
    switch (shape)
    {
    case TileShape::k16x16: launch_shape<L, S, 16, 16>(steps, m, stream); break;
    case TileShape::k32x16: launch_shape<L, S, 32, 16>(steps, m, stream); break;
    default: launch_shape<L, S, 32, 32>(steps, m, stream); break;
    }
}

void tile_launch(int layout, int storage, uint32_t steps, TileShape shape, const MarchParams &m,
                 hipStream_t stream)
{
    auto by_layout = [&](auto st) {
        constexpr int S = decltype(st)::value;
        switch (layout)
        {
        case LBM_LAYOUT_COLLISION: launch<LBM_LAYOUT_COLLISION, S>(steps, shape, m, stream); break;
        case LBM_LAYOUT_STREAM: launch<LBM_LAYOUT_STREAM, S>(steps, shape, m, stream); break;
        default: launch<LBM_LAYOUT_BUNDLE, S>(steps, shape, m, stream); break;
        }
    };
    switch (storage)
    {
    case LBM_STORE_F64: by_layout(std::integral_constant<int, LBM_STORE_F64>{}); break;
    case LBM_STORE_F32: by_layout(std::integral_constant<int, LBM_STORE_F32>{}); break;
    case LBM_STORE_F16_SHIFTED: by_layout(std::integral_constant<int, LBM_STORE_F16_SHIFTED>{}); break;
    default: by_layout(std::integral_constant<int, LBM_STORE_BF16_SHIFTED>{}); break;
    }
}

template <int S>
static void batch_shape(uint32_t steps, int halo, TileShape shape, const BatchFused &a, uint32_t blocks,
                        hipStream_t stream)
{
    switch (shape)
    {
    case TileShape::k16x16:
        hipLaunchKernelGGL((k_batch_tiles<S, 16, 16>), dim3(blocks), dim3(256), 0, stream, a, steps, halo);
        break;
    case TileShape::k32x16:
        hipLaunchKernelGGL((k_batch_tiles<S, 32, 16>), dim3(blocks), dim3(512), 0, stream, a, steps, halo);
        break;
    default:
        hipLaunchKernelGGL((k_batch_tiles<S, 32, 32>), dim3(blocks), dim3(1024), 0, stream, a, steps, halo);
        break;
    }
}

void batch_tile_launch(int storage, uint32_t steps, uint32_t halo, TileShape shape, const BatchFused &a,
                       uint32_t blocks, hipStream_t stream)
{
    switch (storage)
    {
    case LBM_STORE_F64: batch_shape<LBM_STORE_F64>(steps, int(halo), shape, a, blocks, stream); break;
    case LBM_STORE_F32: batch_shape<LBM_STORE_F32>(steps, int(halo), shape, a, blocks, stream); break;
    case LBM_STORE_F16_SHIFTED: batch_shape<LBM_STORE_F16_SHIFTED>(steps, int(halo), shape, a, blocks, stream); break;
    default: batch_shape<LBM_STORE_BF16_SHIFTED>(steps, int(halo), shape, a, blocks, stream); break;
    }
}

}  // namespace lbm_dev
