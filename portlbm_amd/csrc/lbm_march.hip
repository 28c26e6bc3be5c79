// Up to four time steps of the two-lattice algorithms in one pass over the
// lattice (nptl.hpp:116-141 and lptl.hpp:112-137 step by step, the same fields
// bit for bit).
//
// A one-step kernel is bound by HBM: it moves the whole state once per step,
// at the rate of a device copy.  Here a wave owns a strip of columns (one
// 8-byte word of every direction per lane: 1 node in FP64, 2 in FP32, 4 in
// 16-bit storage) and walks up a segment of rows.  It loads each row once
// (stage 0) and keeps, for every stage k < T, the last rows of step k's
// populations in registers: stage k + 1 works one row behind and pulls from
// them, its x neighbours arriving by a one-lane shift across the wave (DPP).
// Only stage T's row is stored, to the other lattice.  Neighbouring strips
// overlap by four halo lanes on each side and segments by T rows, which are
// computed twice.  No barrier and, in the stream layout, no LDS.
//
// 56 of 64 lanes store: 56 * 8 bytes are whole 64-byte segments in every
// layout, and four halo lanes allow T = 4.  Eight halo lanes (whole 128-byte
// lines, 48 of 64) measured 151.8 against 139.6 us per step, stores that pass
// through L2 instead of non-temporal ones 155, contiguous strips per XCD 140
// to 144 (reads -10 %: traffic is no longer the bound).
//
// us per step, 8192 x 2048 porous channel, one step per launch -> T = 4
// (T = 2, 3 in between: FP64 stream 239, 168):
//            stream          collision       bundle
//   FP64     383 -> 139      362 -> 151      366 -> 151
//   FP32     204 -> 104      235 -> 115      242 -> 116
//   FP16     128 -> 106      177 -> 113      184 -> 113
// (FP16 with stochastic rounding, cylinder channel: 160 -> 122.)
// What bounds it at T = 4 (rocprofv3; stream FP64 / collision FP64 / stream FP32
// / stream FP16): vector instructions take 0.68 / 0.70 / 0.83 / 0.91 of the
// SIMDs' cycles; 1.60 / 1.64 / 1.48 / 1.45 of the two waves that a SIMD's
// registers hold are there, for the last round of waves is ragged; they wait
// 0.22 / 0.26 / 0.17 / 0.11 of their time.  FP64 stream moves 2.65 GB per launch
// (4.7 TB/s).

#include "lbm_march.hpp"

#include <algorithm>
#include <iterator>
#include <utility>

namespace lbm_dev
{

typedef unsigned int u32x2 __attribute__((ext_vector_type(2)));
typedef unsigned int u32x4 __attribute__((ext_vector_type(4)));

constexpr int MARCH_BLOCK = 256;
constexpr int MARCH_HALO = 4;                       // halo lanes on each side of a wave's window
constexpr uint32_t MARCH_NOWHERE = 0xfffffff0u;     // a buffer offset past every row
constexpr int MARCH_OWN = 64 - 2 * MARCH_HALO;      // lanes whose nodes the wave stores

template <int S>
struct Lane
{
    using T = typename Storage<S>::T;
    using C = typename Storage<S>::C;
    static constexpr int N = 8 / int(sizeof(T));  // nodes of a lane: 8 bytes of every direction
    static constexpr int CW = (N + 1) / 2;        // words of their codes
};

__device__ __forceinline__ uint32_t left_word(uint32_t v)
{
    return uint32_t(__builtin_amdgcn_update_dpp(0, int(v), 0x138, 0xf, 0xf, true));  // wave_shr:1
}
__device__ __forceinline__ uint32_t right_word(uint32_t v)
{
    return uint32_t(__builtin_amdgcn_update_dpp(0, int(v), 0x130, 0xf, 0xf, true));  // wave_shl:1
}

// a where m is set, else b (v_bfi_b32)
__device__ __forceinline__ uint32_t pick(uint32_t m, uint32_t a, uint32_t b)
{
    uint32_t r;
    asm("v_bfi_b32 %0, %1, %2, %3" : "=v"(r) : "v"(m), "v"(a), "v"(b));
    return r;
}

// the values of the nodes one to the left (cx = 1) or right (cx = -1)
template <int N>
__device__ __forceinline__ u32x2 shifted(u32x2 v, int cx)
{
    if (cx == 0)
        return v;
    if constexpr (N == 1)
        return cx > 0 ? u32x2{left_word(v.x), left_word(v.y)} : u32x2{right_word(v.x), right_word(v.y)};
    else if constexpr (N == 2)
        return cx > 0 ? u32x2{left_word(v.y), v.x} : u32x2{v.y, right_word(v.x)};
    else
        return cx > 0 ? u32x2{__builtin_amdgcn_alignbit(v.x, left_word(v.y), 16), __builtin_amdgcn_alignbit(v.y, v.x, 16)}
                      : u32x2{__builtin_amdgcn_alignbit(v.y, v.x, 16),
                              __builtin_amdgcn_alignbit(right_word(v.x), v.y, 16)};
}

template <int S>
__device__ __forceinline__ typename Storage<S>::C value_of(u32x2 v, int i)
{
    if constexpr (S == LBM_STORE_F64)
        return __builtin_bit_cast(double, v);
    else if constexpr (S == LBM_STORE_F32)
        return __uint_as_float(i ? v.y : v.x);
    else
    {
        const uint32_t w = i < 2 ? v.x : v.y;
        if constexpr (S == LBM_STORE_F16_SHIFTED)
            return float(__builtin_bit_cast(_Float16, uint16_t(i & 1 ? w >> 16 : w)));
        else
            return __uint_as_float(i & 1 ? w & 0xffff0000u : w << 16);
    }
}

template <int S>
__device__ __forceinline__ u32x2 pack_of(const typename Storage<S>::T (&t)[Lane<S>::N])
{
    return __builtin_bit_cast(u32x2, t);
}

template <int S>
__device__ __forceinline__ typename Storage<S>::C left_value(typename Storage<S>::C v)
{
    if constexpr (S == LBM_STORE_F64)
    {
        const u32x2 w = __builtin_bit_cast(u32x2, v);
        return __builtin_bit_cast(double, u32x2{left_word(w.x), left_word(w.y)});
    }
    else
        return __uint_as_float(left_word(__float_as_uint(v)));
}

// What a row holds anywhere in the wave's window, so that the work for it
// is skipped where it does not occur.
constexpr uint32_t ROW_FLUID = 1, ROW_GHOST = 2, ROW_BOUNCE = 4, ROW_OUTLET = 8;

// The row buffers of a level rotate through three roles: in three copies of
// the loop body without a move, or with moves in one.
template <int S>
constexpr int march_phases()
{
    return Lane<S>::N == 4 ? 1 : 3;
}

template <int L>
using MarchLds = u32x4[2][L == LBM_LAYOUT_STREAM ? 1 : 320];  // a wave's two row slots (not used in the stream layout)

// One wave: column strip `strip`, rows y0 to y1 - 1 of the lattice that p
// describes.
template <int L, int S, int T>
__device__ __forceinline__ void march_wave(const StepParams &p, const uint32_t (&sr)[kFusedMaxSteps], uint32_t strip,
                                           int y0, int y1, MarchLds<L> &lds)
{
    using E = typename Storage<S>::T;
    using C = typename Storage<S>::C;
    constexpr int N = Lane<S>::N, CW = Lane<S>::CW;
    constexpr int K = L == LBM_LAYOUT_COLLISION ? 9 : (L == LBM_LAYOUT_BUNDLE ? 3 : 1), NA = 9 / K;
    constexpr int VA = 64 * K / 2;  // 16-byte vectors of a window in one array
    auto lds_of = [&](int j) { return lds[j & 1]; };  // the slot of row j
    auto wave_sync = [] { __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront"); };
    const int lane = int(threadIdx.x & 63u);
    const int Hx = int(p.Hx), Vx = int(p.Vx);
    const int xw = 1 + int(strip) * (MARCH_OWN * N) - MARCH_HALO * N;  // the window's first column
    const int x = xw + lane * N;
    const bool in_range = x <= Hx - 1 && x + N - 1 >= 0;
    const bool owned = lane >= MARCH_HALO && lane < 64 - MARCH_HALO;
    const int jb = max(y0 - T, 0), je = y1 - 1 + T;
    const E *src = static_cast<const E *>(p.src);
    E *dst = static_cast<E *>(p.dst);

    // Codes: the ghost columns never update; lanes off the lattice count as solid
    uint32_t keep[CW], add[CW];
#pragma unroll
    for (int w = 0; w < CW; ++w)
    {
        keep[w] = add[w] = 0u;
#pragma unroll
        for (int h = 0; h < 2 && 2 * w + h < N; ++h)
        {
            const int xi = x + 2 * w + h;
            const bool inner = xi >= 1 && xi <= Hx - 2;
            keep[w] |= (in_range ? (inner ? 0xffffu : uint32_t(LBM_CODE_SOLID)) : 0u) << (16 * h);
            add[w] |= (in_range ? 0u : uint32_t(LBM_CODE_SOLID)) << (16 * h);
        }
    }
    // rho_ref differences of the pulls from x - 1 and x + 1, times the two weights (16-bit forms)
    float rl[N], rr[N], rc[N];
#pragma unroll
    for (int i = 0; i < N; ++i)
    {
        rl[i] = rr[i] = 0.f;
        rc[i] = 1.f;
        if constexpr (shifted_storage<S>())
        {
            const uint32_t xi = uint32_t(min(max(x + i, 0), Hx - 1));
            const Rt3 r3 = rt3_of<S>(p.ref_in, xi);
            rl[i] = r3.rel(1);
            rr[i] = r3.rel(-1);
            rc[i] = r3.own();
        }
    }

    // bytes between direction arrays; opaque, so that nine row addresses are
    // stepped through and not kept
    auto array_bytes = [&]() -> size_t {
        size_t n = size_t(p.S) * (K * uint32_t(sizeof(E)));
        asm volatile("" : "+s"(n));
        return n;
    };
    u32x2 buf[T][3][9] = {}, last_row[9] = {};
    uint32_t code[T + 1][CW] = {}, rowf[T + 1] = {};
    C uy[T][N] = {}, uy_row[T][N] = {};  // stage k's jy: of its latest row, of the row before (stage k + 1's)

    // Lanes right of the lattice and rows above it load the last column's lane
    // and the last row again (their codes make them solid), so that no load
    // depends on a branch.
    const int last = (Hx - 1 - xw) / N;  // the last lane that holds a column of the lattice
    const uint32_t lp = uint32_t(int(p.X0) + xw + min(lane, last) * N);  // place in a row; X0 + xw >= 0
    const uint32_t wp = uint32_t(int(p.X0) + xw);                        // the window's first place
    u32x2 pre2[L == LBM_LAYOUT_STREAM ? 9 : 1] = {};
    uint32_t pcode[CW] = {};
    auto fetch = [&](int j) {
        const uint32_t y = uint32_t(min(j, Vx - 1));
        const uint16_t *cp = p.code + size_t(y) * p.P + lp;
        if constexpr (N == 1)
            pcode[0] = *cp;
        else if constexpr (N == 2)
            pcode[0] = *reinterpret_cast<const uint32_t *>(cp);
        else
        {
            const u32x2 v = *reinterpret_cast<const u32x2 *>(cp);
            pcode[0] = v.x;
            pcode[1] = v.y;
        }
        const char *row = reinterpret_cast<const char *>(src) + (size_t(y) * p.P + wp) * (K * sizeof(E));
        const size_t dir = array_bytes();
        if constexpr (L == LBM_LAYOUT_STREAM)
        {
#pragma unroll
            for (int d = 0; d < 9; ++d, row += dir)
                pre2[d] = *reinterpret_cast<const u32x2 *>(row + uint32_t(min(lane, last)) * 8u);
        }
        else
        {
            // the window's 64 * 72 bytes as 288 16-byte vectors, VA per array
            int ln = lane;  // opaque: the five offsets are computed per row
            asm volatile("" : "+v"(ln));
            const int top = int((uint32_t(min(last, 63)) + 1u) * (8u * K) - 1u) / 16;  // an array's last vector
#pragma unroll
            for (int r = 0; r < 5; ++r)
            {
                int v = ln + 64 * r;  // of all arrays
                const char *at = row;
                if constexpr (L == LBM_LAYOUT_BUNDLE)
                {
                    if (r == 1)  // lanes 32 .. 63 begin the second array
                    {
                        at += ln < 32 ? size_t(0) : dir;
                        v -= ln < 32 ? 0 : VA;
                    }
                    else if (r > 1)
                    {
                        at += r == 2 ? dir : 2 * dir;
                        v -= r == 2 ? VA : 2 * VA;
                    }
                }
                __builtin_amdgcn_global_load_lds(
                    reinterpret_cast<const __attribute__((address_space(1))) void *>(
                        reinterpret_cast<uintptr_t>(at + uint32_t(min(v, top)) * 16u)),
                    (__attribute__((address_space(3))) void *)(lds_of(j) + 64 * r), 16, 0, 0);
            }
        }
    };
    // row j into level 0: elements q, K + q, ... of a lane's K N elements of
    // array a are direction K a + q of its nodes
    auto arrive = [&](u32x2(&to)[9], int j) {
        if constexpr (L == LBM_LAYOUT_STREAM)
        {
#pragma unroll
            for (int d = 0; d < 9; ++d)
                to[d] = pre2[d];
        }
        else
        {
            // The copies of row j into LDS are older than the stores of the row
            // emitted since (at least STORES on every row: one per 64 vectors
            // of an array, as many again where the lattice ends inside a
            // vector), and vector memory operations complete in order: they
            // have landed once at most that many are in flight.
            constexpr int STORES = L == LBM_LAYOUT_COLLISION ? 4 : 6;
            asm volatile("s_waitcnt vmcnt(%0)" ::"n"(STORES) : "memory");
            const u32x4 *stage_lds = lds_of(j);
#pragma unroll
            for (int ar = 0; ar < NA; ++ar)
            {
                const u32x2 *l = reinterpret_cast<const u32x2 *>(stage_lds) + ar * (64 * K) + lane * K;
                E e[K * N];
#pragma unroll
                for (int w = 0; w < K; ++w)
                {
                    const u32x2 v = l[w];
                    __builtin_memcpy(e + w * N, &v, 8);
                }
#pragma unroll
                for (int q = 0; q < K; ++q)
                {
                    E t[N];
#pragma unroll
                    for (int i = 0; i < N; ++i)
                        t[i] = e[K * i + q];
                    to[K * ar + q] = pack_of<S>(t);
                }
            }
            wave_sync();
        }
    };

    auto stage = [&](auto kc, auto ph, int j) {
        constexpr int k = decltype(kc)::value, P0 = decltype(ph)::value;
        const int r = j - k;
        if (r < max(y0 - (T - k), 0) || r > min(y1 - 1 + (T - k), Vx - 1))
        {
#pragma unroll
            for (int d = 0; d < 9; ++d)  // never used
                if constexpr (k < T)
                    buf[k][P0][d] = __builtin_nondeterministic_value(buf[k][P0][d]);
                else
                    last_row[d] = __builtin_nondeterministic_value(last_row[d]);
            return;
        }
        const u32x2(&nw)[9] = buf[k - 1][P0];
        const u32x2(&A)[9] = buf[k - 1][(P0 + 2) % 3];
        const u32x2(&B)[9] = buf[k - 1][(P0 + 1) % 3];
        const uint32_t(&cd)[CW] = code[k];
        const uint32_t rf = rowf[k];
        auto bit = [&](int i, uint32_t mask) -> bool { return cd[i / 2] & (mask << (16 * (i & 1))); };
        u32x2 g[9];
#pragma unroll
        for (int d = 0; d < 9; ++d)
            g[d] = shifted<N>(d < 3 ? nw[d] : (d < 6 ? A[d] : B[d]), cx_of(d));
        C f[N][9];
        if (rf & ROW_BOUNCE)
        {
            // all ones where a node's pull of direction d bounces back
            auto ones = [&](int i, int d) -> uint32_t {
                return uint32_t(__builtin_amdgcn_sbfe(int(cd[i / 2]), 16u * (i & 1) + d, 1u));
            };
#pragma unroll
            for (int d = 0; d < 9; ++d)
            {
                if (d == 4)
                    continue;
                u32x2 m;
                if constexpr (N == 1)
                    m.x = m.y = ones(0, d);
                else if constexpr (N == 2)
                    m = u32x2{ones(0, d), ones(1, d)};
                else
                    m = u32x2{pick(0xffffu, ones(0, d), ones(1, d)), pick(0xffffu, ones(2, d), ones(3, d))};
                g[d] = u32x2{pick(m.x, A[8 - d].x, g[d].x), pick(m.y, A[8 - d].y, g[d].y)};
#pragma unroll
                for (int i = 0; i < N; ++i)
                {
                    f[i][d] = value_of<S>(g[d], i);
                    if constexpr (shifted_storage<S>())
                        if (cx_of(d) != 0)
                            f[i][d] += __uint_as_float(__float_as_uint(shift_of(d, cx_of(d) > 0 ? rl[i] : rr[i])) &
                                                       ~ones(i, d));
                }
            }
        }
        else
        {
#pragma unroll
            for (int d = 0; d < 9; ++d)
#pragma unroll
                for (int i = 0; i < N; ++i)
                {
                    f[i][d] = value_of<S>(g[d], i);
                    if constexpr (shifted_storage<S>())
                        if (cx_of(d) != 0)
                            f[i][d] += shift_of(d, cx_of(d) > 0 ? rl[i] : rr[i]);
                }
        }
#pragma unroll
        for (int i = 0; i < N; ++i)
            f[i][4] = value_of<S>(A[4], i);
        if (rf & ROW_OUTLET)
        {
#pragma unroll
            for (int i = 0; i < N; ++i)
            {
                const C ul = i ? uy_row[k - 1][i - 1] : left_value<S>(uy_row[k - 1][N - 1]);
                const uint32_t lw = left_word(cd[CW - 1]);
                const uint32_t lc = N == 1 ? lw : (i == 0 ? lw >> 16 : cd[(i - 1) / 2] >> (16 * ((i - 1) & 1)));
                if (bit(i, LBM_CODE_OUTLET))
                {
                    const C u = (k > 1 && (lc & LBM_CODE_UY_SOURCE)) ? ul : C(p.uy_in[r]);
                    if constexpr (shifted_storage<S>())
                        zou_he_outlet<C>(f[i], C(p.rho_out) - rc[i], u);
                    else
                        zou_he_outlet<C, Storage<S>::kPromote>(f[i], C(p.rho_out), u);
                }
            }
        }
        E t[N][9];
        C rhos[N], jxs[N], jys[N], usqs[N];
        collide_nodes<C, Storage<S>::kPromote, Storage<S>::kFull, N>(f, C(p.omega), rhos, jxs, jys, usqs);
#pragma unroll
        for (int i = 0; i < N; ++i)
        {
            const C rho = rhos[i], jx = jxs[i], jy = jys[i], usq = usqs[i];
            if constexpr (k < T)
                uy[k][i] = N == 4 ? clamp_output(jy, p.nan_protection) : jy;
            else if ((p.write_macros || bit(i, LBM_CODE_UY_SOURCE)) && owned && bit(i, LBM_CODE_FLUID))
            {
                const uint32_t c = (cd[i / 2] >> (16 * (i & 1))) & 0xffffu;
                if constexpr (shifted_storage<S>())
                    write_moments<C, double>(p, c, uint32_t(x + i), uint32_t(r), double(rc[i]) + double(rho), jx, jy,
                                             usq);
                else
                    write_moments<C>(p, c, uint32_t(x + i), uint32_t(r), rho, jx, jy, usq);
            }
            node_bits<S>(f[i], uint32_t(r) * p.P + lp + uint32_t(i), sr[k - 1], t[i], 0.f);
        }
        // The next stage reads them only beside an outlet.  (With four nodes a
        // lane the clamp of all four at once costs registers: 252 against 245
        // ms over 2000 steps; with fewer it saves 1 %.)
        if constexpr (k < T && N < 4)
            if (rf & ROW_OUTLET)
#pragma unroll
                for (int i = 0; i < N; ++i)
                    uy[k][i] = clamp_output(uy[k][i], p.nan_protection);
        u32x2 out[9];
#pragma unroll
        for (int d = 0; d < 9; ++d)
        {
            E e[N];
#pragma unroll
            for (int i = 0; i < N; ++i)
                e[i] = t[i][d];
            out[d] = pack_of<S>(e);
        }
        if constexpr (k < T)
        {
            // nodes that are neither fluid nor solid keep their populations
            if (rf & ROW_GHOST)
            {
                asm volatile("");  // a branch: few rows have such nodes
#pragma unroll
                for (int d = 0; d < 9; ++d)
                {
                    E e[N], o[N];
                    __builtin_memcpy(e, &out[d], 8);
                    __builtin_memcpy(o, &A[d], 8);
#pragma unroll
                    for (int i = 0; i < N; ++i)
                        e[i] = bit(i, LBM_CODE_FLUID) ? e[i] : o[i];
                    out[d] = pack_of<S>(e);
                }
            }
#pragma unroll
            for (int d = 0; d < 9; ++d)
                buf[k][P0][d] = out[d];
        }
        else
#pragma unroll
            for (int d = 0; d < 9; ++d)
                last_row[d] = out[d];
    };

    // The stores of stage T's row.  They are issued on every row, lanes with
    // nothing to store at an offset past the row (the hardware drops them): a
    // wait for the next row's loads can then leave them in flight (nine in the
    // stream layout, at least STORES in the others); stores behind a branch
    // would have to be waited for.
    auto emit = [&](auto ph, int j) {
        constexpr int P0 = decltype(ph)::value;
        const int r = j - T;
        const uint32_t(&cd)[CW] = code[T];
        const uint32_t rf = r >= y0 ? rowf[T] : 0u;
        auto bit = [&](int i, uint32_t mask) -> bool { return cd[i / 2] & (mask << (16 * (i & 1))); };
        auto words = [&](uint32_t mask) -> u32x2 {  // all ones over the nodes with a bit of mask
            if constexpr (N == 1)
                return bit(0, mask) ? u32x2{~0u, ~0u} : u32x2{0u, 0u};
            else if constexpr (N == 2)
                return u32x2{bit(0, mask) ? ~0u : 0u, bit(1, mask) ? ~0u : 0u};
            else
                return u32x2{(bit(0, mask) ? 0xffffu : 0u) | (bit(1, mask) ? 0xffff0000u : 0u),
                             (bit(2, mask) ? 0xffffu : 0u) | (bit(3, mask) ? 0xffff0000u : 0u)};
        };
        const u32x2 fm = words(LBM_CODE_FLUID);
        const unsigned long long m = __ballot(owned && (fm.x | fm.y));
        int ln = lane;  // opaque: what follows is computed per row and not kept in registers across them
        asm volatile("" : "+v"(ln));
        const u32x2 nm = words(LBM_CODE_FLUID | LBM_CODE_SOLID);
        if (L != LBM_LAYOUT_STREAM || N > 1 ? (rf & ROW_GHOST) != 0u : false)
        {
#pragma unroll
            for (int d = 0; d < 9; ++d)  // nodes that are neither fluid nor solid keep their populations
                last_row[d] = (last_row[d] & fm) | (buf[T - 1][(P0 + 2) % 3][d] & ~nm);
        }
        else
        {
#pragma unroll
            for (int d = 0; d < 9; ++d)
                last_row[d] &= fm;
        }
        char *row = reinterpret_cast<char *>(dst) + (size_t(uint32_t(max(r, 0))) * p.P + wp) * (K * sizeof(E));
        constexpr int window = 64 * 8 * K;  // bytes of an array's row that the wave may store to
        const size_t dir = array_bytes();
        if constexpr (L == LBM_LAYOUT_STREAM)
        {
            // the lane's eight-lane segment holds a fluid node, and the lane a node of the lattice
            const int g0 = ((ln - MARCH_HALO) & ~7) + MARCH_HALO;
            const bool write = owned && lane <= last && (nm.x | nm.y) && ((m >> (g0 & 63)) & 0xffull) && rf;
            const uint32_t off = write ? uint32_t(ln) * 8u : MARCH_NOWHERE;
#pragma unroll
            for (int d = 0; d < 9; ++d, row += dir)
                __builtin_amdgcn_raw_buffer_store_b64(
                    last_row[d], __builtin_amdgcn_make_buffer_rsrc(row, 0, window, 0x00027000), int(off), 0,
                    2 /* nt */);
        }
        else
        {
            u32x4 *stage_lds = lds_of(j);
#pragma unroll
            for (int ar = 0; ar < NA; ++ar)
            {
                u32x2 *l = reinterpret_cast<u32x2 *>(stage_lds) + ar * (64 * K) + ln * K;
                E e[K * N];
#pragma unroll
                for (int q = 0; q < K; ++q)
                {
                    E t[N];
                    __builtin_memcpy(t, &last_row[K * ar + q], 8);
#pragma unroll
                    for (int i = 0; i < N; ++i)
                        e[K * i + q] = t[i];
                }
#pragma unroll
                for (int w = 0; w < K; ++w)
                {
                    u32x2 v;
                    __builtin_memcpy(&v, e + w * N, 8);
                    l[w] = v;
                }
            }
            wave_sync();
            // Of every array the owned lanes' 56 * 8 K bytes, in whole 64-byte
            // segments that hold a fluid node; the lattice ends after `lanes`
            // of them.
            const unsigned long long mo = rf ? m >> MARCH_HALO : 0ull;
            const int lanes = min(MARCH_OWN, (Hx - 2 - xw) / N + 1 - MARCH_HALO);
            const uint32_t bytes = uint32_t(lanes) * (8u * K);
            row += MARCH_HALO * 8 * K;
#pragma unroll
            for (int ar = 0; ar < NA; ++ar, row += dir)
            {
                const auto rsrc = __builtin_amdgcn_make_buffer_rsrc(row, 0, window, 0x00027000);
                const u32x4 *l = stage_lds + ar * VA + MARCH_HALO * K / 2;
                constexpr int VO = MARCH_OWN * K / 2, NV = (VO + 63) / 64;  // the owned vectors, per lane
                u32x4 w[NV];
                uint32_t off[NV];
#pragma unroll
                for (int n = 0; n < NV; ++n)
                {
                    const uint32_t v = uint32_t(64 * n + ln), seg64 = v / 4u;
                    const uint32_t la = seg64 * 8u / K, lb = (seg64 * 8u + 7u) / K;  // its first and last lane
                    const bool any = (mo >> (la & 63u)) & ((2ull << (lb - la)) - 1ull);
                    w[n] = l[v < uint32_t(VO) ? v : 0u];
                    off[n] = any && v * 16u < bytes ? v * 16u : MARCH_NOWHERE;
                }
#pragma unroll
                for (int n = 0; n < NV; ++n)
                    __builtin_amdgcn_raw_buffer_store_b128(
                        w[n], rsrc, int(off[n] != MARCH_NOWHERE && off[n] + 16u > bytes ? MARCH_NOWHERE : off[n]), 0,
                        2 /* nt */);
                if (bytes % 16u)  // the lattice ends inside a vector
#pragma unroll
                    for (int n = 0; n < NV; ++n)
                        __builtin_amdgcn_raw_buffer_store_b64(
                            u32x2{w[n].x, w[n].y}, rsrc,
                            int(off[n] != MARCH_NOWHERE && off[n] + 16u > bytes ? off[n] : MARCH_NOWHERE), 0,
                            2 /* nt */);
            }
            wave_sync();
        }
    };

    auto body = [&](auto ph, int j) {
        constexpr int P0 = decltype(ph)::value;
        // row j arrives
#pragma unroll
        for (int m = T; m > 0; --m)
        {
            rowf[m] = rowf[m - 1];
#pragma unroll
            for (int w = 0; w < CW; ++w)
                code[m][w] = code[m - 1][w];
        }
        const bool edge = j == 0 || j >= Vx - 1;
        bool fluid = false, ghost = false, bounce = false, outlet = false;
#pragma unroll
        for (int w = 0; w < CW; ++w)
        {
            uint32_t c = (pcode[w] & keep[w]) | add[w];
            if (edge)
                c &= uint32_t(LBM_CODE_SOLID) * 0x10001u;
            code[0][w] = c;
            fluid |= c & (LBM_CODE_FLUID * 0x10001u);
            bounce |= c & (LBM_CODE_BOUNCE_MASK * 0x10001u);
            outlet |= c & (LBM_CODE_OUTLET * 0x10001u);
            ghost |= !(c & (LBM_CODE_FLUID | LBM_CODE_SOLID)) ||
                     (N > 1 && !(c & ((LBM_CODE_FLUID | LBM_CODE_SOLID) << 16)));
        }
        rowf[0] = (__any(fluid) ? ROW_FLUID : 0u) | (__any(ghost) ? ROW_GHOST : 0u) |
                  (__any(bounce) ? ROW_BOUNCE : 0u) | (__any(outlet) ? ROW_OUTLET : 0u);
        arrive(buf[0][P0], j);
        fetch(j + 1);
#pragma unroll
        for (int k = 1; k < T; ++k)
#pragma unroll
            for (int i = 0; i < N; ++i)
                uy_row[k][i] = uy[k][i];
        [&]<int... K>(std::integer_sequence<int, K...>) {
            (stage(std::integral_constant<int, K + 1>{}, ph, j), ...);
        }(std::make_integer_sequence<int, T>{});
        emit(ph, j);
    };

    fetch(jb);
    if constexpr (L != LBM_LAYOUT_STREAM)
        asm volatile("s_waitcnt vmcnt(0)" ::: "memory");  // the first row has no stores after it
    if constexpr (march_phases<S>() == 1)
    {
        for (int j = jb; j <= je; ++j)
        {
            body(std::integral_constant<int, 0>{}, j);
#pragma unroll
            for (int m = 0; m < T; ++m)
#pragma unroll
                for (int d = 0; d < 9; ++d)
                {
                    buf[m][1][d] = buf[m][2][d];
                    buf[m][2][d] = buf[m][0][d];
                }
        }
    }
    else
    {
        for (int j = jb; j <= je;)
        {
            body(std::integral_constant<int, 0>{}, j);
            if (++j > je)
                break;
            body(std::integral_constant<int, 1>{}, j);
            if (++j > je)
                break;
            body(std::integral_constant<int, 2>{}, j);
            ++j;
        }
    }
}

template <int L, int S, int T>
__global__ __launch_bounds__(MARCH_BLOCK, 2) void k_march(MarchParams a)
{
    __shared__ MarchLds<L> lds[MARCH_BLOCK / 64];
    const uint32_t in_block = __builtin_amdgcn_readfirstlane(threadIdx.x / 64);
    const uint32_t wave = blockIdx.x * (MARCH_BLOCK / 64) + in_block;
    if (wave >= a.strips * a.segs)
        return;
    const uint32_t seg = wave / a.strips, strip = wave - seg * a.strips;
    const int y0 = 1 + int(seg * a.rows), y1 = min(y0 + int(a.rows), int(a.p.Vx) - 1);
    march_wave<L, S, T>(a.p, a.sr, strip, y0, y1, lds[in_block]);
}

// The time of `waves` waves of `rows` rows each, in row visits.  A wave costs
// rows + T + 1 of them; w waves come to each SIMD, which holds two at a time.
// One left over runs alone and takes about 1.4 of its share of a pair; an
// uneven end costs about a third of a wave.  (FP32 stream, 8192 x 2048,
// T = 4: rows 76 / 50 / 38 / 30 / 25, that is 2 / 3 / 4 / 5 / 6 waves,
// 106.7 / 117.4 / 102.5 / 112.3 / 103.4 us per step.)
double march_cost(uint64_t waves, double rows, uint32_t steps, int cus)
{
    const uint64_t simds = uint64_t(std::max(cus, 1)) * 4u, each = (waves + simds - 1u) / simds;
    return (double(each) + (each % 2u ? 0.4 : 0.0)) * (rows + steps + 1.0) + 0.3 * rows;
}

template <int L, int S, int T>
static void launch(MarchParams m, int cus, hipStream_t stream)
{
    constexpr uint32_t own = uint32_t(MARCH_OWN * Lane<S>::N);
    m.strips = (m.p.Hx - 2u + own - 1u) / own;
    const uint32_t inner = m.p.Vx - 2u;
    const uint32_t simds = uint32_t(std::max(cus, 1)) * 4u;
    double best = 0.0;
    for (uint32_t w = 1; w <= 12u; ++w)
    {
        const uint32_t most = std::max(1u, w * simds / m.strips);
        const uint32_t rows = std::max(4u, (inner + most - 1u) / most);
        const double cost = march_cost(m.strips * ((inner + rows - 1u) / rows), rows, T, cus);
        if (w == 1u || cost < best)
        {
            best = cost;
            m.rows = rows;
        }
    }
    m.segs = (inner + m.rows - 1u) / m.rows;
    const uint32_t blocks = (m.strips * m.segs + MARCH_BLOCK / 64 - 1u) / (MARCH_BLOCK / 64);
    hipLaunchKernelGGL((k_march<L, S, T>), dim3(blocks), dim3(MARCH_BLOCK), 0, stream, m);
}

// The same for the domains of a batch: each wave has its own domain, strip and rows.
template <int S, int T>
__global__ __launch_bounds__(MARCH_BLOCK, 2) void k_batch_march(BatchFused a, uint32_t waves)
{
    __shared__ MarchLds<LBM_LAYOUT_STREAM> lds[1];
    const uint32_t wave = blockIdx.x * (MARCH_BLOCK / 64) + __builtin_amdgcn_readfirstlane(threadIdx.x / 64);
    if (wave >= waves)
        return;
    const BatchPart part = a.parts[wave];
    const StepParams p = batch_params<S>(a, part.dom);
    constexpr uint32_t sr[kFusedMaxSteps] = {};
    march_wave<LBM_LAYOUT_STREAM, S, T>(p, sr, part.x, int(part.y0), int(part.y1), lds[0]);
}

// What of the columns that marching waves own, or of the nodes that blocks
// own, lies in the domains.
static double march_share(size_t elem, const FuseExtent *domains, size_t count)
{
    const uint32_t own = uint32_t(MARCH_OWN) * uint32_t(8u / elem);
    double in = 0.0, all = 0.0;
    for (size_t d = 0; d < count; ++d)
    {
        in += double(domains[d].w) * domains[d].h;
        all += double((domains[d].w + own - 1u) / own * own) * domains[d].h;
    }
    return in / all;
}
static double tile_share(uint32_t w, uint32_t h, uint32_t steps, const FuseExtent *domains, size_t count)
{
    const uint32_t ow = w - 2u * (steps - 1u), oh = h - 2u * (steps - 1u);
    double in = 0.0, all = 0.0;
    for (size_t d = 0; d < count; ++d)
    {
        in += double(domains[d].w) * domains[d].h;
        all += double((domains[d].w + ow - 1u) / ow * ow) * double((domains[d].h + oh - 1u) / oh * oh);
    }
    return in / all;
}

FusePlan plan_fusion(size_t elem, int layout, const FuseExtent *domains, size_t count)
{
    const FusePlan march{kMarchMaxSteps, false, TileShape::k32x32}, one{};
    uint64_t nodes = 0;
    for (size_t d = 0; d < count; ++d)
        nodes += uint64_t(domains[d].w) * domains[d].h;
    if (count == 1u && domains->h <= 4u && layout == LBM_LAYOUT_STREAM && nodes >= 100000u)
        return one;
    if (count == 1u && (domains->h <= 10u ? nodes > 36000u : domains->h <= 12u && nodes >= 300000u))
        return FusePlan{domains->h <= 10u ? 4u : 3u, true, TileShape::k32x16};
    // 16-bit tiles and how much of them is used
    struct
    {
        FusePlan plan;
        double share;
    } tiles[3] = {{{3u, true, TileShape::k32x16}, tile_share(32, 16, 3, domains, count)},
                  {{4u, true, TileShape::k32x16}, tile_share(32, 16, 4, domains, count) / 1.15},
                  {{5u, true, TileShape::k32x32}, tile_share(32, 32, 5, domains, count) / 1.04}};
    const auto &fit = *std::max_element(std::begin(tiles), std::end(tiles),
                                        [](const auto &a, const auto &b) { return a.share < b.share; });
    // whether the stream layout's one-step kernel has full blocks of 256 columns
    const bool full = count == 1u && layout == LBM_LAYOUT_STREAM &&
                      domains->w >= 0.85 * ((domains->w + 255u) / 256u * 256u);
    if (nodes >= (elem == 8 ? 1500000u : (elem == 4 ? 2500000u : 3500000u)))
    {
        const double share = march_share(elem, domains, count);
        if (elem >= 4)
        {
            if (share >= 0.5)
                return march;
        }
        else
        {
            const double marched = share >= 0.6 ? 5.7 / share + 8e6 / double(nodes) : 1e3, tiled = 9.9 / fit.share;
            if (full && 8.2 < 0.95 * std::min(marched, tiled))
                return one;
            if (marched <= tiled)
                return march;
        }
    }
    if (nodes <= 36000u)
        return FusePlan{5u, true, TileShape::k16x16};
    if (nodes <= (elem == 8 ? 300000u : 500000u))
        return FusePlan{nodes <= 200000u ? 6u : 5u, true, TileShape::k32x32};
    if (elem >= 4)
        return FusePlan{elem == 8 ? 4u : 3u, true, TileShape::k32x16};
    return full && fit.share < 0.6 ? one : fit.plan;
}

uint32_t march_strips(int storage, uint32_t inner_width)
{
    const uint32_t own = uint32_t(MARCH_OWN) * (storage == LBM_STORE_F64 ? 1u : (storage == LBM_STORE_F32 ? 2u : 4u));
    return (inner_width + own - 1u) / own;
}

template <int S>
static void batch_steps(uint32_t steps, const BatchFused &a, uint32_t waves, hipStream_t stream)
{
    const dim3 grid((waves + MARCH_BLOCK / 64 - 1u) / (MARCH_BLOCK / 64)), block(MARCH_BLOCK);
    switch (steps)
    {
    case 2: hipLaunchKernelGGL((k_batch_march<S, 2>), grid, block, 0, stream, a, waves); break;
    case 3: hipLaunchKernelGGL((k_batch_march<S, 3>), grid, block, 0, stream, a, waves); break;
    default: hipLaunchKernelGGL((k_batch_march<S, 4>), grid, block, 0, stream, a, waves); break;
    }
}

void batch_march_launch(int storage, uint32_t steps, const BatchFused &a, uint32_t waves, hipStream_t stream)
{
    switch (storage)
    {
    case LBM_STORE_F64: batch_steps<LBM_STORE_F64>(steps, a, waves, stream); break;
    case LBM_STORE_F32: batch_steps<LBM_STORE_F32>(steps, a, waves, stream); break;
    case LBM_STORE_F16_SHIFTED: batch_steps<LBM_STORE_F16_SHIFTED>(steps, a, waves, stream); break;
    default: batch_steps<LBM_STORE_BF16_SHIFTED>(steps, a, waves, stream); break;
    }
}

template <int L, int S>
static void launch_steps(uint32_t steps, const MarchParams &m, int cus, hipStream_t stream)
{
    switch (steps)
    {
    case 2: launch<L, S, 2>(m, cus, stream); break;
    case 3: launch<L, S, 3>(m, cus, stream); break;
    default: launch<L, S, 4>(m, cus, stream); break;
    }
}

template <int L>
static void launch_storage(int storage, uint32_t steps, const MarchParams &m, int cus, hipStream_t stream)
{
    switch (storage)
    {
    case LBM_STORE_F64: launch_steps<L, LBM_STORE_F64>(steps, m, cus, stream); break;
    case LBM_STORE_F32: launch_steps<L, LBM_STORE_F32>(steps, m, cus, stream); break;
    case LBM_STORE_F16_SHIFTED: launch_steps<L, LBM_STORE_F16_SHIFTED>(steps, m, cus, stream); break;
    default: launch_steps<L, LBM_STORE_BF16_SHIFTED>(steps, m, cus, stream); break;
    }
}

void march_launch(int layout, int storage, uint32_t steps, const MarchParams &m, int cus, hipStream_t stream)
{
    switch (layout)
    {
    case LBM_LAYOUT_COLLISION: launch_storage<LBM_LAYOUT_COLLISION>(storage, steps, m, cus, stream); break;
    case LBM_LAYOUT_STREAM: launch_storage<LBM_LAYOUT_STREAM>(storage, steps, m, cus, stream); break;
    default: launch_storage<LBM_LAYOUT_BUNDLE>(storage, steps, m, cus, stream); break;
    }
}

}  // namespace lbm_dev
