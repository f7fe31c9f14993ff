// Several pull steps per launch for small D2Q9 lattices: the numbers of that
// many k_pull launches, bit for bit.
//
// A D2Q9 lattice of a few thousand to a few hundred thousand cells is done
// with one step in less time than a launch takes, so a step per launch is
// bound by launches.  Here a workgroup owns a tile of OX x OZ cells of the x-z
// plane and takes them `steps` (up to kMultiSteps) steps further: step 1 on the
// tile grown by steps - 1 cells on each side, gathered from the populations in
// memory, each further step on a region one cell smaller all round, gathered
// from the LDS copy of the step before, the last on the tile itself, written to
// the other population array.  Grown cells are computed by several workgroups,
// so none waits for another.  One cell per thread for the whole launch (its
// neighbour mask and seams stay in registers); the LDS copy has two buffers, so
// a step needs one barrier.  256 x 64 cells, 200 steps and the read-out: FP64
// 1,074 -> 321 us; a step takes 1.2 to 1.4 us there, bound by the
// instructions of the two wavefronts per SIMD and by their latency.  Values
// pass through the storage type between steps, as they would through memory.
#pragma once

#include "fused_two.hpp"

namespace plb {

namespace {

__host__ __device__ constexpr int multi_cells(int ox, int oz) {
    return (ox + 2 * (kMultiSteps - 1)) * (oz + 2 * (kMultiSteps - 1));
}
__host__ __device__ constexpr int multi_threads(int ox, int oz) { return (multi_cells(ox, oz) + 63) / 64 * 64; }

// Population k of the cell at index li (rows of GX cells) from the LDS copy of
// the step before: from li - c_k, or the cell's own slot rev(k) where that
// neighbour is not fluid.
template <int K, int V, int NB, int NC>
__device__ inline void multi_gather(typename Prec<V>::T (&f)[9], const typename Prec<V>::S* buf, uint32_t li,
                                    uint32_t GX, uint32_t m, const Seams<uint32_t>& s) {
    if constexpr (K < 9) {
        constexpr int R = rev_k<9>(K);
        const bool solid = NB ? ((m >> R) & 1u) != 0 : pull_wall<9, K>(s);
        const uint32_t moved = (uint32_t)(K * NC) + li - ((uint32_t)Lat<9>::cx(K) + (uint32_t)Lat<9>::cz(K) * GX);
        const uint32_t own = (uint32_t)(R * NC) + li;
        f[K] = Prec<V>::load_raw(buf[solid ? own : moved]);
        multi_gather<K + 1, V, NB, NC>(f, buf, li, GX, m, s);
    }
}

template <int V, int NB, bool MOV, int OX, int OZ>
__global__ __launch_bounds__(multi_threads(OX, OZ)) void k_multi9(const typename Prec<V>::S* __restrict__ A,
                                                                  typename Prec<V>::S* __restrict__ B,
                                                                  const uint32_t* __restrict__ nbmask,
                                                                  FusedArgs<typename Prec<V>::T> a, uint32_t steps) {
    using P = Prec<V>;
    using S = typename P::S;
    using T = typename P::T;
    using I = uint32_t;
    constexpr int NC = multi_cells(OX, OZ);
    __shared__ S buf[2][9 * NC];

    const uint32_t X = a.X, Z = a.Z, h = steps - 1u;
    const uint32_t GX = (uint32_t)OX + 2u * h, GZ = (uint32_t)OZ + 2u * h;
    const uint32_t x0 = blockIdx.x * (uint32_t)OX, z0 = blockIdx.y * (uint32_t)OZ, y = blockIdx.z;
    const uint32_t ix = threadIdx.x % GX, iz = threadIdx.x / GX;
    // wrapped coordinates (a lattice narrower than the grown tile holds some
    // of its cells more than once); threads past the grown tile take any cell
    // and leave every step out
    const uint32_t lx = (h + X - 1u) / X * X, lz = (h + Z - 1u) / Z * Z;
    const uint32_t gx = (x0 + ix + lx - h) % X, gz = (z0 + iz + lz - h) % Z;
    const bool in = iz < GZ;
    const I ps = (I)a.pstride;
    const I c = (gz * a.Y + y) * X + gx;
    const Seams<I> sm = seams<I>(gx, y, gz, a);
    uint32_t m = 0;
    bool self_solid;
    S fv[9];
    constexpr I sz = (I)sizeof(S);
    const I psz = ps * sz;
    const PopBuffers<9, 1> ra(A, psz), rb(B, psz);
    if (NB) {
        m = nbmask[c];
        self_solid = m & 1u;
    } else {
        self_solid = (a.bc.wall_lo[0] && gx == 0) || (a.bc.wall_hi[0] && gx + 1u == X) ||
                     (a.bc.wall_lo[2] && gz == 0) || (a.bc.wall_hi[2] && gz + 1u == Z);
    }
    Seams<I> sb = sm;
    sb.xm *= sz, sb.xp *= sz, sb.ym *= sz, sb.yp *= sz, sb.zm *= sz, sb.zp *= sz;
    gather<9, 0, V, NB, 1, kAll>(fv, ra, A, c * sz, psz, m, sb);
    T f[9];
#pragma unroll
    for (int k = 0; k < 9; ++k) f[k] = P::load_raw(fv[k]);
    const uint32_t li = iz * GX + ix;
    for (uint32_t s = 1;; ++s) {
        // the region of step s: s - 1 cells off the grown tile on each side
        const bool on = in && ix + 1u >= s && ix + s <= GX && iz + 1u >= s && iz + s <= GZ;
        if (on && !self_solid) {
            if (s > 1u) multi_gather<0, V, NB, NC>(f, buf[s & 1u], li, GX, m, sm);
            const T rho = bgk<9, P>(f, a, true);
            if (MOV && a.bc.moving) moving_wall_terms<9, P>(f, rho, sm, a);
        }
        if (s == steps) {
            // the tile's own cells; zeros for those that are not fluid
            const bool own = on && x0 + ix - h < X && z0 + iz - h < Z;
            store_own<9, V, 1>(f, rb, B, own ? c * sz : kNoStore, psz, self_solid);
            return;
        }
        if (on && !self_solid) {
#pragma unroll
            for (int k = 0; k < 9; ++k) buf[(s & 1u) ^ 1u][k * NC + li] = P::store_raw(f[k]);
        }
        lds_barrier();
    }
}

template <int V, int OX, int OZ>
void launch_multi9_tile(const FusedArgs<typename Prec<V>::T>& a, uint32_t steps, bool nb, bool mov,
                        const typename Prec<V>::S* A, typename Prec<V>::S* B, const uint32_t* nbmask,
                        hipStream_t stream) {
    const dim3 grid((a.X + OX - 1) / OX, (a.Z + OZ - 1) / OZ, a.Y), block(multi_threads(OX, OZ));
#define PLB_MULTI(NBv, MVv) \
    hipLaunchKernelGGL((k_multi9<V, NBv, MVv, OX, OZ>), grid, block, 0, stream, A, B, nbmask, a, steps)
    if (nb && mov) PLB_MULTI(1, true);
    else if (nb) PLB_MULTI(1, false);
    else if (mov) PLB_MULTI(0, true);
    else PLB_MULTI(0, false);
#undef PLB_MULTI
}

}  // namespace

template <int V>
void launch_multi9(const FusedArgs<typename Prec<V>::T>& a, uint32_t steps, int tile, bool nb, bool mov,
                   const typename Prec<V>::S* A, typename Prec<V>::S* B, const uint32_t* nbmask,
                   hipStream_t stream) {
    if (tile == 8)
        launch_multi9_tile<V, 8, 8>(a, steps, nb, mov, A, B, nbmask, stream);
    else
        launch_multi9_tile<V, 16, 16>(a, steps, nb, mov, A, B, nbmask, stream);
}

#define PLB_MULTI9_INST(V)                                                                                      \
    template void launch_multi9<V>(const FusedArgs<typename Prec<V>::T>&, uint32_t, int, bool, bool,            \
                                   const typename Prec<V>::S*, typename Prec<V>::S*, const uint32_t*,          \
                                   hipStream_t);

}  // namespace plb
