// Two pull steps per launch for a batch of domains: the sweep of fused_two.hpp
// over tiles of every domain, each workgroup with its own domain's extents,
// relaxation time and force.  The numbers of two launches of the one-step
// batch kernel, bit for bit, from one read and one write of the populations.
// Each lattice instantiates this in its own file (batch_two_q{19,27}.hip).
#pragma once

#include "batch.hpp"
#include "fused_two.hpp"

namespace plb {

namespace {

// One domain as pull2_tile reads its arguments (FusedArgs for a single domain).
template <class T>
struct BatchTileArgs {
    uint32_t X, Y, Z;
    uint64_t pstride;
    T tau, om, omm, F0, F1, F2;
    const FusedBC<T>& bc;
    const T (&wcub)[27][3];
};

template <class T>
struct BatchWalls {
    FusedBC<T> bc;
    T wcub[27][3];
};

template <int Q, int V, bool MOV>
__global__ __launch_bounds__(two_cap(Q, (int)sizeof(typename Prec<V>::S)), 1) void k_batch2(
    const typename Prec<V>::S* __restrict__ A, typename Prec<V>::S* __restrict__ B,
    const BDom<typename Prec<V>::T>* __restrict__ doms, const BTile* __restrict__ tiles,
    BatchWalls<typename Prec<V>::T> w) {
    using T = typename Prec<V>::T;
    const BTile t = tiles[blockIdx.x];
    const BDom<T> D = doms[t.dom];
    const BatchTileArgs<T> a{D.X, D.Y, D.Z, D.ps, D.tau, D.om, D.omm, D.F0, D.F1, D.F2, w.bc, w.wcub};
    pull2_tile<Q, V, 0, MOV, 1, two_split(Q, (int)sizeof(typename Prec<V>::S), false)>(
        A + D.off, B + D.off, nullptr, nullptr, a, t.bx, t.by, t.x0, t.y0, t.z0, t.zc);
}

}  // namespace

template <int Q, int V>
void launch_batch2(const typename Prec<V>::S* A, typename Prec<V>::S* B, const BDom<typename Prec<V>::T>* doms,
                   const BTile* tiles, uint32_t ntiles, const FusedBC<typename Prec<V>::T>& bc, hipStream_t stream) {
    using T = typename Prec<V>::T;
    BatchWalls<T> w;
    w.bc = bc;
    fill_wall_cub<Q, T>(bc, w.wcub);
    const dim3 grid(ntiles), block(two_cap(Q, (int)sizeof(typename Prec<V>::S)));
    if (two_walls(bc, false, (int)sizeof(typename Prec<V>::S)))
        hipLaunchKernelGGL((k_batch2<Q, V, true>), grid, block, 0, stream, A, B, doms, tiles, w);
    else
        hipLaunchKernelGGL((k_batch2<Q, V, false>), grid, block, 0, stream, A, B, doms, tiles, w);
}

#define PLB_BATCH2_INST(Q, V)                                                                                  \
    template void launch_batch2<Q, V>(const typename Prec<V>::S*, typename Prec<V>::S*,                        \
                                      const BDom<typename Prec<V>::T>*, const BTile*, uint32_t,                \
                                      const FusedBC<typename Prec<V>::T>&, hipStream_t);
#define PLB_BATCH2_INST_Q(Q)                                                                       \
    PLB_BATCH2_INST(Q, kF64) PLB_BATCH2_INST(Q, kF32) PLB_BATCH2_INST(Q, kF64A32) PLB_BATCH2_INST(Q, kF32S) \
    PLB_BATCH2_INST(Q, kF16S)

}  // namespace plb
