// What the batched one-step (batch.hip) and two-step (batch_two.hpp) kernels share.
#pragma once

#include "fastdiv.hpp"
#include "state.hpp"

namespace plb {

// One domain of a batch.
template <class T>
struct BDom {
    uint32_t X, Y, Z, N;
    FastDiv dX, dY;  // division by X and Y (cell -> coordinates)
    uint64_t off;    // element offset of population 0 in the pool
    uint64_t ps;     // elements between populations
    T tau, om, omm, F0, F1, F2;
};

// One workgroup's share of a two-step launch: the planes [z0, z0 + zc) of the
// bx x by cells at (x0, y0) of a domain.
struct BTile {
    uint32_t dom, x0, y0, z0, zc, bx, by, pad;
};

// Two pull steps of every domain, A -> B (batch_two.hpp).
template <int Q, int V>
void launch_batch2(const typename Prec<V>::S* A, typename Prec<V>::S* B, const BDom<typename Prec<V>::T>* doms,
                   const BTile* tiles, uint32_t ntiles, const FusedBC<typename Prec<V>::T>& bc, hipStream_t stream);

}  // namespace plb
