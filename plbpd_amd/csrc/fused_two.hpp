// Two pull steps per pass over HBM (temporal blocking) for the fused mode:
// the numbers of two k_pull launches (gather from x - c_k with halfway
// bounce-back, BGK with the velocity-shift force, the moving-wall term where
// a wall face is hit; CollisionSRT.cpp:153-176, Streaming.cpp:63-74,
// Boundary.cpp:189-221), bit for bit, from one read of the populations of
// step t and one write of those of step t + 2.
//
// A workgroup owns a tile of bx x-cells by by y-rows and sweeps it along z
// over a chunk of planes.  At each plane zi it computes step t + 1 on the
// tile grown by one cell in x and y ((bx + 2) x (by + 2) cells, one per
// thread), gathering step t from HBM, and keeps the result in an LDS ring
// (ZRing: the directions with c_z = +1 for three planes, the others for two,
// or, where two_hold() holds, two and one).  It then computes step t + 2 on the tile at plane zi - 1, gathering
// from the ring (planes zi - 2, zi - 1, zi), and writes it to the other
// population array.  The grown border is computed by both neighbouring tiles,
// so workgroups never wait for each other: every workgroup reads only A and
// writes only its own cells of B.  The step t + 1 values pass through the
// storage type on their way into LDS, exactly as a single step stores them,
// so the result equals two single steps bit for bit.  The loads of plane
// zi + 1 are issued before the step t + 2 work of plane zi - 1, whose
// arithmetic hides their latency; where two_split() holds, those of the
// c_z = +1 directions a plane earlier still, so that the bounce-back reads of
// a cache line fall in the iteration of its pulls.  Each lattice instantiates
// these templates in its own file (fused_two_q19.hip, fused_two_q27.hip).
#pragma once

#include <algorithm>
#include <type_traits>

#include "fused_kernels.hpp"

namespace plb {

namespace {

// Buffer accesses: a buffer's bytes [0, bytes), byte offset voff (per lane) +
// soff (uniform).  A lane whose voff is kNoStore stores nothing: it lies past
// every buffer's end (buffers end below it), and the memory unit drops stores
// past the end of a buffer.
constexpr uint32_t kNoStore = 0xfffffff8u;
typedef uint32_t u32x2 __attribute__((ext_vector_type(2)));

__device__ inline __amdgpu_buffer_rsrc_t buffer_of(const void* p, uint32_t bytes) {
    return __builtin_amdgcn_make_buffer_rsrc(const_cast<void*>(p), (short)0, (int)bytes, 0x00027000);
}
template <class S>
__device__ inline S buf_load(__amdgpu_buffer_rsrc_t r, uint32_t voff, uint32_t soff) {
    if constexpr (sizeof(S) == 8)
        return __builtin_bit_cast(S, __builtin_amdgcn_raw_buffer_load_b64(r, (int)voff, (int)soff, 0));
    else if constexpr (sizeof(S) == 4)
        return __builtin_bit_cast(S, __builtin_amdgcn_raw_buffer_load_b32(r, (int)voff, (int)soff, 0));
    else
        return __builtin_bit_cast(S, __builtin_amdgcn_raw_buffer_load_b16(r, (int)voff, (int)soff, 0));
}
template <class S>
__device__ inline void buf_store(__amdgpu_buffer_rsrc_t r, S v, uint32_t voff, uint32_t soff) {
    if constexpr (sizeof(S) == 8)
        __builtin_amdgcn_raw_buffer_store_b64(__builtin_bit_cast(u32x2, v), r, (int)voff, (int)soff, 0);
    else if constexpr (sizeof(S) == 4)
        __builtin_amdgcn_raw_buffer_store_b32(__builtin_bit_cast(uint32_t, v), r, (int)voff, (int)soff, 0);
    else
        __builtin_amdgcn_raw_buffer_store_b16(__builtin_bit_cast(unsigned short, v), r, (int)voff, (int)soff, 0);
}

// A population array as W buffers, whole pairs of opposite directions each
// (W = 0: none).  Two to four of them cost a few scalar registers; a buffer for
// each pair, and pointers, cost D3Q27 384^3 FP32-shifted 1,841 and 1,711 us per
// step (1,560 with two buffers).
template <int Q, int W>
struct PopBuffers {
    __amdgpu_buffer_rsrc_t r[W ? W : 1];
    __device__ PopBuffers(const void* A, uint32_t psz) {
#pragma unroll
        for (int g = 0; g < (W ? W : 1); ++g) {
            const int first = two_group_first(Q, W, g), end = two_group_first(Q, W, g + 1);
            r[g] = buffer_of(reinterpret_cast<const char*>(A) + (uint64_t)first * psz,
                             W ? (uint32_t)(end - first) * psz : 0u);
        }
    }
};

// The arguments of one domain of a batch (batch_two.hpp).
template <class T>
struct BatchTileArgs;

// Direction groups of the step t gathers: kAll, or, where the c_z = +1
// directions are issued a plane ahead of the others, kUp (c_z = +1) and
// kFlat (c_z = 0 and -1).
enum : int { kAll = 0, kUp = 1, kFlat = 2 };
template <int Q, int K, int G>
__device__ constexpr bool in_group() {
    return G == kAll || (Lat<Q>::cz(K) > 0) == (G == kUp);
}

// Step t loads for the directions of group G: population k from x - c_k, or
// the cell's own slot rev(k) where that neighbour is not fluid, by the
// neighbour mask m around interior solids (NB) and by the coordinates without
// (so no load waits on a flag); one load per population.  c, psz (the bytes of
// a population) and the seams s are in bytes.  Directions k and rev(k) are
// neighbours in the array (1 and 2, 3 and 4, ...), so with the lower one's
// base as the uniform part of the address, the two candidates differ by a
// per-lane offset and psz only.  The array is W buffers of up to 4 GiB
// (PopBuffers); W = 0: pointers (larger arrays, every byte offset of one
// population within 32 bits).
template <int Q, int K, int V, int NB, int W, int G>
__device__ inline void gather(typename Prec<V>::S (&fv)[Q], const PopBuffers<Q, W>& ra,
                              const typename Prec<V>::S* __restrict__ A, uint32_t c, uint32_t psz, uint32_t m,
                              const Seams<uint32_t>& s) {
    if constexpr (K < Q) {
        if constexpr (in_group<Q, K, G>()) {
            using S = typename Prec<V>::S;
            constexpr uint32_t R = (uint32_t)rev_k<Q>(K);
            const bool solid = NB ? ((m >> R) & 1u) != 0 : pull_wall<Q, K>(s);
            const uint32_t to = c + pull_offset<Q, K>(s);
            if constexpr (W == 0) {
                const char* p = reinterpret_cast<const char*>(A) + (uint64_t)(solid ? R : (uint32_t)K) * psz;
                fv[K] = *reinterpret_cast<const S*>(p + (solid ? c : to));
            } else {
                constexpr uint32_t lower = (uint32_t)K < R ? (uint32_t)K : R;
                const uint32_t moved = (uint32_t)K == lower ? to : to + psz, own = (uint32_t)K == lower ? c + psz : c;
                const uint32_t off = K == 0 ? c : (solid ? own : moved);
                constexpr int g = two_group(Q, W, K);
                fv[K] = buf_load<S>(ra.r[g], off, (lower - (uint32_t)two_group_first(Q, W, g)) * psz);
            }
        }
        gather<Q, K + 1, V, NB, W, G>(fv, ra, A, c, psz, m, s);
    }
}

// Step t + 2 of a cell into its own slots (zeros where zero is set), at byte
// offset voff of each population; kNoStore: no store (a lane's, without a
// branch).
template <int Q, int V, int W>
__device__ inline void store_own(const typename Prec<V>::T (&f)[Q], const PopBuffers<Q, W>& rb,
                                 typename Prec<V>::S* __restrict__ B, uint32_t voff, uint32_t psz, bool zero) {
    using P = Prec<V>;
#pragma unroll
    for (int k = 0; k < Q; ++k) {
        const typename P::S v = P::store_raw(zero ? (typename P::T)0 : f[k]);
        if constexpr (W == 0) {
            buf_store(buffer_of(reinterpret_cast<const char*>(B) + (uint64_t)k * psz, psz), v, voff, 0u);
        } else {
            const int g = two_group(Q, W, k);
            buf_store(rb.r[g], v, voff, (uint32_t)(k - two_group_first(Q, W, g)) * psz);
        }
    }
}

// Ring plane of direction k in its group's slot: element offset of cell 0.
template <int Q, int K, int NI, bool H>
__device__ inline uint32_t ring_at(uint32_t slot) {
    using Z = ZRing<Q, H>;
    constexpr int g = Z::grp(K);
    return ((uint32_t)Z::base(g) + slot * (uint32_t)Z::size(g) + (uint32_t)Z::idx(K)) * (uint32_t)NI;
}

// Step t + 1 of a cell into the ring: direction k to its group's slot for
// this plane (up for the c_z = +1 group, fl for the others).
template <int Q, int K, int V, int NI, bool H>
__device__ inline void ring_store(const typename Prec<V>::T (&f)[Q], typename Prec<V>::S* ring, uint32_t cell,
                                  uint32_t up, uint32_t fl) {
    if constexpr (K < Q) {
        ring[ring_at<Q, K, NI, H>(ZRing<Q, H>::grp(K) == 0 ? up : fl) + cell] = Prec<V>::store_raw(f[K]);
        ring_store<Q, K + 1, V, NI, H>(f, ring, cell, up, fl);
    }
}

// Step t + 1 values for the step t + 2 cell at ring index li (plane zo):
// population k from li - c_k in plane zo - c_k,z, or the cell's own slot
// rev(k) in plane zo where x - c_k is not fluid.  Slots: pa = the c_z = +1
// group's slot of plane zo - 1, oa = its slot of plane zo, b0 = the other
// groups' slot of plane zo, c1 = the c_z = -1 group's slot of plane zo + 1.
// RX: cells per grown row.  P: kAll, or the directions with c_z = -1 (kDown),
// or the others (kHeld).
enum : int { kDown = 3, kHeld = 4 };
template <int Q, int K, int V, int NB, int NI, bool H, int P>
__device__ inline void ring_gather(typename Prec<V>::T (&f)[Q], const typename Prec<V>::S* ring, uint32_t li,
                                   uint32_t RX, uint32_t pa, uint32_t oa, uint32_t b0, uint32_t c1, uint32_t m,
                                   const Seams<uint32_t>& s) {
    if constexpr (K < Q) {
        using Z = ZRing<Q, H>;
        constexpr int R = rev_k<Q>(K);
        constexpr int cx = Lat<Q>::cx(K), cy = Lat<Q>::cy(K), cz = Lat<Q>::cz(K);
        constexpr int g = Z::grp(K), gr = Z::grp(R);
        if constexpr (P == kAll || (cz < 0) == (P == kDown)) {
            const uint32_t moved =
                ring_at<Q, K, NI, H>(g == 0 ? pa : (g == 1 ? b0 : c1)) + li - ((uint32_t)cx + (uint32_t)cy * RX);
            const uint32_t own = ring_at<Q, R, NI, H>(gr == 0 ? oa : b0) + li;
            if constexpr (NB != 0) {
                // own - moved is uniform (li cancels) and, like every ring index,
                // far inside the signed 24-bit range: one 24-bit multiply-add by
                // the mask bit instead of a compare and a select
                const int d = __mul24((int)((m >> R) & 1u), (int)(own - moved));
                f[K] = Prec<V>::load_raw(ring[moved + (uint32_t)d]);
            } else {
                f[K] = Prec<V>::load_raw(ring[pull_wall<Q, K>(s) ? own : moved]);
            }
        }
        ring_gather<Q, K + 1, V, NB, NI, H, P>(f, ring, li, RX, pa, oa, b0, c1, m, s);
    }
}

// Workgroup barrier that orders LDS only.  The global stores of a step t + 2
// cell are read by no other thread of the launch, so the barrier need not
// wait for them -- nor for the step t loads of the next plane, which are in
// flight across it (__syncthreads would wait for every outstanding global
// access).
__device__ inline void lds_barrier() {
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "workgroup", "local");
    __builtin_amdgcn_s_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "workgroup", "local");
}

// The sweep of one workgroup over the planes [z0, z0 + zc) of the tile of
// bx x by cells at (x0, y0), of any shape with at most two_cap() grown cells.
// (With 64 x 8 and 32 x 11 tiles compiled in, before values were held, D3Q19
// 256^3 ran 269 / 591 us per step walls only, FP32-shifted / FP64, against 263 /
// 595 with the shape as an argument.)  a: FusedArgs, or the like for one domain of a batch.  MOV
// (two_walls()): the form for moving walls and for walls on x.
template <int Q, int V, int NB, bool MOV, int W, bool SPLIT, class Args>
__device__ __forceinline__ void pull2_tile(const typename Prec<V>::S* __restrict__ A,
                                           typename Prec<V>::S* __restrict__ B, const uint8_t* __restrict__ flags,
                                           const uint32_t* __restrict__ nbmask, const Args& a, uint32_t bx,
                                           uint32_t by, uint32_t x0, uint32_t y0, uint32_t z0, uint32_t zc) {
    using P = Prec<V>;
    using S = typename P::S;
    using T = typename P::T;
    using I = uint32_t;
    constexpr int NI = two_cap(Q, (int)sizeof(S));  // threads, and cells per ring plane
    static_assert(NI % 64 == 0 && NI * two_lds(Q, (int)sizeof(S)) <= 160 * 1024, "whole wavefronts, a ring that fits");
    const uint32_t RX = bx + 2u;  // grown row
    constexpr bool HOLD = two_hold(Q, (int)sizeof(S));
    __shared__ S ring[ZRing<Q, HOLD>::planes() * NI];
    __shared__ uint32_t mring[(HOLD ? 1 : 2) * NI];  // the step t + 1 cells' masks or flags

    const uint32_t tid = threadIdx.x;
    const uint32_t X = a.X, Y = a.Y, Z = a.Z;
    const I XY = X * Y, ps = (I)a.pstride;
    const uint32_t nplanes = std::min(zc, Z - z0) + 2u;

    // step t + 1: this thread's cell of the grown tile (wrapped coordinates)
    const uint32_t ix = tid % RX, iy = tid / RX;
    const uint32_t gx = (x0 + ix + X - 1u) % X, gy = (y0 + iy + Y - 1u) % Y;
    // step t + 2: this thread's cell of the tile
    const uint32_t ox = tid % bx, oy = tid / bx;
    const bool in_o = oy < by && y0 + oy < Y && x0 + ox < X;
    const uint32_t px = x0 + ox, py = y0 + oy;
    // (a thread without a cell reads those of the first one and stores nothing)
    const I li = in_o ? (oy + 1u) * RX + ox + 1u : RX + 1u;

    // Loads of step t, issued an iteration ahead of the plane that uses them.
    // SPLIT issues the directions with c_z = +1 two iterations ahead instead,
    // so that the bounce-back read of a cell's own slot rev(k) falls in the
    // same iteration as the pulls from the same cache line: a line of a
    // c_z = +1 population in plane p is pulled by the cells of plane p + 1
    // and read back by those of plane p for their c_z = -1 directions, and a
    // line of a c_z = -1 population is pulled by the cells of plane p - 1 and
    // read back, for their c_z = +1 directions, by those of plane p.  (The
    // c_z = +1 values then stay in registers for an extra iteration.)
    // Around interior solids the gather addresses depend on the neighbour
    // mask, loaded at the start of the iteration before the gather.
    //
    // Neighbour mask (NB) or flag of this thread's step t + 1 cell in plane n.
    // Every thread loads, also past the grown tile (its wrapped coordinates
    // stay in the lattice; the values are not used): loads under a branch
    // made the compiler wait for loads in flight where the branches merge.
    // A batch has no flags: its solid cells are the wall layers, known from
    // the coordinates.
    constexpr bool FLAGS = !std::is_same<Args, BatchTileArgs<T>>::value;
    auto wall_cell = [&](uint32_t x, uint32_t y, uint32_t z) __attribute__((always_inline)) -> uint32_t {
        return (a.bc.wall_lo[0] && x == 0) || (a.bc.wall_hi[0] && x + 1u == X) || (a.bc.wall_lo[1] && y == 0) ||
               (a.bc.wall_hi[1] && y + 1u == Y) || (a.bc.wall_lo[2] && z == 0) || (a.bc.wall_hi[2] && z + 1u == Z);
    };
    auto load_mask = [&](uint32_t n) __attribute__((always_inline)) -> uint32_t {
        const uint32_t zn = (z0 + n + Z - 1u) % Z;
        const I c = zn * XY + gy * X + gx;
        if constexpr (!FLAGS) return wall_cell(gx, gy, zn);
        else return NB ? nbmask[c] : (uint32_t)flags[c];
    };
    // the loads of plane n's directions of group G into fv
    constexpr I sz = (I)sizeof(S);
    const I psz = ps * sz;
    const PopBuffers<Q, W> ra(A, psz), rb(B, psz);
    auto fetch = [&](auto group, uint32_t n, S (&fv)[Q], uint32_t m) __attribute__((always_inline)) {
        constexpr int G = decltype(group)::value;
        const uint32_t zi = (z0 + n + Z - 1u) % Z;
        const I c = zi * XY + gy * X + gx;
        Seams<I> sb = seams<I>(gx, gy, zi, a);
        sb.xm *= sz, sb.xp *= sz, sb.ym *= sz, sb.yp *= sz, sb.zm *= sz, sb.zp *= sz;
        gather<Q, 0, V, NB, W, G>(fv, ra, A, c * sz, psz, m, sb);
    };
    using All = std::integral_constant<int, kAll>;
    using Up = std::integral_constant<int, kUp>;
    using Flat = std::integral_constant<int, kFlat>;

    // Step t + 2 of the tile's cell at plane n - 2 of the chunk (iteration n;
    // none in the first two), zo in the lattice: its values from the ring planes
    // of iterations n - 2, n - 1 and n, with the mask of its step t + 1 cell
    // (stored in mring by iteration n - 1), then its collision and its stores.
    //
    // One straight run of instructions from the ring's reads to the
    // stores, threads without a cell and cells that are not fluid
    // included (what they compute is dropped): the compiler then spreads
    // the stores over the arithmetic, and in step 1 the next plane's loads,
    // instead of issuing them in bursts at the end of a branch.  The
    // kernel is bound by neither alone (D3Q19 256^3 FP32-shifted around
    // solids: vector unit 65% busy, memory unit 67%), so what counts is
    // that both work at the same time: 341 -> 317 us per step with solids,
    // 287 -> 268 walls only; before values were held FP64 647 -> 630 / 601 -> 589,
    // D3Q27 384^3 FP32-shifted 1,634 -> 1,560, FP64 3,638 -> 3,455.  (Stores in every
    // wavefront and plane, dropped where there is nothing to store, so that
    // no wait for a load counts a path without them: no faster on large
    // lattices, 2-10% slower on small ones.)
    auto mask2 = [&](uint32_t slot0, uint32_t z) __attribute__((always_inline)) -> uint32_t {
        if constexpr (FLAGS) return mring[slot0 * NI + li];
        else return wall_cell(px, py, z);
    };
    // The wall terms of a cell, for D3Q27 from coordinates that the compiler
    // takes for new ones in every plane.  From the loop's own it computes each direction's wall
    // test and c_k . u_w before the loop and keeps them in registers through it:
    // next to the held values 51 (FP64) and 45 (FP32) registers then
    // went to scratch memory and back in every plane (128^3, lid on x / y, FP64 193 ->
    // 162 / 164 -> 138 us per step, FP32-shifted 134 -> 111 / 100 -> 86).
    // D3Q19 has the registers (with FP16-shifted storage it ran 7% slower so).
    auto walls = [&](T (&f)[Q], T rho, uint32_t x, uint32_t y, uint32_t z) __attribute__((always_inline)) {
        if (MOV && a.bc.moving) {
            if constexpr (Q == 27) asm volatile("" : "+v"(x), "+v"(y));
            moving_wall_terms<Q, P>(f, rho, seams<I>(x, y, z, a), a);
        }
    };
    auto finish = [&](uint32_t zo, bool zero, T (&f)[Q]) __attribute__((always_inline)) {
        const T rho = bgk<Q, P>(f, a, true);
        walls(f, rho, px, py, zo);
        // Around interior solids and with walls on x, which begin and end
        // every row, a cell that is not fluid stores zeros, so that lines are
        // written whole (but a wavefront of such cells nothing); the wall
        // rows of the other axes store nothing.
        const bool whole = NB || (MOV && sizeof(S) > 2 && a.bc.wall_lo[0]);
        const bool store = in_o && (whole || !zero);
        store_own<Q, V, W>(f, rb, B, store ? (zo * XY + py * X + px) * sz : kNoStore, psz, whole && zero);
    };
    auto step2 = [&](uint32_t n) __attribute__((always_inline)) {
        const uint32_t zo = z0 + n - 2u;
        if (n < 2u) return;
        const uint32_t b0 = (n + 1u) & 1u;
        const uint32_t mo = mask2(b0, zo);
        const bool zero = NB ? (mo & 1u) != 0 : mo != 0;
        if (__any(in_o && !zero)) {
            const Seams<I> sm = seams<I>(px, py, zo, a);
            T f[Q];
            ring_gather<Q, 0, V, NB, NI, HOLD, kAll>(f, ring, li, RX, (n + 1u) % 3u, (n + 2u) % 3u, b0, n & 1u, mo, sm);
            finish(zo, zero, f);
        }
    };
    // HOLD: the cell's values in two parts.  read2 completes the cell of plane
    // n - 1 (fo, its mask mo) with the c_z = -1 directions from plane n, and takes
    // the other directions of the cell of plane n (hold, its mask mhold).
    T hold[Q], fo[Q];
    uint32_t mhold = 1u, mo = 1u;
    auto read2 = [&](uint32_t n) __attribute__((always_inline)) {
        const uint32_t up = (n + 1u) & 1u, zh = (z0 + n + Z - 1u) % Z;  // the c_z = +1 group's slot of plane n - 1
#pragma unroll
        for (int k = 0; k < Q; ++k)
            if (Lat<Q>::cz(k) >= 0) fo[k] = hold[k];
        mo = mhold;
        ring_gather<Q, 0, V, NB, NI, true, kDown>(fo, ring, li, RX, up, up, 0u, 0u, mo,
                                                  seams<I>(px, py, (z0 + n + Z - 2u) % Z, a));
        mhold = mask2(0u, zh);
        ring_gather<Q, 0, V, NB, NI, true, kHeld>(hold, ring, li, RX, up, up, 0u, 0u, mhold, seams<I>(px, py, zh, a));
    };
    auto collide2 = [&](uint32_t n) __attribute__((always_inline)) {
        if (n < 2u) return;
        const uint32_t zo = z0 + n - 2u;
        const bool zero = NB ? (mo & 1u) != 0 : mo != 0;
        if (__any(in_o && !zero)) finish(zo, zero, fo);
    };
    // The second half of an iteration: plane n is in the ring.  HOLD with
    // 4-byte storage collides after the barrier, next to the loads and the
    // collision of the next plane (after / before the barrier: D3Q27
    // FP32-shifted 256^3 457 / 477 us per step, 384^3 1,527 / 1,542; FP64, which waits
    // on its stores there, D3Q19 256^3 602 / 571, D3Q27 384^3 3,085 / 3,017).
    auto second = [&](uint32_t n) __attribute__((always_inline)) {
        lds_barrier();
        if constexpr (!HOLD) {
            step2(n);
            lds_barrier();
        } else {
            read2(n);
            if (sizeof(S) == 8) collide2(n);
            lds_barrier();
            if (sizeof(S) != 8) collide2(n);
        }
    };
    // Step t + 1 of this thread's cell at plane n from the loads in fv, into
    // its ring slots (relative plane numbers: only n mod 3 and mod 2 matter).
    auto step1 = [&](uint32_t n, const S (&fv)[Q]) __attribute__((always_inline)) {
        T f[Q];
#pragma unroll
        for (int k = 0; k < Q; ++k) f[k] = P::load_raw(fv[k]);
        const T rho = bgk<Q, P>(f, a, true);
        walls(f, rho, gx, gy, (z0 + n + Z - 1u) % Z);
        ring_store<Q, 0, V, NI, HOLD>(f, ring, tid, HOLD ? n & 1u : n % 3u, HOLD ? 0u : n & 1u);
    };

    if constexpr (!SPLIT) {
        // One plane n: the step t + 1 cell of plane n from the loads in fv
        // and the mask mcur; the mask of plane n + 1 into mnext and its loads
        // into fv; the step t + 2 cell of plane n - 1.  The loop runs it twice
        // per trip with the two mask registers swapped, so that no register
        // that a load in flight writes is copied (a copy would wait for the
        // load).  (Written with one captured register set: the same body with
        // the set passed by reference compiled to longer waits.)
        S fv[Q];
        auto plane = [&](uint32_t n, uint32_t& mcur, uint32_t& mnext) __attribute__((always_inline)) {
            // (plane numbers wrap modulo Z, so the loads past the chunk's
            // last plane stay in bounds; their values are not used)
            mnext = load_mask(n + 1u);
            // the step t + 2 cells read this mask
            if (FLAGS) mring[(HOLD ? 0u : n & 1u) * NI + tid] = mcur;
            // (a wavefront of solid cells has nothing to compute)
            if (!__all(NB ? (mcur & 1u) != 0 : mcur != 0)) step1(n, fv);
            fetch(All{}, n + 1u, fv, mnext);
            second(n);
        };
        uint32_t m0 = load_mask(0), m1 = 0;
        fetch(All{}, 0, fv, m0);
        for (uint32_t n = 0; n < nplanes; n += 2u) {
            plane(n, m0, m1);
            if (n + 1u < nplanes) plane(n + 1u, m1, m0);
        }
    } else {
        // One plane n: the step t + 1 cell of plane n from fc and the mask mc
        // of plane n; the c_z = 0 and -1 directions of plane n + 1 into fn
        // (its c_z = +1 directions are in flight) with the mask mn of plane
        // n + 1, loaded an iteration ago; the mask of plane n + 2 into mc and
        // its c_z = +1 directions into fc; the step t + 2 cell of plane
        // n - 1.  Step t + 1 runs in every wavefront, also one of solid cells:
        // behind a vote the loads would not spread over it (317 -> 332 us per
        // step).  The loop runs it twice per trip with the register sets
        // swapped (odd: fc = fv1, fn = fv0), so that no register that a load
        // in flight writes is copied.
        S fv0[Q], fv1[Q];
        auto plane = [&](auto odd, uint32_t n, uint32_t& mc, uint32_t& mn) __attribute__((always_inline)) {
            S (&fc)[Q] = decltype(odd)::value ? fv1 : fv0;
            S (&fn)[Q] = decltype(odd)::value ? fv0 : fv1;
            if (FLAGS) mring[(HOLD ? 0u : n & 1u) * NI + tid] = mc;
            mc = load_mask(n + 2u);
            fetch(Flat{}, n + 1u, fn, mn);
            step1(n, fc);
            fetch(Up{}, n + 2u, fc, mc);
            second(n);
        };
        uint32_t m0 = load_mask(0), m1 = load_mask(1);
        fetch(All{}, 0, fv0, m0);
        fetch(Up{}, 1, fv1, m1);
        for (uint32_t n = 0; n < nplanes; n += 2u) {
            plane(std::false_type{}, n, m0, m1);
            if (n + 1u < nplanes) plane(std::true_type{}, n + 1u, m1, m0);
        }
    }
}

template <int Q, int V, int NB, bool MOV, int W>
__global__ __launch_bounds__(two_cap(Q, (int)sizeof(typename Prec<V>::S)), 1) void k_pull2(
    const typename Prec<V>::S* __restrict__ A, typename Prec<V>::S* __restrict__ B,
    const uint8_t* __restrict__ flags, const uint32_t* __restrict__ nbmask, FusedArgs<typename Prec<V>::T> a,
    TwoGeom g) {
    uint32_t tx, ty, tz;
    if (g.xcd) {
        // workgroup i runs on XCD i mod 8, which takes pairs [j kx, (j + 1) kx)
        const uint32_t j = blockIdx.x & 7u, m = blockIdx.x >> 3;
        tx = m % g.ntx;
        const uint32_t pr = j * g.kx + m / g.ntx;
        if (pr >= g.nty * g.nzc) return;  // past the last pair (the whole workgroup)
        ty = pr % g.nty;
        tz = pr / g.nty;
    } else {
        tx = blockIdx.x % g.ntx;
        const uint32_t r = blockIdx.x / g.ntx;
        ty = r % g.nty;
        tz = r / g.nty;
    }
    pull2_tile<Q, V, NB, MOV, W, two_split(Q, (int)sizeof(typename Prec<V>::S), NB != 0)>(
        A, B, flags, nbmask, a, g.bx, g.by, tx * g.bx, ty * g.by, tz * g.zc, g.zc);
}

}  // namespace

template <int Q, int V>
bool launch_pull2(const FusedArgs<typename Prec<V>::T>& a, const TwoGeom& g, bool nb, bool mov,
                  const typename Prec<V>::S* A, typename Prec<V>::S* B, const uint8_t* flags,
                  const uint32_t* nbmask, hipStream_t stream) {
    constexpr int sb = (int)sizeof(typename Prec<V>::S);
    // the tile must fit the ring and the workgroup
    if (g.bx < 1 || g.by < 1 || (uint64_t)(g.bx + 2) * (g.by + 2) > (uint64_t)two_cap(Q, sb)) return false;
    const dim3 grid(two_blocks(g)), block(two_cap(Q, sb));
    auto go = [&](auto nbc, auto mvc, auto wc) {
        hipLaunchKernelGGL((k_pull2<Q, V, decltype(nbc)::value, decltype(mvc)::value, decltype(wc)::value>), grid,
                           block, 0, stream, A, B, flags, nbmask, a, g);
    };
    auto by_walls = [&](auto wc) {
        using N0 = std::integral_constant<int, 0>;
        using N1 = std::integral_constant<int, 1>;
        if (nb) mov ? go(N1{}, std::true_type{}, wc) : go(N1{}, std::false_type{}, wc);
        else mov ? go(N0{}, std::true_type{}, wc) : go(N0{}, std::false_type{}, wc);
    };
    switch (g.buffers) {
        case 1: by_walls(std::integral_constant<int, 1>()); break;
        case 2: by_walls(std::integral_constant<int, 2>()); break;
        case 4: by_walls(std::integral_constant<int, 4>()); break;
        default: by_walls(std::integral_constant<int, 0>()); break;
    }
    return true;
}

#define PLB_TWO_INST(Q, V)                                                                                  \
    template bool launch_pull2<Q, V>(const FusedArgs<typename Prec<V>::T>&, const TwoGeom&, bool, bool,       \
                                     const typename Prec<V>::S*, typename Prec<V>::S*, const uint8_t*,       \
                                     const uint32_t*, hipStream_t);
#define PLB_TWO_INST_Q(Q) \
    PLB_TWO_INST(Q, kF64) PLB_TWO_INST(Q, kF32) PLB_TWO_INST(Q, kF64A32) PLB_TWO_INST(Q, kF32S) PLB_TWO_INST(Q, kF16S)

}  // namespace plb
