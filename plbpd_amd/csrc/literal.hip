// Literal mode: the reference's staged step (PLBPD.cpp:23-30), one kernel per
// reference operator, on halo'd structure-of-arrays buffers: rho[c], u[i * ncell
// + c] and n[at(k) + c], c = (z*(Y+2) + y)*nx + x, x in [0, X+1] etc. (LitDims).
// A collision and the push after it can run as one kernel (k_collide_push),
// which can also take the previous step's moments and resets
// (k_moments_collide_push); every buffer ends as after the separate kernels.
// R = double (FP64 contract) or float (the reference's own rounding, with its
// float/double promotions).  Compiled with -ffp-contract=off: every
// expression below is evaluated in the order written, as in the reference.
#include <string>
#include <type_traits>

#include "host_read.hpp"
#include "state.hpp"

namespace plb {
namespace {

constexpr unsigned kThreads = 256;

// Device layout.  Population k of cell c lies at at(k) + c, at(k) = k * ps +
// base - (c_kx * sx + c_ky * sy + c_kz * sz).  With (sx, sy, sz) = (1, nx, nx * ny)
// the slot (x + c_k, k), which a push from cell x fills, lies at x's own place
// in array k, so that a wavefront of the collide+push kernels writes the same
// cells of every array: whole lines, as rows start on a line (nx and ps whole
// lines, base such that x = 1 begins one); its reads of (x, k) are shifted
// instead, by a cell along the row at most, and a line that two wavefronts read
// is in the cache.  With (0, 0, 0), base 0 and nx = X + 2 (lit_layout's packed
// form) a slot lies at its own cell, and the pushes' stores share lines.
struct LitDims {
    int X, Y, Z;
    int nx, ny;         // cells from row to row (X + 2 or more), Y + 2
    uint64_t ncell;     // nx * ny * (Z + 2)
    uint64_t ps, base;  // elements between the population arrays, and before the first
    int64_t sx, sy, sz;
    __host__ __device__ uint64_t cell(int z, int y, int x) const {
        return ((uint64_t)z * ny + y) * nx + x;
    }
    __host__ __device__ int64_t at(int k, int cx, int cy, int cz) const {
        return (int64_t)(k * ps + base) - (cx * sx + cy * sy + cz * sz);
    }
    template <int Q>
    __device__ int64_t at(int k) const {
        return at(k, Lat<Q>::cx(k), Lat<Q>::cy(k), Lat<Q>::cz(k));
    }
    // where a push from cell c puts population k, less c: the slot of c + c_k
    template <int Q>
    __device__ int64_t to(int k) const {
        const int cx = Lat<Q>::cx(k), cy = Lat<Q>::cy(k), cz = Lat<Q>::cz(k);
        return at(k, cx, cy, cz) + cx + (int64_t)cy * nx + (int64_t)cz * nx * ny;
    }
};

LitDims dims_of(const plb_state* s) {
    LitDims d;
    d.X = s->X;
    d.Y = s->Y;
    d.Z = s->Z;
    d.nx = s->lit_nx;
    d.ny = s->Y + 2;
    d.ncell = lit_cells(s);
    d.ps = s->pstride;
    d.base = s->lit_base;
    const int64_t on = s->lit_base != 0;
    d.sx = on;
    d.sy = on * d.nx;
    d.sz = on * d.nx * d.ny;
    return d;
}

template <class Fn>
int with_q(int q, Fn&& fn) {
    switch (q) {
        case 9: return fn(std::integral_constant<int, 9>());
        case 19: return fn(std::integral_constant<int, 19>());
        case 27: return fn(std::integral_constant<int, 27>());
        default: return fail(PLB_ERR_LOGIC, "Model with q=" + std::to_string(q) + " not yet implemented");
    }
}

template <class Fn>
int with_qr(const plb_state* s, Fn&& fn) {
    return with_q(s->q, [&](auto qc) {
        if (s->variant == kF64) return fn(qc, double());
        return fn(qc, float());
    });
}

// ---------------------------------------------------------------- kernels --
// Domain::initialize (Domain.cpp:46-64): every cell, halo included, gets
// rho0, u and feq(rho0, u); ntmp is zero (SimData.cpp:53-56).
template <int Q, class R>
__global__ void k_init(LitDims g, R* n, R* ntmp, R* rho, R* u, double rho0, double u0x,
                       double u0y, double u0z, int kind, uint64_t seed, double amp,
                       const double* tg) {
    const uint64_t c = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (c >= g.ncell) return;
    const int x = (int)(c % g.nx);
    const int y = (int)((c / g.nx) % g.ny);
    const int z = (int)(c / ((uint64_t)g.nx * g.ny));
    if (x > g.X + 1) return;
    const int xi = (x - 1 + g.X) % g.X, yi = (y - 1 + g.Y) % g.Y, zi = (z - 1 + g.Z) % g.Z;
    const double u0[3] = {u0x, u0y, u0z};
    double uc[3];
    cell_velocity(kind, seed, amp, g.X, g.Y, g.Z, u0, tg, xi, yi, zi, uc);
    const R ur[3] = {(R)uc[0], (R)uc[1], (R)uc[2]};
    const R r0 = (R)rho0;
    rho[c] = r0;
    for (int i = 0; i < 3; ++i) u[i * g.ncell + c] = ur[i];
    const R usq = ur[0] * ur[0] + ur[1] * ur[1] + ur[2] * ur[2];
#pragma unroll
    for (int k = 0; k < Q; ++k) {
        n[g.at<Q>(k) + (int64_t)c] = feq_ref<Q, R>(k, r0, ur, usq);
        ntmp[g.at<Q>(k) + (int64_t)c] = (R)0;
    }
}

// CollisionSRT::_collision_kernel (CollisionSRT.cpp:153-176) for population
// k of one cell, with _get_cu (84-91): the post-collision value of old.  In
// FP32 the reference's promotions are kept: w_k * rho in float, the bracket in
// double (double literals), the blend's first product in float, its sum in
// double, the result rounded to float.
template <int Q, class R>
__device__ inline R collide_value(int k, R old, R rl, const R (&uu)[3], R usq, R om, R omm) {
    const R cu = (k == 0) ? (R)0
                          : (R)Lat<Q>::cx(k) * uu[0] + (R)Lat<Q>::cy(k) * uu[1] + (R)Lat<Q>::cz(k) * uu[2];
    if (std::is_same<R, float>::value) {
        const float wr = (float)Lat<Q>::w(k) * (float)rl;
        const double neq =
            (double)wr * (1.0 + 3.0 * (double)cu + 4.5 * (double)cu * (double)cu - 1.5 * (double)usq);
        const float a = (float)omm * (float)old;
        return (R)((double)a + (double)om * neq);
    } else {
        const double neq =
            (Lat<Q>::w(k) * (double)rl) * (1.0 + 3.0 * (double)cu + 4.5 * (double)cu * (double)cu - 1.5 * (double)usq);
        return (R)((double)omm * (double)old + (double)om * neq);
    }
}

// _get_updated_u (CollisionSRT.cpp:72-81): u* = u + tau F / rho, and |u*|^2.
template <class R>
__device__ inline void updated_u(R u0, R u1, R u2, R rl, R tau, R F0, R F1, R F2, R (&uu)[3], R& usq) {
    const R tri = tau / rl;
    uu[0] = u0 + F0 * tri;
    uu[1] = u1 + F1 * tri;
    uu[2] = u2 + F2 * tri;
    usq = uu[0] * uu[0] + uu[1] * uu[1] + uu[2] * uu[2];
}

// CollisionSRT::operator() (CollisionSRT.cpp:25-176): in place, every interior cell.
template <int Q, class R>
__global__ void k_collide(LitDims g, R* __restrict__ n, const R* __restrict__ rho,
                          const R* __restrict__ u, R tau, R om, R omm, R F0, R F1, R F2) {
    const int x = blockIdx.x * blockDim.x + threadIdx.x + 1;
    const int y = blockIdx.y + 1, z = blockIdx.z + 1;
    if (x > g.X) return;
    const uint64_t c = g.cell(z, y, x);
    const R rl = rho[c];
    R uu[3], usq;
    updated_u(u[c], u[g.ncell + c], u[2 * g.ncell + c], rl, tau, F0, F1, F2, uu, usq);
#pragma unroll
    for (int k = 0; k < Q; ++k) {
        R* p = n + g.at<Q>(k) + c;
        *p = collide_value<Q, R>(k, *p, rl, uu, usq, om, omm);
    }
}

// Whether c - c_k of interior cell c lies in the halo: a slot no push writes.
template <int Q>
__device__ inline bool from_halo(const LitDims& g, int k, int x, int y, int z) {
    const int cx = Lat<Q>::cx(k), cy = Lat<Q>::cy(k), cz = Lat<Q>::cz(k);
    return (cx > 0 && x == 1) || (cx < 0 && x == g.X) || (cy > 0 && y == 1) || (cy < 0 && y == g.Y) ||
           (cz > 0 && z == 1) || (cz < 0 && z == g.Z);
}
// Whether an interior cell lies on one of the faces of the bit mask (face f:
// the layer at coordinate X|Y|Z, f even, or 1, f odd, of axis f / 2).
__device__ inline bool on_faces(unsigned faces, const LitDims& g, int x, int y, int z) {
    return ((faces & 1u) && x == g.X) || ((faces & 2u) && x == 1) || ((faces & 4u) && y == g.Y) ||
           ((faces & 8u) && y == 1) || ((faces & 16u) && z == g.Z) || ((faces & 32u) && z == 1);
}

// The post-collision values that the reference leaves in place, ntmp after the
// swap.  The collide+push kernels store there only the slots (c, k) with
// c - c_k in the halo, which no push writes and the reference's stage order
// reads back (Q1).  The next push overwrites every other slot before anything
// reads it; until then its value is the one the same kernel pushed to
// n(c + c_k, k), which only a no-slip pass changes, and only for its face cells
// c (it writes n(f + c_kp, kp) for face cells f; periodic copies write n(c', k)
// with c' - c_k in the halo): that pass saves what it is about to overwrite
// (k_noslip).  So k_ntmp_restore can put every value in place, before anything
// reads ntmp (a download) or changes n (a collision by itself, an upload).
// On the faces of `saved` the no-slip passes have done so, k = 0 apart.
template <int Q, class R>
__global__ void k_ntmp_restore(LitDims g, unsigned saved, const R* __restrict__ n, R* __restrict__ t) {
    const int x = blockIdx.x * blockDim.x + threadIdx.x + 1;
    const int y = blockIdx.y + 1, z = blockIdx.z + 1;
    if (x > g.X) return;
    const uint64_t c = g.cell(z, y, x);
    const bool done = on_faces(saved, g, x, y, z);
#pragma unroll
    for (int k = 0; k < Q; ++k)
        if ((k == 0 || !done) && !from_halo<Q>(g, k, x, y, z))
            t[g.at<Q>(k) + (int64_t)c] = n[g.to<Q>(k) + (int64_t)c];
}

// The collision followed by Streaming::_push_kernel (Streaming.cpp:63-74) in
// one pass: each post-collision value is stored at x + c_k in t, as k_push
// copies it, and in place where no push will write (see k_ntmp_restore).  Every
// value a caller or a later stage can read equals the one k_collide then
// k_push give; the push's re-read of n and most in-place stores are saved.
template <int Q, class R>
__global__ void k_collide_push(LitDims g, R* __restrict__ n, const R* __restrict__ rho,
                               const R* __restrict__ u, R* __restrict__ t, R tau, R om, R omm, R F0, R F1,
                               R F2) {
    const int x = blockIdx.x * blockDim.x + threadIdx.x + 1;
    const int y = blockIdx.y + 1, z = blockIdx.z + 1;
    if (x > g.X) return;
    const uint64_t c = g.cell(z, y, x);
    const R rl = rho[c];
    R uu[3], usq;
    updated_u(u[c], u[g.ncell + c], u[2 * g.ncell + c], rl, tau, F0, F1, F2, uu, usq);
#pragma unroll
    for (int k = 0; k < Q; ++k) {
        R* p = n + g.at<Q>(k) + c;
        const R v = collide_value<Q, R>(k, *p, rl, uu, usq, om, omm);
        if (from_halo<Q>(g, k, x, y, z)) *p = v;
        t[g.to<Q>(k) + (int64_t)c] = v;
    }
}

// Streaming::_push_kernel (Streaming.cpp:63-74): ntmp(x + c_k, k) = n(x, k).
template <int Q, class R>
__global__ void k_push(LitDims g, const R* __restrict__ n, R* __restrict__ t) {
    const int x = blockIdx.x * blockDim.x + threadIdx.x + 1;
    const int y = blockIdx.y + 1, z = blockIdx.z + 1;
    if (x > g.X) return;
    const uint64_t c = g.cell(z, y, x);
#pragma unroll
    for (int k = 0; k < Q; ++k) {
        t[g.to<Q>(k) + (int64_t)c] = n[g.at<Q>(k) + (int64_t)c];
    }
}

struct FaceBox {
    int lo[3], ex[3];  // first cell and extent per axis (halo'd coordinates)
    __host__ __device__ uint64_t count() const { return (uint64_t)ex[0] * ex[1] * ex[2]; }
};

// Boundary::_get_boundary_extent (Boundary.cpp:113-148)
FaceBox face_box(int face, int X, int Y, int Z) {
    FaceBox b;
    b.lo[0] = 1; b.ex[0] = X;
    b.lo[1] = 1; b.ex[1] = Y;
    b.lo[2] = 1; b.ex[2] = Z;
    const int axis = face / 2;
    const int hi = (face % 2) == 0;  // east, north, up are the high faces
    const int dim = axis == 0 ? X : (axis == 1 ? Y : Z);
    b.lo[axis] = hi ? dim : 1;
    b.ex[axis] = 1;
    return b;
}

// The no-slip faces of one axis that one launch takes.
template <class R>
struct NoslipFaces {
    FaceBox box[2];
    R ub[2][3];
    // t, if not null: ntmp, in which the values about to be overwritten are
    // put in place (k_ntmp_restore), but for the faces of `saved`
    R* t;
    unsigned saved;
};

// Boundary::_apply_noslip (Boundary.cpp:189-221) for one face, as the serial
// z, y, x, kp loop computes it, in place.  Op (c, kp) of face cell c writes
// the slot (y, kp), y = c + c_kp, and reads n(c, k), k = rev kp:
//   y not in the face: (c, k) and (y, kp) belong to this op alone (the only
//     other op that could touch them is (y, k), and y has no ops);
//   y in the face: ops (c, kp) and (y, k) touch the two slots (c, k) and
//     (y, kp), and no other op does.  With L the earlier and U the later of
//     the two cells in loop order and kp the direction from L to U, op (L, kp)
//     writes (U, kp) = n(L, k) - t_U; op (U, k), which comes later, finds
//     n(L, k) = its old value in the slot it writes and n(U, kp) replaced, so
//     (L, k) = (n(L, k) - t(U, kp)) - t_L.  Both come from the old n(L, k):
//     the thread of (L, kp) does both.
// So no slot is shared between threads and the pass needs no staging (two
// kernels and a round trip through scratch memory before: D2Q9 256 x 64 FP64
// 5.7 us per face, D3Q19 128^3 10.5 us).  blockIdx.y is the direction, so c_kp
// and w are uniform; blockIdx.z the face: the two faces of an axis are
// independent when it has at least three layers (noslip_with).
template <int Q, class R>
__global__ void k_noslip(LitDims g, NoslipFaces<R> fs, R* __restrict__ n, const R* __restrict__ rho, R cs2inv,
                         uint32_t total) {
    const uint32_t t = blockIdx.x * blockDim.x + threadIdx.x;
    if (t >= total) return;
    const FaceBox b = fs.box[blockIdx.z];
    const int kp = 1 + (int)blockIdx.y, k = rev<Q>(kp);
    int cxp = 0, cyp = 0, czp = 0;
    R wk = (R)0;
#pragma unroll
    for (int j = 1; j < Q; ++j)
        if (j == kp) {
            cxp = Lat<Q>::cx(j);
            cyp = Lat<Q>::cy(j);
            czp = Lat<Q>::cz(j);
            wk = (R)Lat<Q>::w(j);  // w_k == w_kp
        }
    const uint32_t e0 = (uint32_t)b.ex[0], e1 = (uint32_t)b.ex[1];
    const uint32_t row = t / e0, pl = row / e1;
    const int x = b.lo[0] + (int)(t - row * e0), y = b.lo[1] + (int)(row - pl * e1), z = b.lo[2] + (int)pl;
    const int yx = x + cxp, yy = y + cyp, yz = z + czp;
    const bool in_face = yx >= b.lo[0] && yx < b.lo[0] + b.ex[0] && yy >= b.lo[1] &&
                         yy < b.lo[1] + b.ex[1] && yz >= b.lo[2] && yz < b.lo[2] + b.ex[2];
    const uint64_t cc = g.cell(z, y, x), cy = g.cell(yz, yy, yx);
    if (in_face && cy < cc) return;  // the thread of (y, k) does this pair
    const R ub0 = fs.ub[blockIdx.z][0], ub1 = fs.ub[blockIdx.z][1], ub2 = fs.ub[blockIdx.z][2];
    // c_k = -c_kp
    const R cu_k = (R)(-cxp) * ub0 + (R)(-cyp) * ub1 + (R)(-czp) * ub2;
    const R t_y = (R)2 * wk * rho[cy] * cu_k * cs2inv;
    R* const own = n + g.at(k, -cxp, -cyp, -czp) + cc;
    R* const dst = n + g.at(kp, cxp, cyp, czp) + cy;
    const R v = *own;
    if (fs.t) {
        // (c, kp) was pushed to *dst, and (y, k) to *own
        if (!on_faces(fs.saved, g, x, y, z)) fs.t[g.at(kp, cxp, cyp, czp) + (int64_t)cc] = *dst;
        if (in_face && !on_faces(fs.saved, g, yx, yy, yz)) fs.t[g.at(k, -cxp, -cyp, -czp) + (int64_t)cy] = v;
    }
    *dst = v - t_y;
    if (in_face) {
        // op (y, k): its own term t(y, c_kp of it = c_k) is t_y, then c's
        const R cu_kp = (R)cxp * ub0 + (R)cyp * ub1 + (R)czp * ub2;
        const R t_c = (R)2 * wk * rho[cc] * cu_kp * cs2inv;
        *own = (v - t_y) - t_c;
    }
}

// Which of the reference's two periodic copies apply: east-west and
// north-south (Boundary.cpp:223-281).
struct Periodic {
    int ew, ns;
};

Periodic periodic_of(const plb_boundary* bc) {
    Periodic p;
    p.ew = bc->type[0] == kPeriodic && bc->type[1] == kPeriodic;
    p.ns = bc->type[2] == kPeriodic && bc->type[3] == kPeriodic;
    return p;
}

// Boundary::_apply_periodicity_east_west (Boundary.cpp:234-251): for
// z in 1..Z, y in 1..Y: n(1, k) = n(X+1, k) for c_kx > 0, n(X, k) = n(0, k)
// for c_kx < 0; then _north_south (264-281) likewise with x in 1..X.  Both
// copy from halo slots of interior rows, which neither writes, so one launch
// does both (blockIdx.z the axis, blockIdx.y the direction); on the slots
// that both write, the later north-south copy stands.
template <int Q, class R>
__global__ void k_periodic(LitDims g, Periodic per, R* __restrict__ n) {
    const int axis = (int)blockIdx.z, k = 1 + (int)blockIdx.y;
    if (axis == 0 ? !per.ew : !per.ns) return;
    int cx = 0, cy = 0, cz = 0;
#pragma unroll
    for (int j = 1; j < Q; ++j)
        if (j == k) {
            cx = Lat<Q>::cx(j);
            cy = Lat<Q>::cy(j);
            cz = Lat<Q>::cz(j);
        }
    const int ck = axis == 0 ? cx : cy;
    if (ck == 0) return;
    const uint32_t other = (uint32_t)(axis == 0 ? g.Y : g.X);
    const uint32_t t = blockIdx.x * blockDim.x + threadIdx.x;
    const uint32_t zr = t / other;
    if (zr >= (uint32_t)g.Z) return;
    const int a = 1 + (int)(t - zr * other), z = 1 + (int)zr;
    const int hi = axis == 0 ? g.X : g.Y;
    const int to = ck > 0 ? 1 : hi, from = ck > 0 ? hi + 1 : 0;
    if (axis == 0 && per.ns && ((cy > 0 && a == 1) || (cy < 0 && a == g.Y))) return;
    const uint64_t dst = axis == 0 ? g.cell(z, a, to) : g.cell(z, to, a);
    const uint64_t src = axis == 0 ? g.cell(z, a, from) : g.cell(z, from, a);
    R* const nk = n + g.at(k, cx, cy, cz);
    nk[dst] = nk[src];
}

// Where an interior cell finds its population k when the periodic copies are
// folded into the kernel that reads n next instead of run: at the slot the
// copy that stands would take it from, relative to the cell's own slot (0
// away from the seams).  The copies read halo slots only, which the folded
// kernels do not write.
struct Seam {
    uint32_t xp, xm;  // x from which c_x > 0, c_x < 0 come
    int64_t yp, ym;   // and the shift of the row (uniform) for c_y > 0, c_y < 0
};
__device__ inline Seam seam_of(const LitDims& g, const Periodic& per, int x, int y) {
    Seam s;
    s.xp = per.ew && x == 1 ? (uint32_t)g.X + 1u : (uint32_t)x;
    s.xm = per.ew && x == g.X ? 0u : (uint32_t)x;
    s.yp = per.ns && y == 1 ? (int64_t)g.Y * g.nx : 0;
    s.ym = per.ns && y == g.Y ? -(int64_t)g.Y * g.nx : 0;
    return s;
}
template <int Q>
__device__ inline int64_t seam_row(const Seam& s, int k) {
    const int cy = Lat<Q>::cy(k);
    return cy > 0 ? s.yp : (cy < 0 ? s.ym : 0);
}
template <int Q>
__device__ inline uint32_t seam_x(const Seam& s, int k, uint32_t x) {
    const int cx = Lat<Q>::cx(k);
    return cx == 0 || seam_row<Q>(s, k) != 0 ? x : (cx > 0 ? s.xp : s.xm);
}

// CalcMoments::_get_local_moments (CalcMoments.hpp:22-37): rho = sum_k n_k,
// u = (sum_k n_k c_k) * (1 / rho), k ascending.
template <int Q, class R>
struct MomentSum {
    R rl = (R)0, u0 = (R)0, u1 = (R)0, u2 = (R)0;
    __device__ void add(int k, R nk) {
        rl += nk;
        u0 += nk * (R)Lat<Q>::cx(k);
        u1 += nk * (R)Lat<Q>::cy(k);
        u2 += nk * (R)Lat<Q>::cz(k);
    }
    __device__ void finish(R& rho, R (&u)[3]) const {
        const R ri = (R)1 / rl;
        rho = rl;
        u[0] = u0 * ri;
        u[1] = u1 * ri;
        u[2] = u2 * ri;
    }
};

// Boundary::_set_velocity / _set_density (Boundary.cpp:150-187) on one face.
template <class R>
__global__ void k_set_face(LitDims g, FaceBox b, R* __restrict__ dst, int vlen, R v0, R v1, R v2) {
    const uint64_t t = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (t >= b.count()) return;
    const int x = b.lo[0] + (int)(t % b.ex[0]);
    const int y = b.lo[1] + (int)((t / b.ex[0]) % b.ex[1]);
    const int z = b.lo[2] + (int)(t / ((uint64_t)b.ex[0] * b.ex[1]));
    const uint64_t c = g.cell(z, y, x);
    dst[c] = v0;
    if (vlen == 3) {
        dst[g.ncell + c] = v1;
        dst[2 * g.ncell + c] = v2;
    }
}

// Boundary::reset (Boundary.cpp:58-89, 150-187) for one interior cell: the
// faces in order, a later face overwriting an earlier one, as the per-face
// k_set_face launches of lit_reset_velocity and lit_reset_density do.  Face f
// is the layer at coordinate X|Y|Z (f even) or 1 (f odd) on axis f / 2, all
// interior cells of the other two axes (Boundary.cpp:113-148).
template <class R>
struct FaceResets {
    int has_vel[6], noslip[6];
    R vel[6][3];
    R rho_s;
};

template <class R>
__device__ inline void apply_resets(const FaceResets<R>& fr, const LitDims& g, int x, int y, int z, R& rho,
                                    R (&u)[3]) {
    const int co[3] = {x, y, z}, dim[3] = {g.X, g.Y, g.Z};
#pragma unroll
    for (int f = 0; f < 6; ++f) {
        if (!fr.has_vel[f] || co[f >> 1] != ((f & 1) == 0 ? dim[f >> 1] : 1)) continue;
        u[0] = fr.vel[f][0];
        u[1] = fr.vel[f][1];
        u[2] = fr.vel[f][2];
    }
#pragma unroll
    for (int f = 0; f < 6; ++f)
        if (fr.noslip[f] && co[f >> 1] == ((f & 1) == 0 ? dim[f >> 1] : 1)) rho = fr.rho_s;
}

// CalcMoments::_get_local_moments (CalcMoments.hpp:22-37) on interior cells,
// with the resets that follow it (none: fr empty).  The populations are read
// with non-temporal loads (measured 3-9% faster for this stage on MI355X).
template <int Q, class R>
__global__ void k_moments(LitDims g, const R* __restrict__ n, R* __restrict__ rho, R* __restrict__ u,
                          FaceResets<R> fr) {
    const int x = blockIdx.x * blockDim.x + threadIdx.x + 1;
    const int y = blockIdx.y + 1, z = blockIdx.z + 1;
    if (x > g.X) return;
    const uint64_t c = g.cell(z, y, x);
    MomentSum<Q, R> m;
#pragma unroll
    for (int k = 0; k < Q; ++k) m.add(k, __builtin_nontemporal_load(n + g.at<Q>(k) + c));
    R rl, um[3];
    m.finish(rl, um);
    apply_resets(fr, g, x, y, z, rl, um);
    rho[c] = rl;
    u[c] = um[0];
    u[g.ncell + c] = um[1];
    u[2 * g.ncell + c] = um[2];
}

// Which moments the folded kernel stores: all of them, or (inside plb_step,
// where the next kernel computes them again before anything reads them) only
// the densities that the no-slip pass of the step in progress reads: those of
// the face layers of the no-slip faces and of the layers next to them.
struct MomentStores {
    int all;
    unsigned noslip;  // the no-slip faces, a bit each
};
__device__ inline bool near_noslip(unsigned faces, const LitDims& g, int x, int y, int z) {
    return ((faces & 1u) && x >= g.X - 1) || ((faces & 2u) && x <= 2) || ((faces & 4u) && y >= g.Y - 1) ||
           ((faces & 8u) && y <= 2) || ((faces & 16u) && z >= g.Z - 1) || ((faces & 32u) && z <= 2);
}

// The previous step's periodic copies, moments and resets (Boundary,
// CalcMoments) folded into this step's collision and push, inside plb_step or
// for staged calls that the C ABI deferred until the push.
// Each population is read where the periodic copy would have put it from
// (the slot it would have written is this cell's own, which the in-place
// store below overwrites).  rho and u are computed exactly as k_moments and
// the resets leave them, stored as ms says, and used by the collision at once;
// n and t end as k_collide_push leaves them.  Bound by memory: folding the
// periodic copies in and leaving the dead rho and u stores out took the step
// of plb_step from 252 to 221 us (D3Q19 128^3 FP64: 38 instead of 42 values
// per cell, two launches fewer) and from 10.6 to 8.1 us (D2Q9 256 x 64 FP64).
//
// In-place stores: as in k_collide_push, and fewer still (next_known) where
// plb_step goes on with another of these kernels, the same per and no-slip
// faces and nothing read in between: of the slots no push writes, that step
// reads (c, k) itself only where no periodic copy takes its place, and its
// no-slip pass only those of its face cells.  All of the outer layer's values
// in place (38 one-lane stores per row of a lattice periodic in x, each into
// lines of its own) and stores along c_k cost 191 us per step at 128^3 FP64;
// the stores that remain, 157; whole lines (LitDims), 132, where the packed
// form took 160 (256^3 FP64 990 and 1,209, D2Q9 4000 x 4000 465 and 523): 4.8 TB/s
// of the 38 values per cell at 128^3, 5.2 at 256^3, bound by memory.
template <int Q, class R>
__global__ void k_moments_collide_push(LitDims g, R* __restrict__ n, R* __restrict__ rho, R* __restrict__ u,
                                       R* __restrict__ t, Periodic per, FaceResets<R> fr, MomentStores ms,
                                       int next_known, R tau, R om, R omm, R F0, R F1, R F2) {
    const int x = blockIdx.x * blockDim.x + threadIdx.x + 1;
    const int y = blockIdx.y + 1, z = blockIdx.z + 1;
    if (x > g.X) return;
    const uint64_t c = g.cell(z, y, x);
    // addresses: a uniform row of the population's array, and x
    const int64_t row = (int64_t)g.cell(z, y, 0);
    const Seam sm = seam_of(g, per, x, y);
    R nv[Q];
    MomentSum<Q, R> m;
#pragma unroll
    for (int k = 0; k < Q; ++k)
        nv[k] = (n + g.at<Q>(k) + row + seam_row<Q>(sm, k))[seam_x<Q>(sm, k, (uint32_t)x)];
#pragma unroll
    for (int k = 0; k < Q; ++k) m.add(k, nv[k]);
    R rl, um[3];
    m.finish(rl, um);
    apply_resets(fr, g, x, y, z, rl, um);
    if (ms.all || near_noslip(ms.noslip, g, x, y, z)) rho[c] = rl;
    if (ms.all) {
        u[c] = um[0];
        u[g.ncell + c] = um[1];
        u[2 * g.ncell + c] = um[2];
    }
    R uu[3], usq;
    updated_u(um[0], um[1], um[2], rl, tau, F0, F1, F2, uu, usq);
#pragma unroll
    for (int k = 0; k < Q; ++k) {
        nv[k] = collide_value<Q, R>(k, nv[k], rl, uu, usq, om, omm);
        (t + g.to<Q>(k) + row)[(uint32_t)x] = nv[k];
    }
    const bool any = !next_known || on_faces(ms.noslip, g, x, y, z);
#pragma unroll
    for (int k = 1; k < Q; ++k) {
        const bool own = any || (seam_row<Q>(sm, k) == 0 && seam_x<Q>(sm, k, (uint32_t)x) == (uint32_t)x);
        if (own && from_halo<Q>(g, k, x, y, z)) (n + g.at<Q>(k) + row)[(uint32_t)x] = nv[k];
    }
}

// Where value v of cell 0 of a field lies.
struct ValueSlots {
    int64_t off[27];
};

// Upload: host AoS -> device SoA with dtype conversion.  compact: host cells
// are interior only (X*Y*Z); otherwise the full halo'd array.
template <class H, class R>
__global__ void k_upload(LitDims g, const H* __restrict__ host, R* __restrict__ dev, ValueSlots sl, int vlen,
                         int compact, uint64_t total) {
    for (uint64_t t = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x; t < total;
         t += (uint64_t)gridDim.x * blockDim.x) {
        const int v = (int)(t % vlen);
        const uint64_t hc = t / vlen;
        const int o = compact ? 1 : 0, X = g.X + 2 - 2 * o, Y = g.ny - 2 * o;
        const int x = (int)(hc % X), y = (int)((hc / X) % Y), z = (int)(hc / ((uint64_t)X * Y));
        dev[sl.off[v] + (int64_t)g.cell(z + o, y + o, x + o)] = (R)host[t];
    }
}

// Download: value v of cell c of the full halo'd array (o = 0), or of the
// interior (o = 1).
template <class R>
struct GetValue {
    const R* dev;
    LitDims g;
    ValueSlots sl;
    FastDiv dX, dY;  // a row, a column of 2^32 cells in all is part of a state larger than any device
    int o;
    __device__ R operator()(uint64_t c, uint32_t v) const {
        const uint32_t row = fdiv((uint32_t)c, dX), z = fdiv(row, dY);
        const int x = (int)((uint32_t)c - row * dX.d), y = (int)(row - z * dY.d);
        return dev[sl.off[v] + (int64_t)g.cell((int)z + o, y + o, x + o)];
    }
};

// FP64 sums over interior cells of rho and rho*u (two deterministic passes).
template <class R>
__global__ void k_global_partial(LitDims g, const R* __restrict__ rho, const R* __restrict__ u,
                                 double* __restrict__ partial) {
    __shared__ double sh[4][kThreads];
    double acc[4] = {0, 0, 0, 0};
    const uint64_t total = (uint64_t)g.X * g.Y * g.Z;
    for (uint64_t i = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x; i < total;
         i += (uint64_t)gridDim.x * blockDim.x) {
        const int x = (int)(i % g.X) + 1, y = (int)((i / g.X) % g.Y) + 1,
                  z = (int)(i / ((uint64_t)g.X * g.Y)) + 1;
        const uint64_t c = g.cell(z, y, x);
        const double r = (double)rho[c];
        acc[0] += r;
        for (int d = 0; d < 3; ++d) acc[1 + d] += r * (double)u[d * g.ncell + c];
    }
    for (int d = 0; d < 4; ++d) sh[d][threadIdx.x] = acc[d];
    __syncthreads();
    for (unsigned s = kThreads / 2; s > 0; s >>= 1) {
        if (threadIdx.x < s)
            for (int d = 0; d < 4; ++d) sh[d][threadIdx.x] += sh[d][threadIdx.x + s];
        __syncthreads();
    }
    if (threadIdx.x == 0)
        for (int d = 0; d < 4; ++d) partial[4 * blockIdx.x + d] = sh[d][0];
}

__global__ void k_global_final(const double* __restrict__ partial, int nblocks, double* __restrict__ out) {
    if (threadIdx.x != 0 || blockIdx.x != 0) return;
    double a[4] = {0, 0, 0, 0};
    for (int b = 0; b < nblocks; ++b)
        for (int d = 0; d < 4; ++d) a[d] += partial[4 * b + d];
    for (int d = 0; d < 4; ++d) out[d] = a[d];
}

int ensure_scratch(plb_state* s, size_t bytes) {
    if (s->scratch_bytes >= bytes) return PLB_OK;
    if (s->scratch) PLB_HIP_TRY(hipFree(s->scratch));
    s->scratch = nullptr;
    s->scratch_bytes = 0;
    PLB_HIP_TRY(hipMalloc(&s->scratch, bytes));
    s->scratch_bytes = bytes;
    return PLB_OK;
}

// The per-cell stages (collide, push, moments) launch one block per x-row
// piece of up to 256 interior cells (whole wavefronts), the row's y and z
// taken from the block index.
unsigned interior_block(const plb_state* s) {
    const unsigned w = (unsigned)((s->X + 63) / 64) * 64u;
    return w < 256u ? w : 256u;
}
dim3 interior_grid(const plb_state* s) {
    const unsigned b = interior_block(s);
    return dim3((unsigned)((s->X + b - 1) / b), (unsigned)s->Y, (unsigned)s->Z);
}

// Stores the in-place values the last collide+push kernel left out, before anything reads ntmp or changes n.
int lit_ntmp_restore(plb_state* s) {
    if (!s->lit_ntmp_folded) return PLB_OK;
    const LitDims g = dims_of(s);
    const int rc = with_qr(s, [&](auto qc, auto rr) {
        constexpr int Q = decltype(qc)::value;
        using R = decltype(rr);
        hipLaunchKernelGGL((k_ntmp_restore<Q, R>), interior_grid(s), dim3(interior_block(s)), 0, s->stream, g,
                           s->lit_saved, (const R*)s->buf[s->cur], (R*)s->buf[s->cur ^ 1]);
        PLB_HIP_TRY(hipGetLastError());
        return PLB_OK;
    });
    if (rc == PLB_OK) s->lit_ntmp_folded = false;
    return rc;
}

}  // namespace

// ------------------------------------------------------------ launchers ----
// Device layout of a state (LitDims): rows of whole lines and the shift's two
// planes, up to any size below 1 GiB per buffer and up to an eighth more memory
// above; there rows of X + 2 cells and the two planes, or the packed form, if the
// form before takes more.  packed: the smallest form.
void lit_layout(plb_state* s, bool packed) {
    const uint64_t line = 128 / s->sbytes, X2 = (uint64_t)s->X + 2, ny = (uint64_t)s->Y + 2, nz = (uint64_t)s->Z + 2;
    const uint64_t least = X2 * ny * nz;
    auto stride = [&](uint64_t nx, uint64_t* base) {
        const uint64_t far = nx * ny + nx + 1;  // of a direction's shift
        *base = (far + line - 1) / line * line + line - 1;
        return (*base + nx * ny * nz + far + line - 1) / line * line;
    };
    auto fits = [&](uint64_t ps) { return ps * s->q * s->sbytes <= (1ull << 30) || ps * 8 <= least * 9; };
    for (uint64_t nx : {(X2 + line - 1) / line * line, X2}) {
        uint64_t base;
        const uint64_t ps = stride(nx, &base);
        if (packed || !fits(ps)) continue;
        s->lit_nx = (int)nx;
        s->lit_base = base;
        s->pstride = ps;
        return;
    }
    s->lit_nx = (int)X2;
    s->lit_base = 0;
    s->pstride = least;
}
uint64_t lit_cells(const plb_state* s) { return (uint64_t)s->lit_nx * (s->Y + 2) * (s->Z + 2); }

int lit_initialize(plb_state* s, double rho0, const double u0[3], const plb_init_spec* init,
                   const double* tg_dev) {
    const LitDims g = dims_of(s);
    const int kind = init ? init->kind : PLB_INIT_UNIFORM;
    const uint64_t seed = init ? init->seed : 0;
    const double amp = init ? init->amp : 0.0;
    return with_qr(s, [&](auto qc, auto rr) {
        constexpr int Q = decltype(qc)::value;
        using R = decltype(rr);
        hipLaunchKernelGGL((k_init<Q, R>), dim3(blocks_for(g.ncell, kThreads)), dim3(kThreads), 0,
                           s->stream, g, (R*)s->buf[s->cur], (R*)s->buf[s->cur ^ 1], (R*)s->rho,
                           (R*)s->u, rho0, u0[0], u0[1], u0[2], kind, seed, amp, tg_dev);
        PLB_HIP_TRY(hipGetLastError());
        s->lit_ntmp_folded = false;
        return PLB_OK;
    });
}

namespace {
// tau and omega = 1/tau as CollisionSRT.cpp:19-20 hold them, and 1 - omega.
template <class R>
void relaxation(double tau, R* tr, R* om, R* omm) {
    *tr = (R)tau;
    if (std::is_same<R, float>::value)
        *om = (R)(1. / (double)*tr);
    else
        *om = (R)(1.0 / tau);
    *omm = (R)1 - *om;
}
}  // namespace

int lit_collide(plb_state* s, double tau, const double F[3]) {
    const LitDims g = dims_of(s);
    const int rc = lit_ntmp_restore(s);  // the collision changes the n that ntmp is kept in
    if (rc) return rc;
    return with_qr(s, [&](auto qc, auto rr) {
        constexpr int Q = decltype(qc)::value;
        using R = decltype(rr);
        R tr, om, omm;
        relaxation(tau, &tr, &om, &omm);
        hipLaunchKernelGGL((k_collide<Q, R>), interior_grid(s), dim3(interior_block(s)), 0, s->stream, g,
                           (R*)s->buf[s->cur], (const R*)s->rho, (const R*)s->u, tr, om, omm, (R)F[0], (R)F[1],
                           (R)F[2]);
        PLB_HIP_TRY(hipGetLastError());
        return PLB_OK;
    });
}

int lit_collide_push(plb_state* s, double tau, const double F[3]) {
    const LitDims g = dims_of(s);
    const int rc = with_qr(s, [&](auto qc, auto rr) {
        constexpr int Q = decltype(qc)::value;
        using R = decltype(rr);
        R tr, om, omm;
        relaxation(tau, &tr, &om, &omm);
        hipLaunchKernelGGL((k_collide_push<Q, R>), interior_grid(s), dim3(interior_block(s)), 0, s->stream, g,
                           (R*)s->buf[s->cur], (const R*)s->rho, (const R*)s->u, (R*)s->buf[s->cur ^ 1], tr, om,
                           omm, (R)F[0], (R)F[1], (R)F[2]);
        PLB_HIP_TRY(hipGetLastError());
        return PLB_OK;
    });
    if (rc == PLB_OK) {
        s->cur ^= 1;  // std::swap(simdata.ntmp, simdata.n)
        s->lit_ntmp_folded = true;
        s->lit_saved = 0;
    }
    return rc;
}

namespace {
// The resets of bc_vel's velocities and bc_rho's solid density (null: none).
template <class R>
FaceResets<R> face_resets(const plb_boundary* bc_vel, const plb_boundary* bc_rho) {
    FaceResets<R> fr;
    for (int f = 0; f < 6; ++f) {
        fr.has_vel[f] = bc_vel && bc_vel->has_vel[f] != 0;
        fr.noslip[f] = bc_rho && bc_rho->type[f] == kNoslip;
        for (int i = 0; i < 3; ++i) fr.vel[f][i] = bc_vel ? (R)bc_vel->vel[f][i] : (R)0;
    }
    fr.rho_s = bc_rho ? (R)bc_rho->rho_s : (R)0;
    return fr;
}
}  // namespace

int lit_moments_collide_push(plb_state* s, double tau, const double F[3], const plb_boundary* bc_per,
                             const plb_boundary* bc_vel, const plb_boundary* bc_rho, const plb_boundary* bc_noslip,
                             bool next_known) {
    const LitDims g = dims_of(s);
    const int rc = with_qr(s, [&](auto qc, auto rr) {
        constexpr int Q = decltype(qc)::value;
        using R = decltype(rr);
        R tr, om, omm;
        relaxation(tau, &tr, &om, &omm);
        const Periodic per = bc_per ? periodic_of(bc_per) : Periodic{0, 0};
        MomentStores ms;
        ms.all = bc_noslip == nullptr;
        ms.noslip = 0;
        for (int f = 0; bc_noslip && f < 6; ++f) ms.noslip |= bc_noslip->type[f] == kNoslip ? 1u << f : 0u;
        hipLaunchKernelGGL((k_moments_collide_push<Q, R>), interior_grid(s), dim3(interior_block(s)), 0, s->stream,
                           g, (R*)s->buf[s->cur], (R*)s->rho, (R*)s->u, (R*)s->buf[s->cur ^ 1], per,
                           face_resets<R>(bc_vel, bc_rho), ms, next_known ? 1 : 0, tr, om, omm, (R)F[0], (R)F[1], (R)F[2]);
        PLB_HIP_TRY(hipGetLastError());
        return PLB_OK;
    });
    if (rc == PLB_OK) {
        s->cur ^= 1;  // std::swap(simdata.ntmp, simdata.n)
        s->lit_ntmp_folded = true;
        s->lit_saved = 0;
    }
    return rc;
}

int lit_push(plb_state* s) {
    const LitDims g = dims_of(s);
    const int rc = with_qr(s, [&](auto qc, auto rr) {
        constexpr int Q = decltype(qc)::value;
        using R = decltype(rr);
        hipLaunchKernelGGL((k_push<Q, R>), interior_grid(s), dim3(interior_block(s)), 0, s->stream, g,
                           (const R*)s->buf[s->cur], (R*)s->buf[s->cur ^ 1]);
        PLB_HIP_TRY(hipGetLastError());
        return PLB_OK;
    });
    if (rc == PLB_OK) {
        s->cur ^= 1;  // std::swap(simdata.ntmp, simdata.n)
        s->lit_ntmp_folded = false;  // the push wrote every slot that was not in place
    }
    return rc;
}

int lit_noslip(plb_state* s, const plb_boundary* bc, bool ntmp_read) {
    const LitDims g = dims_of(s);
    const int dims[3] = {s->X, s->Y, s->Z};
    for (int f = 0; f < 6;) {
        if (bc->type[f] != kNoslip) {
            ++f;
            continue;
        }
        if (!bc->has_vel[f])
            return fail(PLB_ERR_OUT_OF_RANGE, "no-slip face without a prescribed velocity");
        // Both faces of an axis in one launch, from three layers on: the high
        // face reads its own layer and writes the populations that leave it
        // inwards one layer below, the low face likewise one layer above;
        // with two layers each would write into the layer the other reads.
        const bool both = f % 2 == 0 && bc->type[f + 1] == kNoslip && bc->has_vel[f + 1] && dims[f / 2] >= 3;
        const int nf = both ? 2 : 1;
        const bool save = s->lit_ntmp_folded && ntmp_read;
        const int rc = with_qr(s, [&](auto qc, auto rr) {
            constexpr int Q = decltype(qc)::value;
            using R = decltype(rr);
            NoslipFaces<R> fs;
            for (int i = 0; i < 2; ++i) {
                const int fi = f + (i < nf ? i : 0);
                fs.box[i] = face_box(fi, s->X, s->Y, s->Z);
                for (int d = 0; d < 3; ++d) fs.ub[i][d] = (R)bc->vel[fi][d];
            }
            fs.t = save ? (R*)s->buf[s->cur ^ 1] : nullptr;
            fs.saved = s->lit_saved;
            // a face of 2^32 cells is part of a state larger than any device
            const uint32_t total = (uint32_t)fs.box[0].count();
            const R cs2inv = (R)1 / (R)(1.0 / 3.0);
            hipLaunchKernelGGL((k_noslip<Q, R>), dim3(blocks_for(total, kThreads), Q - 1, (unsigned)nf),
                               dim3(kThreads), 0, s->stream, g, fs, (R*)s->buf[s->cur], (const R*)s->rho, cs2inv,
                               total);
            PLB_HIP_TRY(hipGetLastError());
            return PLB_OK;
        });
        if (rc) return rc;
        for (int i = 0; save && i < nf; ++i) s->lit_saved |= 1u << (f + i);
        f += nf;
    }
    return PLB_OK;
}

int lit_noslip_noalloc(plb_state* s, const plb_boundary* bc) {
    // the documented limit of the entry point: a face's values within 16 MiB
    constexpr size_t kLimit = (size_t)16 << 20;
    const size_t rbytes = s->variant == kF64 ? sizeof(double) : sizeof(float);
    for (int f = 0; f < 6; ++f) {
        if (bc->type[f] != kNoslip) continue;
        const uint64_t need = face_box(f, s->X, s->Y, s->Z).count() * (uint64_t)(s->q - 1) * rbytes;
        if (need > kLimit)
            return fail(PLB_ERR_INVALID_ARGUMENT, "no-slip face of " + std::to_string(need) +
                                                      " bytes exceeds the no-allocation limit of 16 MiB; use "
                                                      "plb_apply_noslip");
    }
    return lit_noslip(s, bc, true);
}

int lit_periodic(plb_state* s, const plb_boundary* bc) {
    const LitDims g = dims_of(s);
    const Periodic per = periodic_of(bc);
    if (!per.ew && !per.ns) return PLB_OK;
    return with_qr(s, [&](auto qc, auto rr) {
        constexpr int Q = decltype(qc)::value;
        using R = decltype(rr);
        // a seam of 2^32 cells is part of a state larger than any device
        const uint64_t ew = per.ew ? (uint64_t)s->Z * s->Y : 0, ns = per.ns ? (uint64_t)s->Z * s->X : 0;
        hipLaunchKernelGGL((k_periodic<Q, R>), dim3(blocks_for(ew > ns ? ew : ns, kThreads), Q - 1, per.ns ? 2 : 1),
                           dim3(kThreads), 0, s->stream, g, per, (R*)s->buf[s->cur]);
        PLB_HIP_TRY(hipGetLastError());
        return PLB_OK;
    });
}

int lit_moments(plb_state* s, const plb_boundary* bc_vel, const plb_boundary* bc_rho) {
    const LitDims g = dims_of(s);
    return with_qr(s, [&](auto qc, auto rr) {
        constexpr int Q = decltype(qc)::value;
        using R = decltype(rr);
        hipLaunchKernelGGL((k_moments<Q, R>), interior_grid(s), dim3(interior_block(s)), 0, s->stream, g,
                           (const R*)s->buf[s->cur], (R*)s->rho, (R*)s->u, face_resets<R>(bc_vel, bc_rho));
        PLB_HIP_TRY(hipGetLastError());
        return PLB_OK;
    });
}

int lit_reset_velocity(plb_state* s, const plb_boundary* bc) {
    const LitDims g = dims_of(s);
    for (int f = 0; f < 6; ++f) {
        if (!bc->has_vel[f]) continue;
        const FaceBox b = face_box(f, s->X, s->Y, s->Z);
        const int rc = with_qr(s, [&](auto, auto rr) {
            using R = decltype(rr);
            hipLaunchKernelGGL((k_set_face<R>), dim3(blocks_for(b.count(), kThreads)), dim3(kThreads),
                               0, s->stream, g, b, (R*)s->u, 3, (R)bc->vel[f][0], (R)bc->vel[f][1],
                               (R)bc->vel[f][2]);
            PLB_HIP_TRY(hipGetLastError());
            return PLB_OK;
        });
        if (rc) return rc;
    }
    return PLB_OK;
}

int lit_reset_density(plb_state* s, const plb_boundary* bc) {
    const LitDims g = dims_of(s);
    for (int f = 0; f < 6; ++f) {
        if (bc->type[f] != kNoslip) continue;
        const FaceBox b = face_box(f, s->X, s->Y, s->Z);
        const int rc = with_qr(s, [&](auto, auto rr) {
            using R = decltype(rr);
            hipLaunchKernelGGL((k_set_face<R>), dim3(blocks_for(b.count(), kThreads)), dim3(kThreads),
                               0, s->stream, g, b, (R*)s->rho, 1, (R)bc->rho_s, (R)0, (R)0);
            PLB_HIP_TRY(hipGetLastError());
            return PLB_OK;
        });
        if (rc) return rc;
    }
    return PLB_OK;
}

int lit_transfer(plb_state* s, int field, int layout, int dtype, void* host, bool upload) {
    const LitDims g = dims_of(s);
    if ((field == PLB_FIELD_NTMP && !upload) || (field == PLB_FIELD_N && upload)) {
        const int r = lit_ntmp_restore(s);
        if (r) return r;
    }
    int vlen;
    void* dev;
    switch (field) {
        case PLB_FIELD_RHO: vlen = 1; dev = s->rho; break;
        case PLB_FIELD_U: vlen = 3; dev = s->u; break;
        case PLB_FIELD_N: vlen = s->q; dev = s->buf[s->cur]; break;
        case PLB_FIELD_NTMP: vlen = s->q; dev = s->buf[s->cur ^ 1]; break;
        default: return fail(PLB_ERR_INVALID_ARGUMENT, "unknown field");
    }
    ValueSlots sl;
    const bool pop = field == PLB_FIELD_N || field == PLB_FIELD_NTMP;
    const int slots = with_q(s->q, [&](auto qc) {
        using L = Lat<decltype(qc)::value>;
        for (int v = 0; v < vlen; ++v)
            sl.off[v] = pop ? g.at(v, L::cx(v), L::cy(v), L::cz(v)) : (int64_t)(v * g.ncell);
        return PLB_OK;
    });
    if (slots) return slots;
    const int compact = layout == PLB_LAYOUT_COMPACT ? 1 : 0;
    const uint64_t cells = compact ? (uint64_t)s->X * s->Y * s->Z : s->ncell;
    const uint64_t total = cells * vlen;
    if (!upload) {
        return with_qr(s, [&](auto, auto rr) {
            using R = decltype(rr);
            auto read = [&](auto hh) {
                using H = decltype(hh);
                const size_t cell_bytes = vlen * sizeof(H);
                const GetValue<R> get{(const R*)dev, g, sl, make_fastdiv((uint32_t)(s->X + 2 - 2 * compact)),
                                      make_fastdiv((uint32_t)(s->Y + 2 - 2 * compact)), compact};
                return host_read(
                    s->ring, s->device, s->stream, cells, cell_bytes,
                    [&](uint64_t first, uint64_t n, void* slot) {
                        return host_fill<H>(get, first, n, vlen, slot, s->stream);
                    },
                    [&](uint64_t first, uint64_t n, const void* slot) {
                        std::memcpy((char*)host + first * cell_bytes, slot, n * cell_bytes);
                    });
            };
            return dtype == PLB_DTYPE_F64 ? read(double()) : read(float());
        });
    }
    const size_t hbytes = total * (dtype == PLB_DTYPE_F64 ? 8 : 4);
    void* stage = nullptr;
    PLB_HIP_TRY(hipMalloc(&stage, hbytes));
    int rc = PLB_OK;
    hipError_t e = hipMemcpyAsync(stage, host, hbytes, hipMemcpyHostToDevice, s->stream);
    if (e != hipSuccess) rc = fail(PLB_ERR_HIP, std::string("upload: ") + hipGetErrorString(e));
    if (rc == PLB_OK) {
        rc = with_qr(s, [&](auto, auto rr) {
            using R = decltype(rr);
            if (dtype == PLB_DTYPE_F64)
                hipLaunchKernelGGL((k_upload<double, R>), dim3(stride_blocks(total, kThreads)),
                                   dim3(kThreads), 0, s->stream, g, (const double*)stage, (R*)dev, sl, vlen,
                                   compact, total);
            else
                hipLaunchKernelGGL((k_upload<float, R>), dim3(stride_blocks(total, kThreads)),
                                   dim3(kThreads), 0, s->stream, g, (const float*)stage, (R*)dev, sl, vlen,
                                   compact, total);
            PLB_HIP_TRY(hipGetLastError());
            return PLB_OK;
        });
    }
    e = hipStreamSynchronize(s->stream);
    (void)hipFree(stage);
    if (rc == PLB_OK && e != hipSuccess) rc = fail(PLB_ERR_HIP, hipGetErrorString(e));
    if (rc == PLB_OK && field == PLB_FIELD_NTMP) s->lit_ntmp_folded = false;
    return rc;
}

int lit_global(plb_state* s, double out[4]) {
    const LitDims g = dims_of(s);
    const int nb = 512;
    int rc = ensure_scratch(s, (size_t)(4 * nb + 4) * sizeof(double));
    if (rc) return rc;
    double* partial = (double*)s->scratch;
    rc = with_qr(s, [&](auto, auto rr) {
        using R = decltype(rr);
        hipLaunchKernelGGL((k_global_partial<R>), dim3(nb), dim3(kThreads), 0, s->stream, g,
                           (const R*)s->rho, (const R*)s->u, partial);
        PLB_HIP_TRY(hipGetLastError());
        hipLaunchKernelGGL(k_global_final, dim3(1), dim3(64), 0, s->stream, partial, nb, partial + 4 * nb);
        PLB_HIP_TRY(hipGetLastError());
        return PLB_OK;
    });
    if (rc) return rc;
    PLB_HIP_TRY(hipMemcpyAsync(out, partial + 4 * nb, 4 * sizeof(double), hipMemcpyDeviceToHost, s->stream));
    PLB_HIP_TRY(hipStreamSynchronize(s->stream));
    return PLB_OK;
}

}  // namespace plb
