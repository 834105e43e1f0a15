// One cell of the box-Vanka smoother and one node of the residual, written over an
// accessor of the neighbouring nodes, for the levels that are not marched plane by
// plane (st_coarse.hip).  The rows and their order of operations are those of Sten in
// st_kernels.hip (FINE: of the marching kernels in st_march.hip), the block solve is that
// of the marched smoother, so every kernel built on these gives the same bits in FP32 and
// BF16.
//
// An accessor A has, at node offsets (di, dj, dk) from its own node,
//   X(f, di, dj, dk)   field f of x (0: p, 1 + d: velocity d), in the compute type
//   F(di, dj, dk)      the flag byte, 0 outside the level
//   B(f, di, dj, dk), AL(d, di, dj, dk)   right-hand side and face penalty
//   MASK   whether a velocity must be masked by its flag.  On the levels under the
//          finest one the right-hand side of a fixed DOF is 0 and its x starts at 0 and
//          stays 0, so x is its own masked field and 12 of the 19 flags and all the
//          selects of a cell go (MASK = false); the finest level has any values there.
// X is 0 outside the level; with MASK a velocity there may be anything.
// Each velocity, edge curl and divergence of the stencil is named once here: a colour
// cell reads 36 masked velocities, 7 pressures and 19 flags, which is what its 7 rows
// need; evaluating the rows one by one re-derives them.
#pragma once
#include "st_common.h"

namespace st {

// masked velocities, divergences and edge curls around the accessor's node.  FINE: the
// sums are associated as in the kernels of the finest levels (st_march.hip), left to
// right; else as in Sten
template <typename C, int DIM, typename A, bool FINE = false> struct BoxSten {
    const A &a;
    __device__ __forceinline__ C W(int d, int di, int dj, int dk) const
    {
        if (DIM == 2 && d == 2) return C(0);
        const C v = a.X(1 + d, di, dj, dk);
        if (!A::MASK) return v;
        return ((a.F(di, dj, dk) >> (1 + d)) & 1) ? v : C(0);
    }
    __device__ __forceinline__ C dv(int i, int j, int k) const
    {
        C s = W(0, i + 1, j, k) - W(0, i, j, k) + W(1, i, j + 1, k) - W(1, i, j, k);
        if (FINE) return s + W(2, i, j, k + 1) - W(2, i, j, k);
        if (DIM == 3) s += W(2, i, j, k + 1) - W(2, i, j, k);
        return s;
    }
    __device__ __forceinline__ C gdiv(int i, int j, int k) const
    {
        const C d = dv(i, j, k);
        return (a.F(i, j, k) & 1) ? d : C(0);
    }
    __device__ __forceinline__ C ex(int i, int j, int k) const
    { return W(1, i, j, k) - W(1, i, j, k - 1) - W(2, i, j, k) + W(2, i, j - 1, k); }
    __device__ __forceinline__ C ey(int i, int j, int k) const
    { return W(2, i, j, k) - W(2, i - 1, j, k) - W(0, i, j, k) + W(0, i, j, k - 1); }
    __device__ __forceinline__ C ez(int i, int j, int k) const
    { return W(0, i, j, k) - W(0, i, j - 1, k) - W(1, i, j, k) + W(1, i - 1, j, k); }

    // row of the face d at offset (i, j, k): visc, then pressure, then penalty
    template <int d> __device__ __forceinline__ C face(int i, int j, int k) const
    {
        const int di = (d == 0), dj = (d == 1), dk = (d == 2);
        const C u = a.X(1 + d, i, j, k);
        const bool free = (a.F(i, j, k) >> (1 + d)) & 1;
        const C gl = gdiv(i - di, j - dj, k - dk), gh = gdiv(i, j, k);
        const C pl = a.X(0, i - di, j - dj, k - dk), ph = a.X(0, i, j, k);
        if (FINE) {
            C r;
            if (d == 0) r = gl - gh + ey(i, j, k + 1) - ey(i, j, k) + ez(i, j, k) - ez(i, j + 1, k);
            if (d == 1) r = gl - gh + ex(i, j, k) - ex(i, j, k + 1) + ez(i + 1, j, k) - ez(i, j, k);
            if (d == 2) r = gl - gh + ex(i, j + 1, k) - ex(i, j, k) + ey(i, j, k) - ey(i + 1, j, k);
            // (the smoother's high x face adds pressure and penalty as one term)
            if (d == 0 && i == 1) r += pl - ph + a.AL(d, i, j, k) * u;
            else r = r + pl - ph + a.AL(d, i, j, k) * u;
            return free ? r : u;
        }
        C r = gl - gh;
        if (DIM == 3) {
            if (d == 0) r += ey(i, j, k + 1) - ey(i, j, k) + ez(i, j, k) - ez(i, j + 1, k);
            if (d == 1) r += ex(i, j, k) - ex(i, j, k + 1) + ez(i + 1, j, k) - ez(i, j, k);
            if (d == 2) r += ex(i, j + 1, k) - ex(i, j, k) + ey(i, j, k) - ey(i + 1, j, k);
        } else {
            if (d == 0) r += ez(i, j, 0) - ez(i, j + 1, 0);
            if (d == 1) r += ez(i + 1, j, 0) - ez(i, j, 0);
        }
        r += pl - ph;
        r += a.AL(d, i, j, k) * u;
        return free ? r : u;
    }
    __device__ __forceinline__ C cell() const
    {
        const C d = dv(0, 0, 0), p = a.X(0, 0, 0, 0);
        return (a.F(0, 0, 0) & 1) ? d : p;
    }
};

// a / b and 1 / b of the block solve: IEEE, but on the finest levels in FP32 the
// hardware reciprocal (1 ulp)
template <bool FINE, typename C> __device__ __forceinline__ C box_quo(C a, C b)
{
    if constexpr (FINE && sizeof(C) == 4) return a * __builtin_amdgcn_rcpf(b);
    else return a / b;
}

// new values of the cell's pressure and of its low (u0) and high (u1) faces after the
// exact solve of its block: the Schur complement of the pressure in a free cell,
// Sherman-Morrison (K = E - b b^T) in a fixed one; ZERO: x is zero and not read
template <typename C, int DIM, bool ZERO, bool FINE = false, typename A>
__device__ __forceinline__ void box_cell(const A &a, float omega, C &pn, C *u0n, C *u1n)
{
    const BoxSten<C, DIM, A, FINE> s{a};
    const int fb = a.F(0, 0, 0);
    const C mc = (fb & 1) ? C(1) : C(0);
    const C NE = (DIM == 3) ? C(4) : C(2);
    C rp = a.B(0, 0, 0, 0);
    if (!ZERO) rp -= s.cell();
    C beta = C(0), tb = C(0);  // b^T E^-1 b, b^T E^-1 r_u
    C a0[3], a1[3], of[3], id[3], r0[3], r1[3], m0[3], m1[3];
#pragma unroll
    for (int d = 0; d < DIM; d++) {
        const int di = (d == 0), dj = (d == 1), dk = (d == 2);
        const int fh = a.F(di, dj, dk);
        m0[d] = ((fb >> (1 + d)) & 1) ? C(1) : C(0);
        m1[d] = ((fh >> (1 + d)) & 1) ? C(1) : C(0);
        const C c_lo = (C)(a.F(-di, -dj, -dk) & 1);
        const C c_hi = (C)(fh & 1);
        const C al0 = a.AL(d, 0, 0, 0), al1 = a.AL(d, di, dj, dk);
        a0[d] = m0[d] * (c_lo + mc + NE) + al0 + (C(1) - m0[d]) + (C(1) - mc) * m0[d];
        a1[d] = m1[d] * (mc + c_hi + NE) + al1 + (C(1) - m1[d]) + (C(1) - mc) * m1[d];
        of[d] = -m0[d] * m1[d];
        C rl = a.B(1 + d, 0, 0, 0);
        C rh = a.B(1 + d, di, dj, dk);
        if (!ZERO) {
            if (d == 0) { rl -= s.template face<0>(0, 0, 0); rh -= s.template face<0>(1, 0, 0); }
            if (d == 1) { rl -= s.template face<1>(0, 0, 0); rh -= s.template face<1>(0, 1, 0); }
            if (d == 2) { rl -= s.template face<2>(0, 0, 0); rh -= s.template face<2>(0, 0, 1); }
        }
        r0[d] = rl;
        r1[d] = rh;
        id[d] = box_quo<FINE>(C(1), a0[d] * a1[d] - of[d] * of[d]);
        // b_f = (-m0, m1), b_c = mc * b_f
        const C kb0 = id[d] * (a1[d] * (-m0[d]) - of[d] * m1[d]);
        const C kb1 = id[d] * (-of[d] * (-m0[d]) + a0[d] * m1[d]);
        const C kr0 = id[d] * (a1[d] * rl - of[d] * rh);
        const C kr1 = id[d] * (-of[d] * rl + a0[d] * rh);
        beta += (-m0[d]) * kb0 + m1[d] * kb1;
        tb += (-m0[d]) * kr0 + m1[d] * kr1;
    }
    const C Sc = (mc != C(0)) ? -beta : C(1);
    const C dp = (Sc != C(0)) ? box_quo<FINE>(rp - mc * tb, Sc) : C(0);
    const C gm = (mc != C(0)) ? dp : box_quo<FINE>(dp - tb, C(1) - beta);
    const C om = (C)omega;
    const C p0 = ZERO ? C(0) : a.X(0, 0, 0, 0);
    pn = p0 + om * dp;
#pragma unroll
    for (int d = 0; d < DIM; d++) {
        const int di = (d == 0), dj = (d == 1), dk = (d == 2);
        const C e0 = r0[d] + m0[d] * gm;   // r - b_f g, b_f = (-m0, m1)
        const C e1 = r1[d] - m1[d] * gm;
        const C u0 = ZERO ? C(0) : a.X(1 + d, 0, 0, 0);
        const C u1 = ZERO ? C(0) : a.X(1 + d, di, dj, dk);
        u0n[d] = u0 + om * id[d] * (a1[d] * e0 - of[d] * e1);
        u1n[d] = u1 + om * id[d] * (-of[d] * e0 + a0[d] * e1);
    }
}

// value at a 32-bit element offset from a uniform base
template <typename T> __device__ __forceinline__ T at(const T *p, unsigned i)
{
    return *reinterpret_cast<const T *>(reinterpret_cast<const char *>(p) + i * (unsigned)sizeof(T));
}
template <typename T> __device__ __forceinline__ void put(T *p, unsigned i, T v)
{
    *reinterpret_cast<T *>(reinterpret_cast<char *>(p) + i * (unsigned)sizeof(T)) = v;
}

// accessor of a cell (i, j, k all below the level's side) in the node layout: at most
// one offset is negative; below the grid it reads the own node and F, p are 0; the
// only node past the box that a cell's rows name is i + 2 (in the last cell plane)
template <typename TS, int DIM, bool M> struct CellAcc {
    typedef typename Cvt<TS>::C C;
    static constexpr bool MASK = M;
    const uint8_t *fl;
    const TS *x, *b, *al;
    long S, sI, sJ;
    unsigned q, qi, qj, qk;  // own node; the node below along each axis (own at the edge)
    bool li, lj, lk, hi;     // first cell along an axis, last along i

    __device__ __forceinline__ CellAcc(const Lvl &g, const uint8_t *f, const TS *a, const TS *bb, const TS *xx, int i,
                                       int j, int k)
        : fl(f), x(xx), b(bb), al(a), S(g.S), sI((long)g.Py * g.Pz), sJ(g.Pz)
    {
        q = ((unsigned)i * (unsigned)g.Py + (unsigned)j) * (unsigned)g.Pz + (unsigned)k;
        li = i == 0;
        lj = j == 0;
        lk = k == 0;
        hi = i == g.nx - 1;
        qi = li ? q : q - (unsigned)sI;
        qj = lj ? q : q - (unsigned)sJ;
        qk = lk ? q : q - 1u;
    }
    // lane part and uniform part of the offset of a neighbour
    __device__ __forceinline__ unsigned lane(int di, int dj, int dk) const
    { return di < 0 ? qi : (dj < 0 ? qj : (dk < 0 ? qk : q)); }
    __device__ __forceinline__ long uni(int di, int dj, int dk) const
    { return (di > 0 ? di * sI : 0) + (dj > 0 ? dj * sJ : 0) + (dk > 0 ? dk : 0); }
    __device__ __forceinline__ bool out(int di, int dj, int dk) const
    { return (di < 0 && li) || (dj < 0 && lj) || (dk < 0 && lk) || (di > 1 && hi); }

    __device__ __forceinline__ int F(int di, int dj, int dk) const
    {
        if (di > 1) {  // one plane short of i + 2 in the last cell plane, and discarded
            const int f = at(fl + sI, hi ? q : q + (unsigned)sI);
            return hi ? 0 : f;
        }
        const int f = at(fl + uni(di, dj, dk), lane(di, dj, dk));
        return out(di, dj, dk) ? 0 : f;
    }
    __device__ __forceinline__ C X(int f, int di, int dj, int dk) const
    {
        // i + 2 of u_x in the last cell plane lies in u_y's first plane: in bounds, and it
        // enters only the divergence of the cell i + 1, whose flag is 0 there
        const C v = Cvt<TS>::ld(at(x + f * S + uni(di, dj, dk), lane(di, dj, dk)));
        return ((f == 0 || !MASK) && out(di, dj, dk)) ? C(0) : v;
    }
    __device__ __forceinline__ C B(int f, int di, int dj, int dk) const
    { return Cvt<TS>::ld(at(b + f * S + uni(di, dj, dk), q)); }
    __device__ __forceinline__ C AL(int d, int di, int dj, int dk) const
    { return Cvt<TS>::ld(at(al + d * S + uni(di, dj, dk), q)); }
};

// accessor of any node of the box: offsets in -1..1 per axis, 0 outside the box
template <typename TS, int DIM, bool M, typename TX = TS> struct NodeAcc {
    typedef typename Cvt<TS>::C C;
    static constexpr bool MASK = M;
    const uint8_t *fl;
    const TX *x;
    const TS *al;
    long S;
    unsigned q, im, ip, jm, jp, km, kp;  // steps to the neighbours (0 at the edge)
    bool li, lj, lk, hi, hj, hk;

    __device__ __forceinline__ NodeAcc(const Lvl &g, const uint8_t *f, const TS *a, const TX *xx, int i, int j, int k)
        : fl(f), x(xx), al(a), S(g.S)
    {
        const unsigned sI = (unsigned)g.Py * (unsigned)g.Pz, sJ = (unsigned)g.Pz;
        q = (unsigned)i * sI + (unsigned)j * sJ + (unsigned)k;
        li = i == 0; lj = j == 0; lk = k == 0;
        hi = i == g.nx; hj = j == g.ny; hk = (DIM == 2) || k >= g.nz;
        im = li ? 0u : sI; ip = hi ? 0u : sI;
        jm = lj ? 0u : sJ; jp = hj ? 0u : sJ;
        km = lk ? 0u : 1u; kp = hk ? 0u : 1u;
    }
    __device__ __forceinline__ unsigned node(int di, int dj, int dk) const
    {
        return q + (di > 0 ? ip : 0u) + (dj > 0 ? jp : 0u) + (dk > 0 ? kp : 0u) - (di < 0 ? im : 0u) -
               (dj < 0 ? jm : 0u) - (dk < 0 ? km : 0u);
    }
    __device__ __forceinline__ bool out(int di, int dj, int dk) const
    {
        return (di < 0 && li) || (dj < 0 && lj) || (dk < 0 && lk) || (di > 0 && hi) || (dj > 0 && hj) || (dk > 0 && hk);
    }
    __device__ __forceinline__ int F(int di, int dj, int dk) const
    {
        const int f = at(fl, node(di, dj, dk));
        return out(di, dj, dk) ? 0 : f;
    }
    __device__ __forceinline__ C X(int f, int di, int dj, int dk) const
    {
        const C v = (C)Cvt<TX>::ld(at(x + f * S, node(di, dj, dk)));
        return ((f == 0 || !MASK) && out(di, dj, dk)) ? C(0) : v;
    }
    __device__ __forceinline__ C AL(int d, int di, int dj, int dk) const
    { return Cvt<TS>::ld(at(al + d * S, node(di, dj, dk))); }
};

}  // namespace st
