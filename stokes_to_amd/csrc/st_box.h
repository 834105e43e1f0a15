// One cell of the box-Vanka smoother and one node of the residual, written over an
// accessor of the neighbouring nodes, for the levels that are not marched plane by
// plane (st_coarse.hip).  The rows, their order of operations and the block solve are
// those of Sten and smooth_cell in st_kernels.hip, so every kernel built on these
// gives the same bits in FP32 and BF16.
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

// masked velocities, divergences and edge curls around the accessor's node
template <typename C, int DIM, typename A> struct BoxSten {
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
        C r = gdiv(i - di, j - dj, k - dk) - gdiv(i, j, k);
        if (DIM == 3) {
            if (d == 0) r += ey(i, j, k + 1) - ey(i, j, k) + ez(i, j, k) - ez(i, j + 1, k);
            if (d == 1) r += ex(i, j, k) - ex(i, j, k + 1) + ez(i + 1, j, k) - ez(i, j, k);
            if (d == 2) r += ex(i, j + 1, k) - ex(i, j, k) + ey(i, j, k) - ey(i + 1, j, k);
        } else {
            if (d == 0) r += ez(i, j, 0) - ez(i, j + 1, 0);
            if (d == 1) r += ez(i + 1, j, 0) - ez(i, j, 0);
        }
        const C u = a.X(1 + d, i, j, k);
        r += a.X(0, i - di, j - dj, k - dk) - a.X(0, i, j, k);
        r += a.AL(d, i, j, k) * u;
        return ((a.F(i, j, k) >> (1 + d)) & 1) ? r : u;
    }
    __device__ __forceinline__ C cell() const
    {
        const C d = dv(0, 0, 0), p = a.X(0, 0, 0, 0);
        return (a.F(0, 0, 0) & 1) ? d : p;
    }
};

// new values of the cell's pressure and of its low (u0) and high (u1) faces after the
// exact solve of its block (smooth_cell of st_kernels.hip); ZERO: x is zero and not read
template <typename C, int DIM, bool ZERO, typename A>
__device__ __forceinline__ void box_cell(const A &a, float omega, C &pn, C *u0n, C *u1n)
{
    const BoxSten<C, DIM, A> s{a};
    const int fb = a.F(0, 0, 0);
    const C mc = (fb & 1) ? C(1) : C(0);
    const C NE = (DIM == 3) ? C(4) : C(2);
    C rp = a.B(0, 0, 0, 0);
    if (!ZERO) rp -= s.cell();
    C beta = C(0), tb = C(0);  // b^T E^-1 b, b^T E^-1 r_u
    C a0[3], a1[3], of[3], r0[3], r1[3], m0[3], m1[3];
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
        const C id = C(1) / (a0[d] * a1[d] - of[d] * of[d]);
        // b_f = (-m0, m1), b_c = mc * b_f
        const C kb0 = id * (a1[d] * (-m0[d]) - of[d] * m1[d]);
        const C kb1 = id * (-of[d] * (-m0[d]) + a0[d] * m1[d]);
        const C kr0 = id * (a1[d] * rl - of[d] * rh);
        const C kr1 = id * (-of[d] * rl + a0[d] * rh);
        beta += (-m0[d]) * kb0 + m1[d] * kb1;
        tb += (-m0[d]) * kr0 + m1[d] * kr1;
    }
    const C Sc = (mc != C(0)) ? -beta : C(1);
    const C dp = (Sc != C(0)) ? (rp - mc * tb) / Sc : C(0);
    const C gm = (mc != C(0)) ? dp : (dp - tb) / (C(1) - beta);
    const C om = (C)omega;
    const C p0 = ZERO ? C(0) : a.X(0, 0, 0, 0);
    pn = p0 + om * dp;
#pragma unroll
    for (int d = 0; d < DIM; d++) {
        const int di = (d == 0), dj = (d == 1), dk = (d == 2);
        const C id = C(1) / (a0[d] * a1[d] - of[d] * of[d]);
        const C e0 = r0[d] + m0[d] * gm;   // r - b_f g, b_f = (-m0, m1)
        const C e1 = r1[d] - m1[d] * gm;
        const C u0 = ZERO ? C(0) : a.X(1 + d, 0, 0, 0);
        const C u1 = ZERO ? C(0) : a.X(1 + d, di, dj, dk);
        u0n[d] = u0 + om * id * (a1[d] * e0 - of[d] * e1);
        u1n[d] = u1 + om * id * (-of[d] * e0 + a0[d] * e1);
    }
}

}  // namespace st
