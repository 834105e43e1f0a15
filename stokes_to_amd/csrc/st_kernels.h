// Launchers for the HIP kernels of st_kernels.hip (host-callable).
#pragma once
#include "st_common.h"

namespace st {

// alpha(r) = amax + (amin - amax) r(1+q)/(r+q) on r = rho^power, times scale
// (FT/FluidTopoOpt3D.cpp:110-123)
struct AlphaParams {
    double amax, amin, q, power, scale;
};

constexpr int ST_MAX_LEVELS = 12;
// the coarsest levels of a V-cycle in one launch (st_coarse.hip): flags and alpha of the
// first of them and the ones below, by value, so that their loads wait for no pointer
constexpr int ST_TAIL_LEVELS = 5;
template <typename TS> struct TailArgs {
    int nu_pre, nu_post, nd;
    float omega;
    const uint8_t *fl[ST_TAIL_LEVELS];
    const TS *al[ST_TAIL_LEVELS];
    const double *minv;
};
// inner (here and below): the level lies under the finest one, so every fixed DOF has a
// zero right-hand side and a zero x (st_box.h)
// n: side of the first level, 8 in 3D and 8, 16 or 32 in 2D; b0, x0: its right-hand side
// and solution
template <typename TS>
void launch_vcycle_tail(const TailArgs<TS> &a, int dim, int n, const TS *b0, TS *x0, bool inner, hipStream_t);
// smoother colour pass, one lane per pair of cells; fine: with the arithmetic of
// march_smooth, else with that of the levels that are not marched
template <typename TS>
void launch_box(const Lvl &, const uint8_t *, const TS *al, const TS *b, const TS *xin, TS *xout, int color,
                float omega, bool zero, bool inner, bool fine, hipStream_t);
// nsweep (1 to ST_SWEEPS) whole sweeps (first colour col0, then the other) of a 2D level in
// one launch, xin -> xout; zero: from x = 0; ec: from xin + P ec
constexpr int ST_SWEEPS = 2;
template <typename TS>
void launch_sweeps(const Lvl &, const Lvl &gc, const uint8_t *, const TS *al, const TS *b, const TS *xin, const TS *ec,
                   TS *xout, int nsweep, int col0, float omega, bool zero, bool inner, hipStream_t);
// y = A x and r = b - A x (partials of |r|^2 per 256 nodes) of such a level
template <typename TS>
void launch_node_apply(const Lvl &, const uint8_t *, const TS *al, const TS *x, TS *y, hipStream_t);
template <typename TS>
void launch_node_residual(const Lvl &, const uint8_t *, const TS *al, const TS *b, const TS *x, TS *r, double *part,
                          hipStream_t);
// bc = R (b - A x): residual and restriction of such a level in one launch
template <typename TS>
void launch_resid_restrict(const Lvl &gf, const Lvl &gc, const uint8_t *flf, const TS *al, const TS *b, const TS *x,
                           const uint8_t *flc, TS *bc, bool inner, hipStream_t);

template <typename TS> void launch_apply(const Lvl &, const uint8_t *, const TS *, const TS *, TS *, hipStream_t);
template <typename TS>
void launch_residual(const Lvl &, const uint8_t *, const TS *, const TS *b, const TS *x, TS *r, double *part,
                     hipStream_t);
unsigned residual_blocks(const Lvl &);
// the FP64 residual and norm of the plain FP64 solve (plain_residual_blocks partials)
void launch_plain_residual(const Lvl &, const uint8_t *, const double *, const double *b, const double *x, double *r,
                           double *part, hipStream_t);
unsigned plain_residual_blocks(const Lvl &);
template <typename TS>
void launch_smooth(const Lvl &, const uint8_t *, const TS *, const TS *b, const TS *xin, TS *xout, int color,
                   float omega, bool zero, bool inner, hipStream_t);
template <typename TS>
void launch_restrict(const Lvl &gf, const Lvl &gc, const uint8_t *flc, const TS *rf, TS *bc, hipStream_t);
template <typename TS>
void launch_prolong(const Lvl &gf, const Lvl &gc, const uint8_t *flf, const TS *ec, TS *xf, hipStream_t);
template <typename TF, typename TC>
void launch_coarsen(const Lvl &gf, const Lvl &gc, const uint8_t *flf, const TF *alf, uint8_t *flc, TC *alc,
                    hipStream_t);
template <typename TS>
void launch_probe(const Lvl &, const uint8_t *, const TS *, const long *dofs, int nd, int closed, double *A,
                  hipStream_t);
void launch_gauss_jordan(int n, double *A, int *info, hipStream_t);  // n <= 64
template <typename TS>
void launch_pack(const Lvl &, const double *abi, TS *pad, int fixed_only, const uint8_t *fl, double scale,
                 hipStream_t);
template <typename TS> void launch_unpack(const Lvl &, const TS *pad, double *abi, hipStream_t);
void launch_flags(const Lvl &, const uint8_t *abi_fixed, uint8_t *fl, hipStream_t);
template <typename TS> void launch_alpha_from_pen(const Lvl &, const double *pen, const uint8_t *fl, TS *al, hipStream_t);
void launch_design_alpha(const Lvl &, const double *rho, const AlphaParams &, const uint8_t *fl, double *al,
                         hipStream_t);
void launch_sensitivity(const Lvl &, const double *rho, const AlphaParams &, const uint8_t *fl, const double *u,
                        const double *lam, double *dj, hipStream_t);
void launch_lift(const Lvl &, const uint8_t *fl, const double *xd, const double *body, double *b, hipStream_t);
void launch_energy(const Lvl &, const uint8_t *fl, const double *al, const double *x, double *y, double *part,
                   hipStream_t);
unsigned energy_blocks(const Lvl &);
// Wi: reciprocal weight sums of the cells, written by launch_filter_w
void launch_filter(const Lvl &, double R, const double *Wi, const double *in, double *out, int transpose, hipStream_t);
void launch_filter_w(const Lvl &, double R, double *Wi, hipStream_t);
constexpr int OC_K = 16;  // multipliers per pass of the OC search
struct OcFactors {
    double f[OC_K];
};
unsigned oc_grid(long n);
void launch_oc_base(long n, const double *dc, const double *dv, double eta, double *base, hipStream_t);
void launch_oc_vols(long n, const double *rho, const double *base, const double *dv, const OcFactors &f, double move,
                    double rho_min, double *part, hipStream_t);
void launch_oc_apply(long n, const double *rho, const double *base, const double *dv, double fl, double move,
                     double rho_min, double *rn, double *part, hipStream_t);
unsigned absmax_blocks(long n);
void launch_absdiff_max(long n, const double *a, const double *b, double *part, hipStream_t);
void launch_sum(int np, int nvec, const double *part, double *out, hipStream_t s, double *hout = nullptr,
                const double *hsrc = nullptr, double *hdst = nullptr);
unsigned blas_blocks(long n);
template <typename TA, typename TB> void launch_dot(long n, const TA *a, const TB *b, double *part, hipStream_t);
template <typename TW, typename TV>
unsigned launch_multidot(long n, const TW *w, const TV *V, long ld, int m, double *part, hipStream_t);
template <typename TW, typename TV>
unsigned launch_multiaxpy(long n, TW *w, const TV *V, long ld, int m, const double *h, const double *sc, double *part,
                      hipStream_t);
template <typename TX, typename TY> void launch_axpby(long n, double a, const TX *x, double b, TY *y, hipStream_t);
void launch_lincomb3(long n, double a, const double *x, double b, const double *w, double c, double *y, hipStream_t);
// minimal-residual start: d = float(a - b); Gram of nd <= 3 FP32 vectors y_i (stride ld)
// and their products with r (partials: nd(nd+1)/2 + nd per block, mr_blocks(n) blocks);
// x0 = x1 + sum d_i D_i, r -= sum d_i y_i with the partials of the new ||r||^2
struct MrCoef {
    double d[3];
};
void launch_diff_f32(long n, const double *a, const double *b, float *d, hipStream_t);
unsigned mr_blocks(long n);
void launch_mr_gram(int nd, long n, const float *y, long ld, const float *r, double *part, hipStream_t);
void launch_mr_update(int nd, long n, const double *x1, const float *const *D, const float *y, long ld,
                      const MrCoef &cf, double *x0, float *r, double *part, hipStream_t);
template <typename TS> void launch_fill(long n, TS *y, double v, hipStream_t);

// 2.5D marching kernels (st_march.hip) for 3D levels with ny % 4 == 0, nz % 64 == 0
bool march_ok(const Lvl &);
unsigned march_blocks(const Lvl &);
void march_residual(const Lvl &, const uint8_t *, const double *, const double *b, const double *x, double *r,
                    double *part, hipStream_t);
template <typename TS>
void march_smooth(const Lvl &, const uint8_t *, const TS *, const TS *b, const TS *xin, TS *xout, int color,
                  float omega, hipStream_t);
// FP64 residual r = b - A x stored in FP32 (+ FP64 partial sums of |r|^2)
void march_residual_f32(const Lvl &, const uint8_t *, const double *al, const double *b, const double *x, float *r,
                        double *part, hipStream_t);
// operator and residual of the same levels without LDS (st_fine.hip)
template <typename TS> void fine_apply(const Lvl &, const uint8_t *, const TS *, const TS *, TS *, hipStream_t);
template <typename TS>
void fine_residual(const Lvl &, const uint8_t *, const TS *, const TS *b, const TS *x, TS *r, double *part, hipStream_t);
// FP64 operator on vectors in the caller's layout
void user_apply(const Lvl &, const uint8_t *, const double *al, const double *x, double *y, hipStream_t);
// FP64 operator applied to an FP32-stored vector (x float, alpha and y double)
void fine_apply_mixed(const Lvl &, const uint8_t *, const double *al, const float *x, double *y, hipStream_t);
unsigned fine_blocks(const Lvl &);
// one red-black sweep (colour col0, then the other) in one pass (st_sweep.hip);
// FP32 arithmetic, TS = float or bf16 storage, levels with march_ok
template <typename TS>
void march_sweep(const Lvl &, const uint8_t *, const TS *al, const TS *b, const TS *xin, TS *xout, int col0,
                 float omega, hipStream_t);

}  // namespace st
