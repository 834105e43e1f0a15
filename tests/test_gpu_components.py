"""Calls of the component entries (st_mg_*) and what they leave behind, and the coarsest
inverse at the ends of its range, against the oracle."""
import ctypes

import numpy as np
import pytest

from conftest import rel
from helpers import oracle_desc, setup, solver_for
from stokes_to_amd.problems import _split, dof_sizes

pytestmark = pytest.mark.gpu


def open_low_sides(P, seed):
    """P with 2% more fixed cells and interior faces and with free faces on the low side of
    every axis, where a face's row reads a pressure outside the level."""
    rng = np.random.default_rng(seed)
    P.fixed[rng.integers(0, P.fixed.size, P.fixed.size // 50)] = 1
    n, m = P.n, slice(P.n // 4, 3 * P.n // 4)
    fx, fy, fz = _split(3, n, P.fixed)[1:]
    fx[0, m, :] = 0
    fy[:, 0, m] = 0
    fz[m, :, 0] = 0


@pytest.mark.parametrize("call", ["none", "smooth", "prolong", "restrict", "desc"])
def test_vcycle_after_a_call_on_a_coarse_level(make_solver, orc, call):
    """A component call on a coarser level must not change a later V-cycle on the finest
    one (64^3, whose operator reads pressures outside the level from entries that hold 0):
    1e-10 of the oracle, as without it."""
    n = 64
    P, rho = setup(3, n)
    open_low_sides(P, n)
    fixed, vol, pen = oracle_desc(orc, P, rho)
    s = solver_for(make_solver, P, rho)
    rng = np.random.default_rng(7)
    v = [rng.standard_normal(orc.sizes(3, n >> l, n >> l, n >> l)[0]) for l in range(3)]
    if call == "smooth":
        s.mg_smooth(1, 0, v[1], v[1])
    if call == "prolong":
        s.mg_prolong(1, v[2], v[1])
    if call == "restrict":
        s.mg_restrict(0, v[0])
    if call == "desc":
        s.mg_level_desc(1)
    mg = orc.MG(3, P.shape, fixed, pen, nu_pre=1, nu_post=2, omega=1.0, tang=0)
    assert rel(s.mg_vcycle(v[0]), mg.vcycle(v[0])) < 1e-10


@pytest.mark.parametrize("dim,share,seed", [(2, 0.3, 21), (3, 0.5, 21), (3, 0.5, 112)])
def test_coarsest_inverse_pivots_in_full_precision(make_solver, orc, dim, share, seed):
    """Penalties of 1e38 to 1e60, beyond the largest FP32 value: the pivot of the coarsest
    inverse has to be the largest FP64 magnitude (a V-cycle without sweeps is that inverse
    between transfers).  1e-10 of the oracle: eliminated with the largest pivot, these
    matrices keep 1e-15 under any rounding; with a smaller one they can lose all digits."""
    n = 8
    rng = np.random.default_rng(seed)
    nd = orc.sizes(dim, n, n, n if dim == 3 else 1)[0]
    fixed, pen = np.zeros(nd, np.uint8), np.zeros(nd)
    ff, pp = _split(dim, n, fixed), _split(dim, n, pen)
    for d in range(dim):  # one value for the fine faces under each face of the 2^dim grid
        c = 10.0 ** rng.uniform(38, 60, [3 if a == d else 2 for a in range(dim)])
        off = rng.random(c.shape) < share
        at = np.ix_(*[(np.arange(n + 1) + 1) // 4 if a == d else np.arange(n) // 4 for a in range(dim)])
        pp[1 + d][...] = (c * ~off)[at].reshape(pp[1 + d].shape)
        ff[1 + d][...] = off[at].reshape(pp[1 + d].shape)
    ff[0][...] = (rng.random([2] * dim) < 0.3)[np.ix_(*[np.arange(n) // 4] * dim)].reshape(ff[0].shape)
    s = make_solver(dim, n, nu_pre=0, nu_post=0)
    s.init_boundary(fixed)
    s.update_penalty(pen)
    mg = orc.MG(dim, (n, n, n if dim == 3 else 1), fixed, pen, nu_pre=0, nu_post=0, omega=1.0, tang=0)
    b = rng.standard_normal(nd)
    assert rel(s.mg_vcycle(b), mg.vcycle(b)) < 1e-10


@pytest.mark.parametrize("dim,n,prec", [(2, 64, "fp64"), (2, 128, "bf16"), (3, 16, "fp32"), (3, 32, "fp64")])
def test_profiled_bytes_are_those_of_the_launches(make_solver, dim, n, prec):
    """A V(1,2)-cycle's finest-level launches where they do more than one step: in 2D a launch
    from x = 0 and one of two sweeps after the prolongation, and the residual that writes the
    coarse right-hand side only."""
    P, rho = setup(dim, n)
    s = solver_for(make_solver, P, rho, precision=prec)
    s.lib.st_profile(s.h, 1)
    st = s.solve()[1]

    def read(kind):
        ms, cnt, by = ctypes.c_double(), ctypes.c_long(), ctypes.c_double()
        assert s.lib.st_profile_read(s.h, kind, ctypes.byref(ms), ctypes.byref(cnt), ctypes.byref(by)) == 0
        return cnt.value, by.value

    sv, nv, nf = {"fp64": 8, "fp32": 4, "bf16": 2}[prec], s.ndof, s.ndof - s.ncell
    coarse = dof_sizes(dim, n // 2)[-1]
    assert read(2) == (st["iters"], sv * (2 * nv + nf + coarse) + nf / 8)
    if dim == 2:
        zero, prol = sv * (2 * nv + nf) + nf / 8, sv * (3 * nv + nf + coarse) + nf / 8
        assert read(4) == (2 * st["iters"], (zero + prol) / 2)
        assert read(0)[0] == read(3)[0] == 0


@pytest.mark.parametrize("dim,n", [(2, 64), (2, 128), (3, 16)])
@pytest.mark.parametrize("nu,same", [((1, -3), (1, 0)), ((-3, 2), (0, 2)), ((-4, 1), (0, 1))])
def test_negative_sweep_counts_mean_no_sweeps(make_solver, orc, dim, n, nu, same):
    """st_create takes them; 1e-10 of the oracle's V-cycle without these sweeps."""
    P, rho = setup(dim, n, sigma=4.0)
    fixed, vol, pen = oracle_desc(orc, P, rho)
    s = solver_for(make_solver, P, rho, nu_pre=nu[0], nu_post=nu[1])
    mg = orc.MG(dim, P.shape, fixed, pen, nu_pre=same[0], nu_post=same[1], omega=1.0, tang=0)
    b = np.random.default_rng(7).standard_normal(fixed.size)
    assert rel(s.mg_vcycle(b), mg.vcycle(b)) < 1e-10
