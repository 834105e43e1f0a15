"""Kernels that a converging solve would hide an error of, against the oracle: the marched
smoother at the sizes that run it, the V-cycle in FP32 and BF16 storage and on every kind of
level, the operator inside FGMRES, and large host arrays."""
import numpy as np
import pytest

from conftest import rel
from helpers import DeviceArray, oracle_desc, setup, solver_for
from stokes_to_amd.problems import channel_problem
from test_gpu_coarse import scattered
from test_gpu_components import open_low_sides

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n,prec,tol", [(128, "fp32", 1e-6), (128, "bf16", 1e-2), (256, "fp64", 1e-12)])
def test_marched_smoother_matches_oracle(make_solver, orc, n, prec, tol):
    """k_march<., SMOOTH>, which smooths 128^3 in FP32 and BF16 and 256^3 in all precisions (64^3
    and, in FP64, 128^3 run the cell kernel), with fixed cells and faces all over the level.
    The bars are those of the smaller levels."""
    P, rho = setup(3, n)
    P.fixed[:] = scattered(P, n)
    fixed, vol, pen = oracle_desc(orc, P, rho)
    s = solver_for(make_solver, P, rho, precision=prec, restart=2, warm_order=0)
    rng = np.random.default_rng(20)
    b, x = rng.standard_normal(fixed.size), rng.standard_normal(fixed.size)
    for color in (0, 1) if n < 256 else (1,):
        xo = orc.smooth_color(3, P.shape, fixed, pen, b, x, color, 1.0)
        assert rel(s.mg_smooth(0, color, b, x, mixed=True), xo) < tol, color


@pytest.mark.parametrize("prec,tol", [("fp32", 1e-4), ("bf16", 2e-2)])
@pytest.mark.parametrize("dim,n", [(2, 8), (2, 16), (2, 32), (2, 64), (2, 128), (3, 8), (3, 16), (3, 32)])
@pytest.mark.parametrize("nu", [(1, 2), (2, 3)])
def test_low_precision_vcycle_matches_oracle(make_solver, orc, dim, n, nu, prec, tol):
    """The fused coarsest cycle, the 2D sweeps and the one-launch restriction in FP32 and BF16.
    The oracle's cycle with every stored value rounded is off by 8e-8 / 6e-3 from its FP64
    one, and by 2e-5 with arithmetic errors of 1e-6 of the largest value in FP32."""
    P, rho = setup(dim, n, sigma=max(1.5, n / 12))
    P.fixed[:] = scattered(P, n)
    fixed, vol, pen = oracle_desc(orc, P, rho)
    s = solver_for(make_solver, P, rho, nu_pre=nu[0], nu_post=nu[1], precision=prec)
    mg = orc.MG(dim, P.shape, fixed, pen, nu_pre=nu[0], nu_post=nu[1], omega=1.0, tang=0)
    b = np.random.default_rng(7).standard_normal(fixed.size)
    assert rel(s.mg_vcycle(b), mg.vcycle(b)) < tol


def test_vcycle_through_a_padded_inner_level_matches_oracle(make_solver, orc):
    """128^3: its 64^3 level has row padding and runs the cell smoother, the one-launch
    restriction and the paired prolongation of the inner levels."""
    P, rho = setup(3, 128)
    P.fixed[:] = scattered(P, 128)
    fixed, vol, pen = oracle_desc(orc, P, rho)
    s = solver_for(make_solver, P, rho, restart=2)
    mg = orc.MG(3, P.shape, fixed, pen, nu_pre=1, nu_post=2, omega=1.0, tang=0)
    b = np.random.default_rng(7).standard_normal(fixed.size)
    assert rel(s.mg_vcycle(b), mg.vcycle(b)) < 1e-10


@pytest.mark.parametrize("prec,tol", [("fp64", 1e-9), ("fp32", 1e-4)])
def test_fgmres_steps_use_the_oracle_s_operator(make_solver, orc, prec, tol):
    """Three steps of FGMRES from zero, with free faces on the low sides: the solution is that of
    the same steps with the oracle's operator (k_fine inside the solver) and the library's
    V-cycle, to rounding."""
    P, rho = setup(3, 64)
    open_low_sides(P, 64)
    fixed, vol, pen = oracle_desc(orc, P, rho)
    b = np.where(fixed.astype(bool), 0.0, np.random.default_rng(9).standard_normal(fixed.size))
    s = solver_for(make_solver, P, rho, precision=prec, max_iter=3)
    s.update_b(body=b)
    x, _ = s.solve(allow_noconv=True)
    V, Z, H = [b / np.linalg.norm(b)], [], np.zeros((4, 3))
    for j in range(3):
        Z.append(s.mg_vcycle(V[j]))
        w = orc.apply(3, P.shape, fixed, vol, pen, Z[j])
        H[:j + 1, j] = [v @ w for v in V]
        w = w - sum(h * v for h, v in zip(H[:, j], V))
        H[j + 1, j] = np.linalg.norm(w)
        V.append(w / H[j + 1, j])
    y = np.linalg.lstsq(H, np.r_[np.linalg.norm(b), 0, 0, 0], rcond=None)[0]
    assert rel(x, sum(c * z for c, z in zip(y, Z))) < tol


def test_large_host_arrays_reach_the_device_whole(make_solver, orc):
    """128^3, where a vector goes up through the slots too (68 MB): the operator on a host array
    gives the bits of the operator on a device vector copied there by the runtime, and the
    sensitivity of two host vectors is the oracle's (1e-13)."""
    P = channel_problem(3, 128)
    rng = np.random.default_rng(1)
    rho = rng.uniform(0.1, 0.9, 128 ** 3)
    s = solver_for(make_solver, P, rho, restart=2, warm_order=0)
    x, lam = rng.standard_normal(s.ndof), rng.standard_normal(s.ndof)
    dx, dy = DeviceArray(x), DeviceArray(np.zeros(s.ndof))
    assert s.lib.st_apply_device(s.h, dx.ptr, dy.ptr) == 0
    assert np.array_equal(s.applyMapping(x), dy.get())
    nc = 128 ** 3
    ref = orc.sensitivity(3, P.shape, rho, P.alpha.array(), P.fixed[nc:], x[nc:], lam[nc:])
    assert rel(s.sensitivity(rho, x, lam), ref) < 1e-13
    dx.free()
    dy.free()
