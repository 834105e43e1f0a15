"""Kernels that a converging solve would hide an error of, against the oracle: the marched
smoother at the sizes that run it."""
import numpy as np
import pytest

from conftest import rel
from helpers import oracle_desc, setup, solver_for
from test_gpu_coarse import scattered

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
