"""The matrix-free product at every register shape (columns of the O rows per
thread: 2, 4, 7 and 13), with fewer samples than a round of rows, one past it
and many, FP64 and FP32 rows: the conjugate-gradient step against the
factorization of the same S + shift within cond x 1e-12 (cond < 1e4 at the
shift of 0.1: 1e-8; FP32 rows, S built from the same rows in FP64, alike)."""
import numpy as np
import pytest

from _helpers import ising, params, random_keys
from nqhip import Context, _lib

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("net", [_lib.PREC_FP64, _lib.PREC_FP32])
@pytest.mark.parametrize("N,nh,na,chains,Lc", [(2, 1, 1, 2, 2), (6, 6, 6, 3, 3), (8, 16, 16, 37, 4), (10, 32, 32, 150, 7),
                                               (12, 64, 64, 11, 3)])
def test_cg_step_matches_the_factorization(gpu_ok, net, N, nh, na, chains, Lc):
    flat, _, _ = ising(N)
    keys = random_keys(N, chains * Lc, seed=N)
    steps = []
    for solver in (_lib.SOLVER_CHOLESKY, _lib.SOLVER_CG):
        ctx = Context(0, 1)
        ctx.set_problem(flat)
        ctx.set_ndm(N, nh, na)
        ctx.set_params(params(ctx.np_, seed=3, sigma=0.1))
        ctx.set_precision(net, _lib.PREC_FP64)
        ctx.set_sr_solver(solver, 1e-13, 0)
        ctx.grad_from_samples(keys, chains, Lc, want_S=False)
        steps.append(ctx.precondition(0.1))
        ctx.close()
    assert np.linalg.norm(steps[1] - steps[0]) < 1e-8 * np.linalg.norm(steps[0])
