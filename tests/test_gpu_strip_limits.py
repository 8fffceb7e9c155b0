"""Iteration limits of mixed solves that fall back to FP64 over row strips.

A fixed number of iterations far past convergence: the FP32 vectors reach
zero, the denominators vanish, and the solve falls back in whichever iteration
that is, the last one among them.  It must still end after the iterations asked
for (BiCGSTAB: one more when the last one failed and is made again), with x at
least as good as the FP32 payload gives it: the matrix's off-diagonal row sums
are under half of its diagonal, so x is within a few 2^-24 of the solution
before the vectors vanish; 1e-5 covers it."""
import numpy as np
import pytest

from test_gpu_strip_solvers import _band

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("method", ["cg", "bicgstab"])
@pytest.mark.parametrize("policy", ["errbound", "fixed"])
def test_fixed_iterations_that_fall_back(mf, oracle, method, policy):
    n = 3000
    m = _band(n, "near", sym=method == "cg")
    tm = mf.TiledMatrix(*m)
    tm.set_precision(uniform=mf.PREC_FP32)
    b = np.random.default_rng(1).uniform(-1, 1, n)
    db, fell = tm.vector(b), 0
    for k in range(20, 140, 1 if method == "bicgstab" else 3):
        dx = tm.vector()
        rep = getattr(tm, method)(db, dx, policy=policy, tol=1e-30, fixed_iters=k, allow_not_converged=True)
        fell += rep["fell_back"]
        assert rep["status"] == 0 and k <= rep["iterations"] <= k + (method == "bicgstab"), (k, rep)
        assert oracle.rel_residual(*m, b, dx.get()[:n]) <= 1e-5, (k, rep)
        if fell > 12:
            break
    assert fell > 0
