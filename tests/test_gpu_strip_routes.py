"""Which solves run over row strips and which over tiles, by the report's
strips_per_wave, on both sides of every line of the rule; and the tile kernels
with resident windows at the policies that strips otherwise take.

One block is 16 waves of up to 8 strips: 8,192 rows.  Resident windows hold 40
tile-rows a wave, so up to 10,240 rows of one block run on them."""
import numpy as np
import pytest

from test_gpu_strip_solvers import TOL, _band

pytestmark = pytest.mark.gpu


def _solve(mf, oracle, tm, m, method, **kw):
    n = len(m[0]) - 1
    b = np.random.default_rng(n).uniform(-1, 1, n)
    db, dx = tm.vector(b), tm.vector()
    rep = getattr(tm, method)(db, dx, tol=TOL, **kw)
    assert rep["status"] == 0 and oracle.rel_residual(*m, b, dx.get()[:n]) <= TOL, rep
    return rep


def _learned(mf, tm):
    from millefeuille import policy
    policy.install(tm, policy.load())


@pytest.mark.parametrize("n,strips", [(64, 1), (1024, 1), (1025, 2), (2049, 3), (4096, 4), (4097, 5), (8192, 8)])
@pytest.mark.parametrize("method", ["cg", "bicgstab"])
@pytest.mark.parametrize("policy", ["fp64", "errbound", "learned"])
def test_strips_run(mf, oracle, n, strips, method, policy):
    m = _band(n, "diag", sym=method == "cg")
    tm = mf.TiledMatrix(*m)
    _learned(mf, tm)
    rep = _solve(mf, oracle, tm, m, method, policy=policy, blocks=1)
    assert rep["strips_per_wave"] == strips and rep["form_used"] == 2 and rep["fell_back"] == 0, rep


@pytest.mark.parametrize("n", [8193, 10000])
@pytest.mark.parametrize("method", ["cg", "bicgstab"])
@pytest.mark.parametrize("policy", ["fp64", "errbound", "learned"])
def test_more_strips_than_waves_hold_run_on_resident_tiles(mf, oracle, n, method, policy):
    m = _band(n, "near", sym=method == "cg")
    tm = mf.TiledMatrix(*m)
    _learned(mf, tm)
    rep = _solve(mf, oracle, tm, m, method, policy=policy, blocks=1)
    assert rep["strips_per_wave"] == 0 and rep["form_used"] == 2, rep


@pytest.mark.parametrize("method", ["cg", "bicgstab"])
@pytest.mark.parametrize("policy", ["fp64", "errbound", "learned"])
def test_memory_form_runs_on_streamed_tiles(mf, oracle, method, policy):
    m = _band(3000, "near", sym=method == "cg")
    tm = mf.TiledMatrix(*m)
    _learned(mf, tm)
    rep = _solve(mf, oracle, tm, m, method, policy=policy, form="memory")
    assert rep["strips_per_wave"] == 0 and rep["form_used"] == 1, rep


@pytest.mark.parametrize("method", ["cg", "bicgstab"])
def test_sorted_rows(mf, oracle, method):
    """Strips at FP64 and the error bound; learned levels need the row order, so
    only their fallback runs over strips."""
    from millefeuille import gen
    m = gen.knn_laplacian(5000, 8, seed=4)
    tm = mf.TiledMatrix(*m)
    _learned(mf, tm)
    assert tm.strips()["sorted"] == 1
    for policy, strips in (("fp64", True), ("errbound", True), ("learned", False)):
        rep = _solve(mf, oracle, tm, m, method, policy=policy)
        assert (rep["strips_per_wave"] > 0) == (strips or rep["fell_back"] == 1), (policy, rep)


@pytest.mark.parametrize("method", ["cg", "bicgstab"])
@pytest.mark.parametrize("policy", ["fixed", "rule"])
def test_per_tile_levels_run_on_tiles_and_fall_back_to_strips(mf, oracle, method, policy):
    m = _band(5000, "near", sym=method == "cg")
    tm = mf.TiledMatrix(*m)
    # FP64 levels: no fallback (the rule starts there); one refresh allowed: a fallback
    rep = _solve(mf, oracle, tm, m, method, policy="fixed")
    assert rep["strips_per_wave"] == 0 and rep["fell_back"] == 0, rep
    tm.set_precision(uniform=mf.PREC_FP32)
    rep = _solve(mf, oracle, tm, m, method, policy=policy, max_refresh=1, refresh_every=2)
    assert rep["fell_back"] == 1 and rep["strips_per_wave"] > 0, rep
    rep = _solve(mf, oracle, tm, m, method, policy=policy, max_refresh=1, refresh_every=2, form="memory")
    assert rep["fell_back"] == 1 and rep["strips_per_wave"] == 0, rep
