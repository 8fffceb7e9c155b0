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


def _rows(n, lens, cols, values, seed=0):
    """Symmetric matrix: row i gets lens[i] couplings at cols(rng, i-array);
    diagonally dominant."""
    rng = np.random.default_rng(seed)
    r = np.repeat(np.arange(n), lens)
    c = cols(rng, r)
    k = np.unique(np.concatenate([r * np.int64(n) + c, c * np.int64(n) + r]))
    r, c = k // n, k % n
    up = c > r
    v = -np.ones(up.sum()) if values == "ones" else -rng.uniform(0.1, 1, up.sum())
    r, c, v = np.concatenate([r[up], c[up]]), np.concatenate([c[up], r[up]]), np.concatenate([v, v])
    d = np.bincount(r, -v, minlength=n) + 1.0
    r, c, v = np.concatenate([r, np.arange(n)]), np.concatenate([c, np.arange(n)]), np.concatenate([v, d])
    k = np.lexsort((c, r))
    return np.concatenate([[0], np.cumsum(np.bincount(r, minlength=n))]).astype(np.int32), c[k].astype(np.int32), v[k]


def _matrix(name):
    from millefeuille import gen
    rng = np.random.default_rng(1)

    def band(w):
        return lambda g, r: np.clip(r + g.integers(-w, w + 1, len(r)), 0, r.max())

    return {
        "lap2d": lambda: gen.laplace2d(64),
        "lap3d": lambda: gen.laplace3d_scaled(32, seed=2),
        "convdiff": lambda: gen.convdiff3d(24),
        "knn": lambda: gen.knn_laplacian(20000, 8, seed=4),
        "powerlaw": lambda: gen.powerlaw_laplacian(20000, 300000, seed=5),
        "scattered": lambda: _rows(20000, rng.integers(5, 16, 20000), lambda g, r: g.integers(0, 20000, len(r)), "random"),
        # rows of 20 to 70 entries around the diagonal, the longest in pieces
        "wide band, pieces": lambda: _rows(40000, rng.integers(10, 50, 40000), band(160), "ones"),
        # 125 strips whose lanes walk 120 entries each
        "few long rows": lambda: _rows(8000, np.full(8000, 60), band(240), "ones"),
        # as many bytes as the tiles, in another order
        "random band": lambda: _rows(160000, rng.integers(5, 18, 160000), band(60), "random"),
    }[name]()


# kernel of the FP64 product
@pytest.mark.parametrize("name,strips", [("lap2d", True), ("lap3d", True), ("convdiff", True), ("knn", True),
                                         ("powerlaw", True), ("scattered", True), ("wide band, pieces", False),
                                         ("few long rows", False), ("random band", False)])
def test_default_product(mf, oracle, name, strips):
    m = _matrix(name)
    n = len(m[0]) - 1
    tm = mf.TiledMatrix(*m)
    assert tm.strips()["strips"] > 0
    assert tm.spmv_kernel() == (mf._lib.SPMV_STRIP if strips else mf._lib.SPMV_STREAM), tm.strips()
    assert tm.spmv_kernel(1) == mf._lib.SPMV_STREAM
    x = np.random.default_rng(0).uniform(-1, 1, n)
    dx, dy = tm.vector(x), tm.vector()
    bound = oracle.csr_spmv(m[0], m[1], np.abs(m[2]), np.abs(x))
    for kernel in ("auto", "strip", "stream"):
        tm.set_spmv_kernel(kernel)
        tm.spmv(dx, dy)
        # (sums of up to 4,000 terms in any order: 2^-53 a term)
        err = np.abs(dy.get()[:n] - oracle.csr_spmv(*m, x))
        assert np.all(err <= np.maximum(1e-14, 2.3e-16 * np.diff(m[0])) * bound), kernel


# strips at (FP64, error bound); the last two: rows of 40 to 100 entries in full
# tiles, half of them in pieces, at as many blocks over strips as over tiles
@pytest.mark.parametrize("name,blocks,fp64,errbound", [
    ("lap2d", 0, True, True), ("lap3d", 0, True, True), ("knn", 0, True, True), ("powerlaw", 0, True, True),
    ("scattered", 0, True, True), ("few long rows", 0, True, True), ("random band", 0, True, False),
    ("cut rows", 8, False, False), ("cut rows", 16, False, False)])
def test_solver_of_a_matrix(mf, oracle, name, blocks, fp64, errbound):
    if name == "cut rows":
        rng = np.random.default_rng(2)
        m = _rows(16000, rng.integers(20, 60, 16000), lambda g, r: (r // 128 * 128 + g.integers(0, 128, len(r))), "ones")
    else:
        m = _matrix(name)
    tm = mf.TiledMatrix(*m)
    for policy, strips in (("fp64", fp64), ("errbound", errbound)):
        for method in ("cg", "bicgstab"):
            rep = _solve(mf, oracle, tm, m, method, policy=policy, blocks=blocks)
            assert (rep["strips_per_wave"] > 0) == strips, (method, policy, rep, tm.strips())


def test_wide_rows_get_more_blocks(mf, oracle):
    """8,000 rows: one for each 1024 rows, and where they are wide as many as their products need."""
    m = _band(8000, "near")
    assert _solve(mf, oracle, mf.TiledMatrix(*m), m, "cg", policy="fp64")["grid_blocks"] == 8
    m = _matrix("few long rows")
    rep = _solve(mf, oracle, mf.TiledMatrix(*m), m, "cg", policy="fp64")
    assert rep["grid_blocks"] >= 24 and rep["strips_per_wave"] == 1, rep


@pytest.mark.parametrize("name,policy,strips", [("knn", "fp64", True), ("knn", "errbound", True), ("knn", "fixed", False),
                                                ("powerlaw", "fp64", True), ("scattered", "errbound", True),
                                                ("few long rows", "fp64", True), ("wide band, pieces", "errbound", True),
                                                ("cut rows", "fp64", False), ("cut rows", "errbound", True)])
def test_batch_of_a_matrix(mf, oracle, name, policy, strips):
    """Strips unless the pieces of cut rows cost more (16,000 rows fit on chip at the
    mixed policies); every wave count on both."""
    rng = np.random.default_rng(2)
    m = (_rows(16000, rng.integers(20, 60, 16000), lambda g, r: (r // 128 * 128 + g.integers(0, 128, len(r))), "ones")
         if name == "cut rows" else _matrix(name))
    n = len(m[0]) - 1
    tms = [mf.TiledMatrix(*m) for _ in range(2)]
    bs = [np.random.default_rng(k).uniform(-1, 1, n) for k in range(2)]
    for waves in (0, 4, 16):
        xs, rep = mf.batch_cg(tms, bs, tol=TOL, policy=policy, batch_waves=waves)
        assert rep["batch_waves"] == (waves or (16 if strips else 8)), rep
        for k in range(2):
            assert oracle.rel_residual(*m, bs[k], xs[k][0]) <= TOL


def test_learned_levels_over_tiles_move_fewer_bytes_than_the_rule(mf, oracle):
    """Over tiles the levels are what the product reads (9, 5, 3 and 2 bytes an
    entry with its column): the learned policy moves at most 60% of the FP64
    payload per product, and less in all than the rule."""
    from millefeuille import gen
    m = gen.laplace3d_scaled(32, seed=2)
    tm = mf.TiledMatrix(*m)
    _learned(mf, tm)
    full = 9.0 * tm.csrsize
    total = {}
    for policy in ("rule", "learned"):
        rep = _solve(mf, oracle, tm, m, "cg", policy=policy, form="memory")
        assert rep["strips_per_wave"] == 0, rep
        payload = float(np.dot(rep["prec_hist"], [9, 5, 3, 2, 0])) * tm.csrsize / tm.tilenum
        total[policy] = payload + full * rep["refreshes"]
        if policy == "learned":
            assert rep["fell_back"] == 0 and payload <= 0.6 * full * rep["iterations"], rep
    assert total["learned"] < total["rule"], total
