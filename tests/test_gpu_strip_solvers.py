"""CG and BiCGSTAB over row strips against the oracle and against the memory
form (streamed tiles, every vector in memory): the strip classes, one to
eight strips a wave and one too many, sorted rows with pieces, the mixed
policies and the forced fallback to FP64; and the batched CG on both sides
of the sizes that its on-chip vectors hold.

Tolerances.  Converged solves: the oracle's residual within the solve's own
tolerance.  Eight FP64 iterations from zero with the same arithmetic in
another order: sums of under 1e5 terms differ by 1e5 * 2^-53 ~ 1e-11 relative
at worst (1e-14 typically), and eight steps on a matrix of condition
number under 1e2 multiply that by less than 1e2; 1e-9 covers it."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

TOL = 1e-10


def _band(n, kind, sym=True, seed=0):
    """Diagonally dominant matrix with entries at +-1, +-7 (and, kind "full",
    half the rows away): one value per diagonal, powers of two differing by
    row, or random."""
    rng = np.random.default_rng(seed)
    r, c, v = [], [], []
    for o in (1, 7) + ((n // 2,) if kind == "full" and n > 20 else ()):
        if o >= n:
            continue
        i = np.arange(n - o)
        w = {"diag": np.full(n - o, -0.7), "packed": -(2.0 ** -rng.integers(0, 4, n - o))}.get(
            kind, -rng.uniform(0.1, 1, n - o))
        r += [i, i + o]
        c += [i + o, i]
        v += [w, w if sym else 0.5 * w]
    r = np.concatenate(r + [np.arange(n)])
    c = np.concatenate(c + [np.arange(n)])
    d = rng.uniform(7, 9, n) if kind != "diag" else np.full(n, 6.0)
    v = np.concatenate(v + [d])
    k = np.lexsort((c, r))
    rp = np.zeros(n + 1, np.int32)
    np.add.at(rp, r + 1, 1)
    return np.cumsum(rp).astype(np.int32), c[k].astype(np.int32), v[k]


def _run(mf, m, method, seed=1, **kw):
    rp, ci, va = m
    n = len(rp) - 1
    tm = mf.TiledMatrix(rp, ci, va)
    b = np.random.default_rng(seed).uniform(-1, 1, n)
    db, dx = tm.vector(b), tm.vector()
    rep = getattr(tm, method)(db, dx, **kw)
    return tm, b, rep, dx.get()[:n]


def _check(mf, oracle, m, method, strips=True, **kw):
    tm, b, rep, x = _run(mf, m, method, tol=TOL, **kw)
    assert rep["status"] == 0 and oracle.rel_residual(*m, b, x) <= TOL, rep
    if strips:
        assert rep["form_used"] == 2, rep
    return tm, rep, x


# one block: 16 waves, 1024 rows for each strip of a wave
@pytest.mark.parametrize("n", [1, 63, 65, 1024, 1025, 2049, 4095, 4097, 8192])
@pytest.mark.parametrize("method", ["cg", "bicgstab"])
@pytest.mark.parametrize("policy", ["fp64", "errbound"])
def test_strips_per_wave(mf, oracle, n, method, policy):
    m = _band(n, "diag" if n % 2 else "near", sym=method == "cg", seed=n)
    _check(mf, oracle, m, method, policy=policy, blocks=1)


@pytest.mark.parametrize("method", ["cg", "bicgstab"])
def test_more_strips_than_the_waves_hold(mf, oracle, method):
    """A ninth strip a wave: streamed tiles."""
    _check(mf, oracle, _band(8193, "near", sym=method == "cg"), method, strips=False, blocks=1)


@pytest.mark.parametrize("kind,n", [("diag", 3001), ("packed", 3001), ("near", 3001), ("full", 70001)])
@pytest.mark.parametrize("method", ["cg", "bicgstab"])
@pytest.mark.parametrize("policy", ["fp64", "errbound"])
def test_classes(mf, oracle, kind, n, method, policy):
    m = _band(n, kind, sym=method == "cg")
    tm, _, x = _check(mf, oracle, m, method, policy=policy)
    s = tm.strips()
    slots = {"diag": "diag_slots", "packed": "packed_slots"}.get(kind, "full_slots")
    assert s[slots] > 0.9 * (s["diag_slots"] + s["packed_slots"] + s["full_slots"]), s
    if policy == "fp64":
        # the same steps as the memory form
        y = [_run(mf, m, method, fixed_iters=8, form=f)[3] for f in ("auto", "memory")]
        assert np.max(np.abs(y[0] - y[1])) <= 1e-9 * np.max(np.abs(y[1]))


@pytest.mark.parametrize("method", ["cg", "bicgstab"])
@pytest.mark.parametrize("blocks", [0, 4, 7, 16, 40])
@pytest.mark.parametrize("policy", ["fp64", "errbound"])
def test_sorted_rows_and_pieces(mf, oracle, method, blocks, policy):
    """Rows of several pieces whose owner waits for other waves' sums."""
    from millefeuille import gen
    m = gen.powerlaw_laplacian(20000, 300000, seed=5)
    tm, rep, _ = _check(mf, oracle, m, method, policy=policy, blocks=blocks)
    s = tm.strips()
    assert s["sorted"] == 1 and s["pieces"] > 0
    again = _run(mf, m, method, tol=TOL, policy=policy, blocks=blocks)
    assert again[2]["iterations"] == rep["iterations"]


@pytest.mark.parametrize("policy", ["errbound", "rule"])
@pytest.mark.parametrize("method", ["cg", "bicgstab"])
@pytest.mark.parametrize("kind", ["diag", "near"])
def test_fallback_goes_on_over_strips(mf, oracle, policy, method, kind):
    """max_refresh 1: the first recomputed residual but one ends the mixed
    solve (strips for the error bound, tiles for the rule), and FP64 strips
    go on from its x (BiCGSTAB under the rule stays on tiles)."""
    m = _band(5000, kind, sym=method == "cg")
    _, rep, _ = _check(mf, oracle, m, method, strips=(method, policy) != ("bicgstab", "rule"), policy=policy,
                       max_refresh=1, refresh_every=2)
    assert rep["fell_back"] == 1 and rep["refreshes"] >= 2, rep


@pytest.mark.parametrize("method", ["cg", "bicgstab"])
def test_guess_maxiter_and_noalloc(mf, oracle, method):
    m = _band(2500, "near", sym=method == "cg")
    tm, rep, x = _check(mf, oracle, m, method)
    b = np.random.default_rng(1).uniform(-1, 1, len(x))
    db, dx = tm.vector(b), tm.vector(x)
    assert getattr(tm, method)(db, dx, tol=10 * TOL)["iterations"] == 0
    rep = _run(mf, m, method, tol=1e-14, maxiter=2, allow_not_converged=True)[2]
    assert rep["iterations"] == 2 and rep["status"] == 1
    if method == "cg":
        d2 = tm.vector()
        r2 = tm.cg_noalloc(db, d2, tol=TOL)
        assert r2["status"] == 0 and oracle.rel_residual(*m, b, d2.get()[: len(b)]) <= TOL


# vectors on chip up to 64 * 8 * waves rows at FP64, twice that at the mixed policies
@pytest.mark.parametrize("n,waves", [(2048, 4), (2049, 4), (4096, 4), (4097, 4), (8192, 16), (8193, 16), (16384, 16),
                                     (16385, 16), (1, 16), (65, 8)])
@pytest.mark.parametrize("policy", ["fp64", "errbound"])
def test_batch_on_chip_and_in_memory(mf, oracle, n, waves, policy):
    ms = [_band(n, "near"), _band(n, "diag", seed=2)]
    tms = [mf.TiledMatrix(*m) for m in ms]
    bs = [np.random.default_rng(k).uniform(-1, 1, (2, n)) for k in range(2)]
    xs, rep = mf.batch_cg(tms, bs, nrhs=2, tol=TOL, policy=policy, batch_waves=waves)
    for k, m in enumerate(ms):
        for j in range(2):
            assert oracle.rel_residual(*m, bs[k][j], xs[k][j]) <= TOL


@pytest.mark.parametrize("policy", ["fp64", "errbound"])
@pytest.mark.parametrize("waves", [4, 16])
@pytest.mark.parametrize("refresh", [64, 1])
def test_batch_sorted_rows_pieces_and_fallback(mf, oracle, policy, waves, refresh):
    from millefeuille import gen
    m = gen.powerlaw_laplacian(6000, 90000, seed=6)
    tm = mf.TiledMatrix(*m)
    assert tm.strips()["pieces"] > 0
    b = np.random.default_rng(0).uniform(-1, 1, (3, 6000))
    xs, rep = mf.batch_cg([tm], [b], nrhs=3, tol=TOL, policy=policy, batch_waves=waves, max_refresh=refresh)
    for j in range(3):
        assert oracle.rel_residual(*m, b[j], xs[0][j]) <= TOL


@pytest.mark.parametrize("offs", [4, 5, 6, 7, 9])
@pytest.mark.parametrize("kind", ["packed", "near"])
@pytest.mark.parametrize("method", ["cg", "bicgstab"])
def test_wide_rows_at_eight_strips_a_wave(mf, oracle, offs, kind, method):
    """Two pairs of entries in flight: every remainder of 4 to 9 pairs."""
    n, rng = 8150, np.random.default_rng(offs)
    r, c, v = [np.arange(n)], [np.arange(n)], [rng.uniform(2 * offs + 1, 2 * offs + 2, n)]
    for o in (1, 2, 3, 17, 64, 65, 200, 901, 3000)[:offs]:
        i = np.arange(n - o)
        w = -(2.0 ** -rng.integers(0, 4, n - o)) if kind == "packed" else -rng.uniform(0.1, 1, n - o)
        r += [i, i + o]
        c += [i + o, i]
        v += [w, w]
    r, c, v = np.concatenate(r), np.concatenate(c), np.concatenate(v)
    k = np.lexsort((c, r))
    m = np.concatenate([[0], np.cumsum(np.bincount(r, minlength=n))]).astype(np.int32), c[k].astype(np.int32), v[k]
    _check(mf, oracle, m, method, blocks=1)
    y = [_run(mf, m, method, fixed_iters=8, blocks=1, form=f)[3] for f in ("auto", "memory")]
    assert np.max(np.abs(y[0] - y[1])) <= 1e-9 * np.max(np.abs(y[1]))


@pytest.mark.parametrize("method", ["cg", "bicgstab"])
def test_pieces_at_eight_strips_a_wave(mf, oracle, method):
    from millefeuille import gen
    m = gen.powerlaw_laplacian(8100, 120000, seed=7)
    tm, _, _ = _check(mf, oracle, m, method, blocks=1)
    assert tm.strips()["pieces"] > 0
