"""Row strips (one matrix row per lane) against the oracle's CSR product:
packed strips (every off-diagonal value an 8-bit multiple of a power of two),
full ones, sorted layouts and the pieces of long rows, at the sizes where a
strip, a window of strips, a pair of entries or a piece ends.

Tolerance: a row of n products summed in FP64 in any order is within
n * 2^-53 * sum|a x| of the exact sum; 1e-14 covers two such sums of the
rows here up to 45 terms, and rows of more terms get n * 2.3e-16."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def _csr(n, cols, rng, values, diag=True):
    """CSR with the given off-diagonal columns per row and `values(k)`."""
    rp, ci, va = [0], [], []
    for i in range(n):
        c = sorted(set(int(j) for j in cols[i]) | ({i} if diag else set()))
        ci += c
        va += [float(np.pi + i) if j == i and diag else v for j, v in zip(c, values(len(c)))]
        rp.append(len(ci))
    return np.array(rp, np.int32), np.array(ci, np.int32), np.array(va, np.float64)


def _check(mf, oracle, rp, ci, va, seed=0):
    n = len(rp) - 1
    tm = mf.TiledMatrix(rp, ci, va)
    tm.set_spmv_kernel("strip")
    x = np.random.default_rng(seed).uniform(-1, 1, n)
    dx, dy = tm.vector(x), tm.vector(np.full(n, 7.0))
    tm.spmv(dx, dy)
    y = dy.get()
    bound = oracle.csr_spmv(rp, ci, np.abs(va), np.abs(x))
    tol = np.maximum(1e-14, 2.3e-16 * np.diff(rp)) * bound + 1e-300
    assert np.all(np.abs(y[:n] - oracle.csr_spmv(rp, ci, va, x)) <= tol)
    assert not y[n:].any()
    tm.spmv(dx, dy)
    np.testing.assert_array_equal(dy.get(), y)
    return tm


@pytest.mark.parametrize("n", [1, 15, 16, 63, 64, 65, 130, 1023, 1025])
@pytest.mark.parametrize("kind", ["packed", "full"])
def test_regular_rows(mf, oracle, n, kind):
    rng = np.random.default_rng(n)
    vals = {"packed": lambda k: rng.integers(-127, 128, k) * 0.125, "full": lambda k: rng.standard_normal(k)}[kind]
    cols = [[j for j in (i - 17, i - 1, i + 1, i + 5, i + 64) if 0 <= j < n] for i in range(n)]
    tm = _check(mf, oracle, *_csr(n, cols, rng, vals))
    s = tm.strips()
    # a strip with rows past the matrix is full
    assert s["strips"] == (n + 63) // 64 and (s["packed_slots"] > 0) == (kind == "packed" and n >= 64)


@pytest.mark.parametrize("width", list(range(0, 14)) + [20, 31])
@pytest.mark.parametrize("kind", ["packed", "full"])
def test_row_widths(mf, oracle, width, kind):
    """Every number of pairs up to the software pipeline's second round."""
    n, rng = 128, np.random.default_rng(width)
    vals = {"packed": lambda k: -np.ones(k), "full": lambda k: rng.standard_normal(k)}[kind]
    cols = [rng.choice(np.delete(np.arange(n), i), width, replace=False) for i in range(n)]
    _check(mf, oracle, *_csr(n, cols, rng, vals))


@pytest.mark.parametrize("kind", ["packed", "full", "mixed"])
@pytest.mark.parametrize("diag", [True, False])
def test_sorted_rows_and_pieces(mf, oracle, kind, diag):
    """Row lengths 0 to 1700 over two windows of 1024 rows: sorted strips,
    rows of one and of several pieces (512 entries each), empty rows."""
    n, rng = 1900, np.random.default_rng(3)
    ln = rng.integers(0, 9, n)
    for r, k in ((0, 63), (5, 64), (6, 65), (700, 512), (701, 513), (1030, 514), (1031, 1024), (1500, 1700), (1899, 66)):
        ln[r] = k
    full = lambda k: rng.standard_normal(k)
    one = lambda k: -2.0 ** -3 * np.ones(k)
    vals = {"packed": one, "full": full, "mixed": lambda k: full(k) if k % 5 == 0 else one(k)}[kind]
    cols = [rng.choice(np.delete(np.arange(n), i), ln[i], replace=False) for i in range(n)]
    tm = _check(mf, oracle, *_csr(n, cols, rng, vals, diag))
    s = tm.strips()
    assert s["sorted"] == 1 and s["pieces"] >= 9
    if kind == "packed" and diag:
        assert s["packed_slots"] > s["full_slots"]


@pytest.mark.parametrize("values,packed", [((127.0, -127.0), True), ((128.0, -1.0), False), ((129.0, 1.0), False),
                                           ((2.0 ** -90, 127 * 2.0 ** -90), True), ((2.0 ** -110, 1.0), False),
                                           ((2.0 ** 90, -3 * 2.0 ** 90), True), ((0.0, -0.0), True),
                                           ((0.1, 0.1), False), ((1e300, 1e300), False)])
def test_packing_is_exact_or_not_used(mf, oracle, values, packed):
    n, rng = 128, np.random.default_rng(1)
    cols = [[(i + 1) % n, (i + 9) % n] for i in range(n)]
    tm = _check(mf, oracle, *_csr(n, cols, rng, lambda k: [values[q % 2] for q in range(k)]))
    assert (tm.strips()["full_slots"] == 0) == packed


@pytest.mark.parametrize("kind", ["packed", "full"])
@pytest.mark.parametrize("bad", [np.inf, np.nan])
def test_non_finite_x_reaches_only_coupled_rows(mf, oracle, kind, bad):
    n, rng = 200, np.random.default_rng(2)
    vals = {"packed": lambda k: -np.ones(k), "full": lambda k: rng.uniform(1, 2, k)}[kind]
    ln = rng.integers(0, 9, n)
    cols = [rng.choice(np.delete(np.arange(n), i), ln[i], replace=False) for i in range(n)]
    rp, ci, va = _csr(n, cols, rng, vals)
    tm = mf.TiledMatrix(rp, ci, va)
    tm.set_spmv_kernel("strip")
    x = rng.uniform(1, 2, n)
    x[[0, 77]] = bad
    dx, dy = tm.vector(x), tm.vector()
    tm.spmv(dx, dy)
    rows = np.repeat(np.arange(n), np.diff(rp))
    hit = np.zeros(n, bool)
    hit[rows[np.isin(ci, [0, 77])]] = True
    np.testing.assert_array_equal(~np.isfinite(dy.get()[:n]), hit)


def _stencil(n, offs, vals, diag, rng, shuffle=False):
    """CSR with value vals[k] at offset offs[k] wherever the column exists;
    diag: "same", "each" (its own value per row) or "some" (every third row)."""
    rp, ci, va = [0], [], []
    for i in range(n):
        row = [(i + o, v) for o, v in zip(offs, vals) if 0 <= i + o < n]
        if diag != "some" or i % 3 == 0:
            row.append((i, 5.5 if diag != "each" else 0.3 + i))
        row.sort()
        if shuffle:
            rng.shuffle(row)
        ci += [c for c, _ in row]
        va += [v for _, v in row]
        rp.append(len(ci))
    return np.array(rp, np.int32), np.array(ci, np.int32), np.array(va, np.float64)


@pytest.mark.parametrize("n", [1, 16, 63, 64, 65, 130, 1025])
@pytest.mark.parametrize("diag", ["same", "each", "some"])
@pytest.mark.parametrize("shuffle", [False, True])
def test_diagonals(mf, oracle, n, diag, shuffle):
    """One value for each diagonal of a strip; the first and last rows lack
    entries, as does the last strip."""
    rng = np.random.default_rng(n)
    rp, ci, va = _stencil(n, [-90, -64, -17, -1, 1, 17, 64, 90], [-0.1, 1 / 3, 0.0, -1, -1.7, 2, 1e-3, 1e6], diag, rng, shuffle)
    tm = _check(mf, oracle, rp, ci, va)
    if n == 1025 and not shuffle:
        assert tm.strips()["diag_slots"] > 0
    # the streamed kernel over the same payload
    x = rng.uniform(-1, 1, n)
    dx, ys, yt = tm.vector(x), tm.vector(), tm.vector()
    tm.spmv(dx, ys)
    tm.set_spmv_kernel("stream")
    tm.spmv(dx, yt)
    bound = oracle.csr_spmv(rp, ci, np.abs(va), np.abs(x))
    assert np.all(np.abs(ys.get() - yt.get())[:n] <= 1e-14 * bound + 1e-300)


@pytest.mark.parametrize("slots", list(range(0, 15)) + [63, 64, 65])
def test_diagonal_counts(mf, oracle, slots):
    """Every remainder of the groups of gathers, and the most slots of a strip."""
    n, rng = 600, np.random.default_rng(slots)
    offs = sorted(rng.choice([o for o in range(-150, 151) if o], slots, replace=False))
    rp, ci, va = _stencil(n, offs, list(rng.standard_normal(slots)), "same", rng)
    tm = _check(mf, oracle, rp, ci, va)
    # (strips at the ends have fewer diagonals)
    assert tm.strips()["diag_slots"] > 0 and (tm.strips()["full_slots"] > 0 or slots <= 64)


@pytest.mark.parametrize("bad", [np.inf, np.nan])
def test_diagonals_non_finite_x(mf, oracle, bad):
    n = 1280
    rp, ci, va = _stencil(n, [-65, -1, 1, 65], [1.0] * 4, "some", None)
    tm = mf.TiledMatrix(rp, ci, va)
    tm.set_spmv_kernel("strip")
    x = np.random.default_rng(2).uniform(1, 2, n)
    x[[0, 77]] = bad
    dx, dy = tm.vector(x), tm.vector()
    tm.spmv(dx, dy)
    assert tm.strips()["diag_slots"] > 0
    hit = np.zeros(n, bool)
    hit[np.repeat(np.arange(n), np.diff(rp))[np.isin(ci, [0, 77])]] = True
    np.testing.assert_array_equal(~np.isfinite(dy.get()[:n]), hit)
