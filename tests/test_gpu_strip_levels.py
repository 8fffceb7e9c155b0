"""Learned levels over row strips: a tile of the FP64 class is multiplied from
its FP64 payload wherever it lies and however the tiles are spread over the
tile-rows.

The installed network predicts FP64 for tiles of more than 128 entries and FP32
for all others.  The handle's FP32 payload of the dense tiles is half their
value, so a product that takes it is off by its half.  One iteration from x = 0
gives x in closed form; the vectors p, s and r are FP32 (2^-24 relative each,
a handful of roundings), so 1e-5 covers the right result, and the wrong one is
off by more than 1e-2."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def _dense_is_fp64():
    """8-32-32-4 network: logit 0 = 10 * max(64 * (nnz / 256) - 32, 0), logit 1 = 0.5."""
    w1, b1 = np.zeros((32, 8)), np.zeros(32)
    w2, b2 = np.zeros((32, 32)), np.zeros(32)
    w3, b3 = np.zeros((4, 32)), np.zeros(4)
    w1[0, 0], b1[0] = 64.0, -32.0
    w2[0, 0] = 1.0
    w3[0, 0] = 10.0
    b3[:] = (0.0, 0.5, -1.0, -1.0)
    return np.concatenate([a.ravel() for a in (w1, b1, w2, b2, w3, b3)]).astype(np.float32)


def _matrix(n, dense, light):
    """SPD matrix: rows with couplings at +-1 (rows in `light`: their tile-rows
    hold one to three tiles) or besides at +-40 and +-90 (seven), and the 16 x 16
    diagonal tiles of strip `dense` full.  Values are exact in FP32."""
    a = {}
    rng = np.random.default_rng(n)

    def put(i, j, v):
        a[i, j] = a[j, i] = v

    for i in range(n):
        for o in (1,) if light[0] <= i < light[1] else (1, 40, 90):
            if i + o < n:
                put(i, i + o, -float(rng.integers(1, 2000)) / 4096.0)
    for r in range(64 * dense, min(64 * dense + 64, n)):
        for c in range(16 * (r // 16), min(16 * (r // 16) + 16, n)):
            if c > r:
                put(r, c, -float(rng.integers(1, 2000)) / 4096.0)
    for i in range(n):
        a[i, i] = 20.0 + float(rng.integers(0, 4096)) / 1024.0
    k = sorted(a)
    r, c = np.array([q[0] for q in k]), np.array([q[1] for q in k])
    v = np.array([a[q] for q in k])
    rp = np.concatenate([[0], np.cumsum(np.bincount(r, minlength=n))]).astype(np.int32)
    low = v.astype(np.float32)
    low[(r // 64 == dense) & (r // 16 == c // 16)] *= 0.5
    return rp, c.astype(np.int32), v, low


@pytest.mark.parametrize("blocks", [2, 4, 8])
@pytest.mark.parametrize("dense", [0, 7, 15, 16, 17, 31])
@pytest.mark.parametrize("light", [(0, 1024), (1024, 2048)])
def test_fp64_tiles_run_in_fp64(mf, oracle, blocks, dense, light):
    from millefeuille import policy
    n = 2040
    rp, ci, va, low = _matrix(n, dense, light)
    tm = mf.TiledMatrix(rp, ci, va, val_low=low)
    assert tm.strips()["lean"] == 1 and tm.strips()["sorted"] == 0, tm.strips()
    policy.install(tm, _dense_is_fp64())
    b = np.random.default_rng(dense).integers(-4096, 4097, n) / 4096.0  # exact in FP32
    Ab = oracle.csr_spmv(rp, ci, va, b)
    alpha = b @ b / (b @ Ab)
    want = {"cg": alpha * b}
    # BiCGSTAB: r^ = p = b, s = b - alpha A b, x = alpha b + omega s
    s = b - alpha * Ab
    t = oracle.csr_spmv(rp, ci, va, s)
    want["bicgstab"] = alpha * b + (t @ s) / (t @ t) * s
    for method in ("cg", "bicgstab"):
        db, dx = tm.vector(b), tm.vector()
        rep = getattr(tm, method)(db, dx, policy="learned", fixed_iters=1, blocks=blocks, allow_not_converged=True)
        x = dx.get()[:n]
        assert rep["policy_used"] == mf.POLICY_LEARNED and rep["grid_blocks"] == blocks
        assert rep["prec_hist"][0] > 0 and rep["prec_hist"][1] > 0, rep
        err = np.max(np.abs(x - want[method])) / np.max(np.abs(want[method]))
        assert err <= 1e-5, (method, err)
