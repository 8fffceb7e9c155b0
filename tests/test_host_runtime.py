"""The library's host code on the CPU, over a stand-in for the HIP runtime
(fake_hip.cpp): allocation failures, which kernels are launched, what lives how
long.  Each snippet runs in a process of its own."""
import os
import subprocess
import sys
import textwrap

import pytest

HERE = os.path.dirname(os.path.abspath(__file__))
ROOT = os.path.dirname(HERE)

PRELUDE = """
import ctypes as C, sys
fake = C.CDLL({shim!r}, mode=C.RTLD_GLOBAL)
fake.fake_log.restype = C.c_char_p
fake.fake_in_use.restype = C.c_size_t
fake.fake_budget.argtypes = [C.c_size_t]
fake.fake_cost.argtypes = [C.c_char_p, C.c_float]
sys.path[:0] = [{pkg!r}]
import numpy as np
import millefeuille as mf
from millefeuille import gen
from millefeuille._lib import lib, MfReport, MfSolveOpts, MfTuneReport

ALL = 2 ** 64 - 1

def log():
    out = fake.fake_log().decode().splitlines()
    fake.fake_clear()
    return out

def launched(name):
    return [l for l in log() if l.startswith("launch mf::" + name)]

class Vec:  # a device array
    def __init__(self, n):
        self.a = np.zeros(n)
        self.ptr = self.a.ctypes.data
"""


@pytest.fixture(scope="module")
def run(tmp_path_factory):
    d = tmp_path_factory.mktemp("fake_hip")
    shim = str(d / "libfakehip.so")
    subprocess.run(["g++", "-std=c++17", "-O1", "-shared", "-fPIC", "-o", shim, os.path.join(HERE, "fake_hip.cpp")],
                   check=True)
    prelude = PRELUDE.format(shim=shim, pkg=os.path.join(ROOT, "mille-feuille_amd"))

    def go(body):
        env = dict(os.environ, MALLOC_PERTURB_="165")  # freed memory is overwritten
        r = subprocess.run([sys.executable, "-c", prelude + textwrap.dedent(body)], capture_output=True, text=True,
                           env=env)
        assert r.returncode == 0, r.stdout + r.stderr
        return r.stdout
    return go


def test_handles_without_room_for_strips_run_on_tiles(run):
    """Every budget from nothing to all: either the tiles do not fit and the
    creation fails, or there is a handle, with strips if they fit too."""
    run("""
    m = gen.laplace3d(12)
    tm = mf.TiledMatrix(*m)
    full = fake.fake_in_use()
    assert tm.strips()["strips"] > 0
    tm.free()
    assert fake.fake_in_use() == 0
    sizes = [int(l.split()[1]) for l in log() if l.startswith("malloc")]
    made = failed = without = 0
    for budget in range(0, sum(sizes), 4096):
        fake.fake_budget(budget)
        try:
            tm = mf.TiledMatrix(*m)
        except mf.MfError as e:
            assert e.code == -4, e  # MF_ERR_HIP
            assert made == 0, "a larger budget failed"
            failed += 1
            assert fake.fake_in_use() == 0
            continue
        made += 1
        if tm.strips()["strips"] == 0:
            without += 1
            fake.fake_budget(ALL)
            log()
            x, y = Vec(tm.npad), Vec(tm.npad)
            tm.spmv(x, y)
            assert launched("k_spmv<")
            tm.cg(x, y)
            assert launched("k_cg<")
            try:
                tm.set_spmv_kernel("strip")
                assert False
            except mf.MfError as e:
                assert e.code == -1
        tm.free()
        assert fake.fake_in_use() == 0
    assert failed and without and made > without, (failed, without, made)
    """)


def test_tuning_one_mode_leaves_strips_to_the_other(run):
    """The stand-in's event times make the row-group kernel, then the strip
    kernel, then the streamed one the fastest candidate."""
    run("""
    tm = mf.TiledMatrix(*gen.laplace3d(12))
    tm.set_spmv_kernel("strip")
    x, y, x32 = Vec(tm.npad), Vec(tm.npad), Vec(tm.npad)

    def kernels():
        log()
        tm.spmv(x, y)
        tm.spmv(x, y, mode=1, d_x32=x32)
        return [l.split()[1] for l in log() if l.startswith("launch")]

    assert kernels() == ["mf::k_spmv_strip<false>", "mf::k_spmv<1,false>"], kernels()
    fake.fake_cost(b"k_spmv_rg", 0.5)
    assert tm.tune_spmv(mode=1)["best"] == 0
    assert kernels() == ["mf::k_spmv_strip<false>", "mf::k_spmv_rg<1>"], kernels()
    fake.fake_cost(b"k_spmv_strip", 0.25)
    assert tm.tune_spmv(mode=0)["best"] == -1
    assert kernels() == ["mf::k_spmv_strip<false>", "mf::k_spmv_rg<1>"], kernels()
    fake.fake_cost(b"k_spmv<", 0.125)
    assert tm.tune_spmv(mode=1)["best"] > 0
    assert kernels() == ["mf::k_spmv_strip<false>", "mf::k_spmv<1,false>"], kernels()
    assert tm.tune_spmv(mode=0)["best"] > 0
    assert kernels() == ["mf::k_spmv<0,false>", "mf::k_spmv<1,false>"], kernels()
    assert tm.spmv_kernel() == tm.spmv_kernel(1) == mf._lib.SPMV_STREAM
    """)


def test_batch_takes_any_iterable_of_right_hand_sides(run):
    run("""
    from millefeuille import core

    class Dev(Vec):
        made = []

        def __init__(self, n, dtype=np.float64):
            super().__init__(n)
            Dev.made.append(self)

        @classmethod
        def from_host(cls, a, dtype=None, length=None):
            d = cls(len(a))
            d.a[:] = a
            return d

        def zero(self):
            self.a[:] = 0

        def get(self, n=None):
            return self.a.copy()

    core.DeviceArray = Dev
    tms = [mf.TiledMatrix(*gen.laplace2d(e)) for e in (5, 8)]
    bs = [np.arange(2 * t.rowA).reshape(2, -1) + 1.0 for t in tms]
    want = None
    for v in (bs, tuple(bs), (b for b in bs), iter(bs), map(np.asarray, bs), {k: b for k, b in enumerate(bs)}.values()):
        Dev.made.clear()
        xs, rep = mf.batch_cg(tms, v, nrhs=2, allow_not_converged=True)
        assert [x.shape for x in xs] == [(2, 25), (2, 64)]
        want = Dev.made[0].a if want is None else want
        np.testing.assert_array_equal(Dev.made[0].a, want)
    """)


def test_policy_labels_share_no_state_with_products(run):
    """A product on another stream may be under way: the labels' own product is
    not the streamed kernel's form that counts pieces in the handle."""
    run("""
    from millefeuille import policy
    n = 20000
    r = np.concatenate([np.zeros(n - 1, np.int64), np.arange(1, n), np.arange(n)])
    c = np.concatenate([np.arange(1, n), np.zeros(n - 1, np.int64), np.arange(n)])
    k = np.lexsort((c, r))
    rp = np.concatenate([[0], np.cumsum(np.bincount(r, minlength=n))]).astype(np.int32)
    tm = mf.TiledMatrix(rp, c[k].astype(np.int32), np.ones(len(k)))
    x, y, lab = Vec(tm.npad), Vec(tm.npad), Vec(tm.tilenum)
    for kernel in ("auto", "stream", "strip", "rowgroup"):
        tm.set_spmv_kernel(kernel)
        log()
        assert lib.mf_policy_labels(tm.h, x.ptr, 1e-5, lab.ptr, None) == 0
        l = log()
        assert any("launch mf::k_labels" in q for q in l)
        assert any("k_spmv_" in q for q in l) and not any("k_spmv<" in q for q in l), l
    tm.set_spmv_kernel("stream")
    tm.spmv(x, y)
    assert launched("k_spmv<0,true>")
    """)


NOALLOC = """
def system(n):
    # diagonal, two scattered entries a row, every 997th row of 600: strips with pieces
    rng = np.random.default_rng(n)
    L = np.full(n, 2)
    L[::997] = 600
    r = np.concatenate([np.repeat(np.arange(n), L), np.arange(n)])
    c = np.concatenate([rng.integers(0, n, L.sum()), np.arange(n)])
    k = np.unique(r * n + c)
    rp = np.concatenate([[0], np.cumsum(np.bincount(k // n, minlength=n))]).astype(np.int32)
    tm = mf.TiledMatrix(rp, (k % n).astype(np.int32), np.ones(len(k)))
    assert tm.strips()["pieces"] > 0
    return tm, Vec(tm.npad), Vec(tm.npad)
"""


def test_noalloc_schedules_outlive_their_copies(run):
    """Copies of host arrays wait until the stream is synchronised; the arrays
    must still be there then (freed memory is overwritten)."""
    run(NOALLOC + textwrap.dedent("""
    for n in (2000, 20000):
        tm, b, x = system(n)
        for kw in ({}, {"form": "memory"}, {"policy": "errbound"}, {"policy": "rule"}):
            log()
            tm.cg_noalloc(b, x, **kw)
            l = log()
            assert any("k_cg_strip" in q for q in l) == (kw in ({}, {"policy": "errbound"})), (kw, l)
            assert not any(q.startswith("malloc") for q in l), l
            assert fake.fake_stale_copies() == 0, kw
        tm.free()
    """))


def test_noalloc_takes_the_same_systems_over_strips_as_over_tiles(run):
    """On both sides of the largest system whose tile solve fits the scratch."""
    run(NOALLOC + textwrap.dedent("""
    def accepted(n, **kw):
        tm, b, x = system(n)
        log()
        try:
            tm.cg_noalloc(b, x, **kw)
            l = log()
            assert any("k_cg_strip" in q for q in l) == (not kw), l
            return True
        except mf.MfError as e:
            assert e.code == -1, e
            return False
        finally:
            tm.free()

    lo, hi = 120000, 200000  # fits, does not
    assert accepted(lo, form="memory") and not accepted(hi, form="memory")
    while hi - lo > 32:
        n = (lo + hi) // 2
        lo, hi = (n, hi) if accepted(n, form="memory") else (lo, n)
    for n in range(lo - 64, hi + 64, 16):
        assert accepted(n) == accepted(n, form="memory"), n
    """))
