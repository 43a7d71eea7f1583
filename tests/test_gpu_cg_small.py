"""CG of small systems in one workgroup: solutions, histories and iteration
counts bit for bit the oracle's, around the 256-row blocks, at and
past the 4096 rows, short, long and ragged rows, identity and Jacobi, more passes
than one launch runs, an iteration cap, and a breakdown reported as before."""
import numpy as np
import pytest
import torch

import hala_amd as H
import oracle
from hala_amd import stencils as st
from tests.conftest import bits

pytestmark = pytest.mark.gpu


def spd(n, longest, seed):
    """Symmetric, diagonally dominant, rows of 1 .. about `longest` entries."""
    rng = np.random.default_rng(seed)
    m = n * longest // 3
    a, b = rng.integers(0, n, m), rng.integers(0, n, m)
    key = np.unique(np.concatenate([a * n + b, b * n + a, np.arange(n) * n + np.arange(n)]))
    row, col = key // n, key % n
    v = np.where(row == col, 2.0 * longest + 1.0 + (row % 7), -1.0 / (1 + (row + col) % 5))
    p = np.zeros(n + 1, np.int32)
    p[1:] = np.cumsum(np.bincount(row, minlength=n))
    return p, col.astype(np.int32), v


CASES = {
    "1": lambda: (np.array([0, 1], np.int32), np.array([0], np.int32), np.array([3.0])),
    "16^2": lambda: st.laplace2d(16, 16),
    "257 rows": lambda: spd(257, 3, 1),
    "64^2": lambda: st.laplace2d(64, 64),
    "16^3": lambda: st.laplace3d(16, 16, 16),
    "17x241": lambda: st.laplace2d(17, 241),
    "long rows": lambda: spd(900, 9, 2),
    "long rows, full": lambda: spd(4096, 9, 3),
}


@pytest.mark.parametrize("name", sorted(CASES))
@pytest.mark.parametrize("jacobi", [False, True])
def test_small_cg_bitexact(engine, name, jacobi):
    p, i, v = CASES[name]()
    n = len(p) - 1
    if jacobi:
        v = v * (1.0 + 0.0 * v)
    dg = v[i == np.repeat(np.arange(n), np.diff(p))] * 1.5
    b = st.uniform(7, n)
    x0 = st.uniform(8, n)
    tol = 1e-11 * oracle.cnrm2(b)
    kw = dict(prec=oracle.PREC_JACOBI, mdiag=None, mdata=dg) if jacobi else {}
    gp, gi, gv = engine.load(p), engine.load(i), engine.load(v)
    pre = ("jacobi", engine.load(dg)) if jacobi else None
    longest = int(np.diff(p).max())
    small = n <= 4096 and longest <= 16 and longest * n <= 4 * len(i)
    assert small or name in ("17x241", "long rows", "long rows, full")
    for max_iter in (2**31 - 1, 5):
        it, x, hist = oracle.cg(p, i, v, b, x0=x0, tol=tol, max_iter=max_iter, **kw)
        gx, gh = engine.load(x0), torch.zeros(8192, dtype=torch.float64, device="cuda")
        git = H.solve_cg(engine, H.stop_criteria(tol, max_iter), gp, gi, gv, pre, engine.load(b), gx, hist=gh)
        assert engine.get_option("path_cg") == (2 if small else 1)
        assert git == it
        assert np.array_equal(bits(gh.cpu().numpy()[: it - 1]), bits(hist))
        assert np.array_equal(bits(gx.cpu().numpy()), bits(x))


def test_small_cg_many_passes_and_breakdown(engine):
    # a tolerance never met: the cap stops it after several launches' worth of passes
    p, i, v = st.laplace2d(12, 12)
    n = len(p) - 1
    b = st.uniform(3, n)
    gp, gi, gv = engine.load(p), engine.load(i), engine.load(v)
    cap = 1500
    it, x, hist = oracle.cg(p, i, v, b, tol=1e-280, max_iter=cap)
    gx = engine.vector(n)
    assert H.solve_cg(engine, H.stop_criteria(1e-280, cap), gp, gi, gv, None, engine.load(b), gx) == it
    assert np.array_equal(gx.cpu().numpy(), x, equal_nan=True)
    b[5] = np.inf
    with pytest.raises(H.HalaError, match="non-finite"):
        H.solve_cg(engine, 1e-8, gp, gi, gv, None, engine.load(b), engine.vector(n))
