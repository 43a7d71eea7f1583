"""Register-wavefront triangular sweeps of complete 5- and 7-point grid
patterns (used by default): bit for bit the oracle's apply, transposed apply,
FP32 applies and triangular solves, on grids around the tiles' edges (8 x 8
lines in 3-D, 64 in 2-D, rows a multiple of 8 steps), repeated (the polled
boundary values re-arm themselves), in place and after a refactorisation;
patterns with a missing coupling keep the general sweeps; NaN and infinity
reach exactly the rows they reach in the oracle."""
import numpy as np
import pytest
import torch

import hala_amd as H
import oracle
from hala_amd import stencils as st
from tests.conftest import bits

pytestmark = pytest.mark.gpu

GRIDS = {
    "2x2": lambda: st.laplace2d(2, 2),
    "3x64": lambda: st.laplace2d(3, 64),
    "9x65": lambda: st.laplace2d(9, 65),
    "70x129": lambda: st.laplace2d(70, 129),
    "300x3": lambda: st.laplace2d(300, 3),
    "2x2x2": lambda: st.laplace3d(2, 2, 2),
    "10x8x8": lambda: st.laplace3d(10, 8, 8),
    "11x9x8": lambda: st.laplace3d(11, 9, 8),
    "34x17x25": lambda: st.laplace3d(34, 17, 25),
    "5x40x9": lambda: st.laplace3d(5, 40, 9),
    "diffusion12": lambda: (lambda d: (d["pntr"], d["indx"], d["vals"]))(st.diffusion3d(12, seed=5)),
}


GRID_SWEEP = 2  # path_sweep of the kernels tested here


def host(t):
    return t.detach().cpu().numpy()


def setup(engine, p, i, v, **kw):
    dg, _ = oracle.diag(p, i)
    M = H.make_ilu(engine, engine.load(p), engine.load(i), engine.load(v), **kw)
    return M, dg, oracle.ilu0(p, i, v, dg)


@pytest.mark.parametrize("name", sorted(GRIDS))
def test_grid_apply_bitexact(engine, name):
    p, i, v = GRIDS[name]()
    n = len(p) - 1
    M, dg, f = setup(engine, p, i, v, want_f32=True)
    gr, g32 = engine.vector(n), engine.vector(n, dtype=torch.float32)
    for seed in (71, 72, 73):
        x = st.uniform(seed, n)
        gx = engine.load(x)
        M.apply(gx, gr)
        assert engine.get_option("path_sweep") == GRID_SWEEP
        assert np.array_equal(bits(host(gr)), bits(oracle.ilu_apply(p, i, dg, f, x)))
        M.apply_t(gx, gr)
        assert engine.get_option("path_sweep") == GRID_SWEEP
        assert np.array_equal(bits(host(gr)), bits(oracle.ilu_apply_t(p, i, dg, f, x)))
        ref32 = oracle.ilu_apply_f32(p, i, dg, f.astype(np.float32), x.astype(np.float32))
        M.apply_f32x64(gx, gr)
        assert np.array_equal(bits(host(gr)), bits(ref32.astype(np.float64)))
        M.apply(engine.load(x.astype(np.float32)), g32)
        assert np.array_equal(bits(host(g32)), bits(ref32))
        M.apply(gx, gx)
        assert np.array_equal(bits(host(gx)), bits(oracle.ilu_apply(p, i, dg, f, x)))
    w = v * np.where(i == np.repeat(np.arange(n), np.diff(p)), 1.25, 1.0)
    M.factor(engine.load(w))
    M.apply(engine.load(x), gr)
    assert np.array_equal(bits(host(gr)), bits(oracle.ilu_apply(p, i, dg, oracle.ilu0(p, i, w, dg), x)))


@pytest.mark.parametrize("name", ["9x65", "11x9x8", "34x17x25"])
@pytest.mark.parametrize("uplo", ["L", "U"])
@pytest.mark.parametrize("diag", ["U", "N"])
def test_grid_trsv_bitexact(engine, name, uplo, diag):
    p, i, v = GRIDS[name]()
    n = len(p) - 1
    row = np.repeat(np.arange(n), np.diff(p))
    keep = i <= row if uplo == "L" else i >= row
    q = np.zeros(n + 1, np.int32)
    q[1:] = np.cumsum(np.bincount(row[keep], minlength=n))
    i, v = i[keep].copy(), v[keep] * np.linspace(0.2, 0.3, keep.sum())
    b = st.uniform(5, n)
    T = H.make_triangular_matrix(engine, uplo, diag, engine.load(q), engine.load(i), engine.load(v))
    T32 = H.make_triangular_matrix(engine, uplo, diag, T.pntr, T.indx, T.vals.float())
    for trans in "NT":
        for _ in range(2):
            x, x32 = engine.vector(n), engine.vector(n, dtype=torch.float32)
            T.trsv(trans, 1.5, engine.load(b), x)
            assert engine.get_option("path_sweep") == GRID_SWEEP
            assert np.array_equal(bits(host(x)), bits(oracle.trsv(uplo, trans, diag, 1.5, q, i, v, b)))
            T32.trsv(trans, 1.5, engine.load(b.astype(np.float32)), x32)
            ref = oracle.trsv_f32(uplo, trans, diag, 1.5, q, i, v.astype(np.float32), b.astype(np.float32))
            assert np.array_equal(bits(host(x32)), bits(ref))


@pytest.mark.parametrize("name", ["70x129", "34x17x25"])
def test_grid_incomplete_pattern(engine, name):
    # one symmetric pair of couplings missing in the middle: the general sweeps, same bits
    p, i, v = GRIDS[name]()
    n = len(p) - 1
    row = np.repeat(np.arange(n), np.diff(p))
    r = n // 2
    while not np.any((row == r) & (i == r + 1)):
        r += 1
    keep = ~(((row == r) & (i == r + 1)) | ((row == r + 1) & (i == r)))
    q = np.zeros(n + 1, np.int32)
    q[1:] = np.cumsum(np.bincount(row[keep], minlength=n))
    M, dg, f = setup(engine, q, i[keep].copy(), v[keep].copy())
    x = st.uniform(3, n)
    gr = engine.vector(n)
    M.apply(engine.load(x), gr)
    assert engine.get_option("path_sweep") != GRID_SWEEP
    assert np.array_equal(bits(host(gr)), bits(oracle.ilu_apply(q, i[keep].copy(), dg, f, x)))


@pytest.mark.parametrize("name", ["9x65", "34x17x25"])
@pytest.mark.parametrize("bad", [np.inf, np.nan])
def test_grid_nonfinite(engine, name, bad):
    p, i, v = GRIDS[name]()
    n = len(p) - 1
    M, dg, f = setup(engine, p, i, v)
    x = st.uniform(4, n)
    gr = engine.vector(n)
    for at in (0, n // 2, n - 1):
        y = x.copy()
        y[at] = bad
        M.apply(engine.load(y), gr)
        assert np.array_equal(host(gr), oracle.ilu_apply(p, i, dg, f, y), equal_nan=True)
    M.apply(engine.load(x), gr)  # and nothing stays behind
    assert np.array_equal(bits(host(gr)), bits(oracle.ilu_apply(p, i, dg, f, x)))
