"""Solver paths that the grid sweeps and the one-workgroup CG took over from on
the other tests' complete grids, and that every other matrix still runs: the
column sweeps fused into PCG (hand-off, x updated on the helper workgroups, the
stopping pass's own update), the column and level-pool sweeps, and CG whose
direction update rides in the product.  Bit for bit the oracle's, with the path
checked."""
import numpy as np
import pytest
import torch

import hala_amd as H
import oracle
from hala_amd import stencils as st
from tests.conftest import bits

pytestmark = pytest.mark.gpu


def host(t):
    return t.detach().cpu().numpy()


class options:
    def __init__(self, engine, **kw):
        self.engine, self.kw = engine, kw

    def __enter__(self):
        self.saved = {k: self.engine.get_option(k) for k in self.kw}
        for k, v in self.kw.items():
            self.engine.set_option(k, v)

    def __exit__(self, *a):
        for k, v in self.saved.items():
            self.engine.set_option(k, v)


def holes(p, i, v, every):
    """The matrix without the symmetric pairs of couplings (r, r + 1) of every `every`-th row r."""
    n = len(p) - 1
    row = np.repeat(np.arange(n), np.diff(p))
    gone = ((i == row + 1) & (row % every == 0)) | ((row == i + 1) & (i % every == 0))
    q = np.zeros(n + 1, np.int32)
    q[1:] = np.cumsum(np.bincount(row[~gone], minlength=n))
    return q, i[~gone].copy(), v[~gone].copy()


PCG = {  # name: (matrix, options, path_pcg)
    "grid": (lambda: st.laplace3d(32, 32, 32), {}, 2),
    "columns": (lambda: st.laplace3d(32, 32, 32), {"tri_grid": 0}, 1),
    "columns ragged": (lambda: st.laplace3d(30, 31, 29), {"tri_grid": 0}, 1),
    "columns ragged, dispatch order": (lambda: st.laplace3d(30, 31, 29), {"tri_grid": 0, "cg_xcd": 0}, 1),
    "columns separate": (lambda: st.laplace3d(32, 32, 32), {"tri_grid": 0, "cg_fuse": 0}, 0),
    "columns, grid-stride product": (lambda: st.laplace3d(40, 40, 40), {"tri_grid": 0, "spmv_blocks_per_cu": 2}, 1),
    "mesh with holes": (lambda: holes(*st.laplace3d(30, 31, 29), 97), {}, 1),
    "mesh with holes, separate": (lambda: holes(*st.laplace3d(30, 31, 29), 97), {"cg_fuse": 0}, 0),
    "level pool": (lambda: st.laplace3d(20, 21, 19), {"tri_col": 0}, 0),
}


@pytest.mark.parametrize("name", sorted(PCG))
def test_pcg_paths_bitexact(engine, name):
    mat, opts, path = PCG[name]
    p, i, v = mat()
    n = len(p) - 1
    b = st.uniform(202, n)
    tol = 1e-10 * oracle.cnrm2(b)
    dg, _ = oracle.diag(p, i)
    it, x, hist = oracle.cg(p, i, v, b, tol=tol, prec=oracle.PREC_ILU, mpntr=p, mindx=i, mdiag=dg,
                            mdata=oracle.ilu0(p, i, v, dg))
    with options(engine, **opts):
        gp, gi, gv = engine.load(p), engine.load(i), engine.load(v)
        M = H.make_ilu(engine, gp, gi, gv)
        for _ in range(2):  # the polled outputs re-arm themselves
            gx, gh = engine.vector(n), torch.zeros(2000, dtype=torch.float64, device="cuda")
            git = H.solve_cg_ilu(engine, tol, gp, gi, gv, M, engine.load(b), gx, hist=gh)
            assert engine.get_option("path_pcg") == path
            assert git == it
            assert np.array_equal(bits(host(gh)[: it - 1]), bits(hist))
            assert np.array_equal(bits(host(gx)), bits(x))


SWEEPS = {  # name: (matrix, options, path_sweep)
    "columns of a grid": (lambda: st.laplace3d(24, 24, 24), {"tri_grid": 0}, 1),
    "mesh with holes": (lambda: holes(*st.laplace3d(24, 23, 22), 50), {}, 1),
    "2-D mesh with holes": (lambda: holes(*st.laplace2d(90, 71), 64), {}, 1),
    "27-point": (lambda: st.convdiff27(16, seed=3), {}, 1),
    "level pool": (lambda: st.laplace3d(24, 24, 24), {"tri_col": 0}, 0),
}


@pytest.mark.parametrize("name", sorted(SWEEPS))
def test_sweep_paths_bitexact(engine, name):
    mat, opts, path = SWEEPS[name]
    p, i, v = mat()
    n = len(p) - 1
    dg, _ = oracle.diag(p, i)
    f = oracle.ilu0(p, i, v, dg)
    x = st.uniform(22, n)
    with options(engine, **opts):
        M = H.make_ilu(engine, engine.load(p), engine.load(i), engine.load(v), want_f32=True)
        gx, gr = engine.load(x), engine.vector(n)
        for _ in range(2):
            M.apply(gx, gr)
            assert engine.get_option("path_sweep") == path
            assert np.array_equal(bits(host(gr)), bits(oracle.ilu_apply(p, i, dg, f, x)))
            M.apply_f32x64(gx, gr)
            assert engine.get_option("path_sweep") == path
            ref = oracle.ilu_apply_f32(p, i, dg, f.astype(np.float32), x.astype(np.float32)).astype(np.float64)
            assert np.array_equal(bits(host(gr)), bits(ref))
            M.apply_t(gx, gr)
            assert engine.get_option("path_sweep") == path
            assert np.array_equal(bits(host(gr)), bits(oracle.ilu_apply_t(p, i, dg, f, x)))


THIN = {  # name: (matrix, path_sweep of one vector); complete grids, on the columns where a hop comes every few levels
    "8x8x400": (lambda: st.laplace3d(8, 8, 400), 1),
    "9x400x9": (lambda: st.laplace3d(9, 400, 9), 1),
    "400x9x9": (lambda: st.laplace3d(400, 9, 9), 2),
    "3x60x60": (lambda: st.laplace3d(3, 60, 60), 1),
    "12x60x60": (lambda: st.laplace3d(12, 60, 60), 2),
    "2x500": (lambda: st.laplace2d(2, 500), 2),
}


@pytest.mark.parametrize("name", sorted(THIN))
def test_thin_grids(engine, name):
    mat, path = THIN[name]
    p, i, v = mat()
    n = len(p) - 1
    dg, _ = oracle.diag(p, i)
    f = oracle.ilu0(p, i, v, dg)
    gp, gi, gv = engine.load(p), engine.load(i), engine.load(v)
    M = H.make_ilu(engine, gp, gi, gv)
    x = st.uniform(31, n)
    gx, gr = engine.load(x), engine.vector(n)
    for _ in range(2):
        M.apply(gx, gr)
        assert engine.get_option("path_sweep") == path
        assert np.array_equal(bits(host(gr)), bits(oracle.ilu_apply(p, i, dg, f, x)))
        M.apply_t(gx, gr)
        assert np.array_equal(bits(host(gr)), bits(oracle.ilu_apply_t(p, i, dg, f, x)))
        # several vectors take the grid sweeps in every case
        B = np.stack([st.uniform(40 + k, n) for k in range(3)])
        X = torch.zeros(3, n, dtype=torch.float64, device="cuda")
        H.solve_batch_cg_ilu(engine, H.stop_criteria(0.0, 6), gp, gi, gv, M, engine.load(B), X)
        assert engine.get_option("path_sweep") == engine.get_option("path_pcg") == 2
        gx1 = engine.vector(n)
        H.solve_cg_ilu(engine, H.stop_criteria(0.0, 6), gp, gi, gv, M, engine.load(B[1]), gx1)
        assert engine.get_option("path_pcg") == path
        _, ref, _ = oracle.cg(p, i, v, B[1], tol=0.0, max_iter=6, prec=oracle.PREC_ILU, mpntr=p, mindx=i, mdiag=dg, mdata=f)
        assert np.array_equal(bits(host(X[1])), bits(ref)) and np.array_equal(bits(host(gx1)), bits(ref))


@pytest.mark.parametrize("prec", ["identity", "jacobi"])
@pytest.mark.parametrize("side,opts,path", [(64, {"cg_small": 0}, 1), (65, {}, 1), (64, {}, 2), (520, {}, 0)])
def test_cg_paths_bitexact(engine, prec, side, opts, path):
    p, i, v = st.laplace2d(side, side, diag=4.3)
    n = len(p) - 1
    d = np.full(n, 4.3)
    b = st.uniform(404 + side, n)
    kind = oracle.PREC_JACOBI if prec == "jacobi" else oracle.PREC_IDENTITY
    it, x, hist = oracle.cg(p, i, v, b, tol=0.0, max_iter=40, prec=kind, mdata=d)
    gp, gi, gv = engine.load(p), engine.load(i), engine.load(v)
    gx, gh = engine.vector(n), torch.zeros(64, dtype=torch.float64, device="cuda")
    pre = ("jacobi", engine.load(d)) if prec == "jacobi" else None
    with options(engine, **opts):
        git = H.solve_cg(engine, H.stop_criteria(0.0, 40), gp, gi, gv, pre, engine.load(b), gx, hist=gh)
    assert engine.get_option("path_cg") == path
    assert git == it == 40
    assert np.array_equal(bits(host(gh)[: it - 1]), bits(hist[: it - 1]))
    assert np.array_equal(bits(host(gx)), bits(x))


def test_path_names_are_read_only(engine):
    with pytest.raises(H.HalaError, match="unknown option"):
        engine.set_option("path_cg", 1)
    with pytest.raises(H.HalaError, match="unknown option"):
        engine.get_option("path_none")


def test_layouts_follow_options_and_factorisations(engine):
    # the factor's values are packed for the sweeps that run: every other layout on its first use, and
    # none of them survives a new factorisation (FP32 ones too, where it asked for FP64 only)
    p, i, v = st.laplace3d(13, 12, 11)
    n = len(p) - 1
    dg, _ = oracle.diag(p, i)
    w = v * np.where(i == np.repeat(np.arange(n), np.diff(p)), 1.25, 1.0)
    x = st.uniform(9, n)
    M = H.make_ilu(engine, engine.load(p), engine.load(i), engine.load(v), want_f32=True)
    gx, gr = engine.load(x), engine.vector(n)

    def check(vals, path):
        f = oracle.ilu0(p, i, vals, dg)
        M.apply(gx, gr)
        assert engine.get_option("path_sweep") == path
        assert np.array_equal(bits(host(gr)), bits(oracle.ilu_apply(p, i, dg, f, x)))
        M.apply_f32x64(gx, gr)
        ref = oracle.ilu_apply_f32(p, i, dg, f.astype(np.float32), x.astype(np.float32)).astype(np.float64)
        assert np.array_equal(bits(host(gr)), bits(ref))
        M.apply_t(gx, gr)
        assert np.array_equal(bits(host(gr)), bits(oracle.ilu_apply_t(p, i, dg, f, x)))
        gs = engine.vector(n)
        H.solve_cg_ilu(engine, H.stop_criteria(0.0, 5), M.pntr, M.indx, engine.load(vals), M, gx, gs)
        _, ref, _ = oracle.cg(p, i, vals, x, tol=0.0, max_iter=5, prec=oracle.PREC_ILU, mpntr=p, mindx=i, mdiag=dg, mdata=f)
        assert np.array_equal(bits(host(gs)), bits(ref))

    ways = [({}, 2), ({"tri_grid": 0}, 1), ({"tri_col": 0}, 0), ({}, 2), ({"tri_col_cols": 4}, 1)]
    for opts, path in ways:
        with options(engine, **opts):
            check(v, path)
    for first, _ in ways[:3]:
        with options(engine, **first):
            M.factor(engine.load(w))  # FP64 only
        for opts, path in ways:
            with options(engine, **opts):
                check(w, path)
        with options(engine, **first):
            M.factor(engine.load(v), want_f32=True)
        for opts, path in ways:
            with options(engine, **opts):
                check(v, path)


def test_layout_first_used_under_capture():
    # a pack that a capture recorded has not run: the next eager call packs again, and replays give the same bits
    p, i, v = st.laplace3d(13, 12, 11)
    n = len(p) - 1
    dg, _ = oracle.diag(p, i)
    f = oracle.ilu0(p, i, v, dg)
    s = torch.cuda.Stream()
    with torch.cuda.stream(s):
        eng = H.gpu_engine(0, stream=s)
        eng.set_option("sync_checks", 0)
        M = H.make_ilu(eng, eng.load(p), eng.load(i), eng.load(v))
        gx, gr, ge = eng.load(st.uniform(1, n)), eng.vector(n), eng.vector(n)
        M.apply(gx, ge)  # the grid sweeps
        eng.set_option("tri_grid", 0)
        torch.cuda.synchronize()
        g = torch.cuda.CUDAGraph()
        with torch.cuda.graph(g, stream=s):
            M.apply(gx, gr)
        for seed in (1, 2, 3):
            x = st.uniform(seed, n)
            ref = bits(oracle.ilu_apply(p, i, dg, f, x))
            gx.copy_(eng.load(x))
            M.apply(gx, ge)
            assert eng.get_option("path_sweep") == 1
            assert np.array_equal(bits(host(ge)), ref)
            g.replay()
            torch.cuda.synchronize()
            assert np.array_equal(bits(host(gr)), ref)
            eng.synchronize()


def test_pair_keeps_no_unused_buffers():
    # a factor's grid sweeps: input and output of L, output of U, one set of boundary values each, and the
    # records; nothing that no sweep reads (U's input and second sets made it 5 packed vectors instead of 3.5)
    eng = H.gpu_engine(0)
    p, i, v = st.laplace3d(128, 128, 64)
    n = len(p) - 1
    gp, gi, gv = eng.load(p), eng.load(i), eng.load(v)
    B = torch.zeros(16, n, dtype=torch.float64, device="cuda")
    X = torch.zeros_like(B)
    M = H.make_ilu(eng, gp, gi, gv)
    H.solve_batch_cg_ilu(eng, H.stop_criteria(0.0, 2), gp, gi, gv, M, B[:1].contiguous(), X[:1].contiguous())
    B[:] = 1.0
    H.solve_batch_cg(eng, H.stop_criteria(0.0, 2), gp, gi, gv, None, B, X)  # the context's partials for 16
    held = eng.get_option("held_mib")
    H.solve_batch_cg_ilu(eng, H.stop_criteria(0.0, 2), gp, gi, gv, M, B, X)
    packed = 16 * 16 * 8 * 144 * 64 * 8 >> 20  # 16 vectors of 16 x 8 tiles, 144 steps of 64 lanes
    grown = eng.get_option("held_mib") - held
    assert abs(grown - 3.5 * packed) <= 1, grown / packed  # 3 vectors + 2 sets of a quarter


@pytest.mark.parametrize("name", ["grid", "columns"])
def test_captured_sweeps_survive_larger_solves(name):
    # a captured apply and a captured trsm hold their buffers' addresses: solves of more vectors on the same
    # objects leave them alone, and replays give the eager bits
    p, i, v = st.laplace3d(13, 12, 11)
    n = len(p) - 1
    row = np.repeat(np.arange(n), np.diff(p))
    keep = i <= row
    q = np.zeros(n + 1, np.int32)
    q[1:] = np.cumsum(np.bincount(row[keep], minlength=n))
    li, lv = i[keep].copy(), v[keep].copy()
    dg, _ = oracle.diag(p, i)
    f = oracle.ilu0(p, i, v, dg)
    s = torch.cuda.Stream()
    with torch.cuda.stream(s):
        eng = H.gpu_engine(0, stream=s)
        eng.set_option("sync_checks", 0)
        eng.set_option("tri_grid", 1 if name == "grid" else 0)
        gp, gi, gv = eng.load(p), eng.load(i), eng.load(v)
        M = H.make_ilu(eng, gp, gi, gv)
        T = H.make_triangular_matrix(eng, "L", "N", eng.load(q), eng.load(li), eng.load(lv))
        gx, gr = eng.load(st.uniform(1, n)), eng.vector(n)
        b = np.stack([st.uniform(20 + k, n) for k in range(3)])
        gb = eng.load(b)
        M.apply(gx, gr)
        T.trsm("N", "N", 3, 1.5, gb.clone())
        eng.synchronize()
        torch.cuda.synchronize()
        g = torch.cuda.CUDAGraph()
        with torch.cuda.graph(g, stream=s):
            M.apply(gx, gr)
            T.trsm("N", "N", 3, 1.5, gb)
        for seed in (4, 5, 6):
            # more vectors than the captured calls had, on the same objects
            k = 4 * seed
            B = torch.rand(k, n, dtype=torch.float64, device="cuda")
            T.trsm("N", "N", k, 1.0, B)
            X = torch.zeros(k, n, dtype=torch.float64, device="cuda")
            H.solve_batch_cg_ilu(eng, H.stop_criteria(0.0, 3), gp, gi, gv, M, torch.ones_like(X), X)
            x = st.uniform(seed, n)
            gx.copy_(eng.load(x))
            gb.copy_(eng.load(b * seed))
            g.replay()
            torch.cuda.synchronize()
            assert np.array_equal(bits(host(gr)), bits(oracle.ilu_apply(p, i, dg, f, x)))
            for c in range(3):
                ref = oracle.trsv("L", "N", "N", 1.5, q, li, lv, b[c] * seed)
                assert np.array_equal(bits(host(gb[c])), bits(ref))
            eng.synchronize()
