"""Several vectors at once: the fused sparse-times-dense product around its
group sizes and tiles, triangular solves with many right-hand sides on the
grid, column and level-pool sweeps, and multi-right-hand-side ILU-PCG -- every
column bit for bit what the oracle (or the one-column call, pinned elsewhere)
gives."""
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


def raw(a):
    a = np.ascontiguousarray(a)
    return bits(a.view(np.float64 if a.dtype in (np.complex128, np.float64) else np.float32))


def ragged(nr, nc, seed, longest, full=True):
    """Rows of 0 .. longest entries, with `full` one row with all nc columns."""
    rng = np.random.default_rng(seed)
    p, i = [0], []
    for r in range(nr):
        k = nc if full and r == nr // 3 else int(rng.integers(0, longest + 1))
        i.extend(np.sort(rng.choice(nc, size=min(k, nc), replace=False)))
        p.append(len(i))
    return np.array(p, np.int32), np.array(i, np.int32)


MATS = {
    "band": lambda: (lambda p, i, v: (p, i, len(p) - 1))(*st.laplace3d(9, 8, 8)),  # int16 offsets, tile remainders
    "ragged": lambda: (*ragged(517, 3000, 3, 9), 3000),  # a row and a tile longer than the staging
    "wide": lambda: (*ragged(260, 70000, 4, 5), 70000),  # int32 columns, a row for the wavefront kernel
    "wide short": lambda: (*ragged(260, 70000, 6, 5, full=False), 70000),
    "wide pairs": lambda: (*ragged(260, 140000, 7, 5, full=False), 140000),  # FP64 two columns at once, FP32 four
    "wide alone": lambda: (*ragged(260, 540000, 8, 5, full=False), 540000),  # FP64 one, FP32 one
    "one": lambda: (np.array([0, 1], np.int32), np.array([0], np.int32), 1),
    "empty": lambda: (np.zeros(301, np.int32), np.zeros(0, np.int32), 40),
}


@pytest.mark.parametrize("mat", sorted(MATS))
@pytest.mark.parametrize("ct", [np.float64, np.float32, np.complex128, np.complex64])
def test_spmm_columns(engine, mat, ct):
    p, i, nc = MATS[mat]()
    nr = len(p) - 1
    rng = np.random.default_rng(9)
    cplx = np.issubdtype(ct, np.complexfloating)

    def rnd(*shape):
        a = rng.uniform(-1, 1, shape)
        return (a + 1j * rng.uniform(-1, 1, shape) if cplx else a).astype(ct)

    v = rnd(len(i))
    A = H.make_sparse_matrix(engine, nc, engine.load(p), engine.load(i), engine.load(v))
    z = np.zeros(0)
    for ta in ("N", "T", "C") if cplx else ("N", "T"):
        k, m = (nc, nr) if ta == "N" else (nr, nc)
        for tb, cols, beta in (("N", 1, 0.0), ("N", 2, 0.5), ("N", 3, 0.0), ("N", 5, 0.5), ("N", 8, 0.0), ("N", 9, 0.5),
                               ("T", 5, 0.0), ("C", 9, 0.5)):
            ldb, ldc = (k + 3 if tb == "N" else cols + 1), m + 2
            B = rnd(cols if tb == "N" else k, ldb)  # column-major: row q of this array is column q of B
            C0 = rnd(cols, ldc)
            gC = engine.load(C0)
            A.gemm(ta, tb, k if tb == "N" else cols, cols if tb == "N" else k, 1.5, engine.load(B), ldb, beta, gC, ldc)
            got = host(gC)
            assert np.array_equal(raw(got[:, m:]), raw(C0[:, m:]))  # nothing written past a column
            assert engine.get_option("path_product") == product_path(A, ct, nr, nc, len(i), ta, tb, cols)
            for c in range(cols):
                x = np.ascontiguousarray(B[c, :k] if tb == "N" else (B[:, c].conj() if tb == "C" else B[:, c]))
                y = np.ascontiguousarray(C0[c, :m])
                if ct == np.float64:
                    y = oracle.spmv(ta, nr, nc, 1.5, p, i, v, x, beta, y)
                elif ct == np.float32 and ta == "N":
                    y = oracle.spmv_f32(p, i, v, x, alpha=1.5, beta=beta, y=y)
                else:  # FP32 'T': the complex product with zero imaginary parts, term by term
                    w = ct if cplx else np.complex64
                    yc = y.astype(w)
                    oracle.zspmv(ta, nr, nc, 1.5 + 0j, p, i, v.astype(w), x.astype(w), complex(beta), yc)
                    y = yc if cplx else yc.real.astype(np.float32)
                assert np.array_equal(raw(got[c, :m]), raw(y)), (ta, tb, cols, c)


def product_path(A, ct, nr, nc, nnz, ta, tb, cols):
    """The product's dispatch: 0 single products, 1 staged tiles, 2 rows walked in memory."""
    es = np.dtype(ct).itemsize
    cplx = np.issubdtype(ct, np.complexfloating)
    # vectors past half an XCD's L2 on a pattern without parallel rows: one by one
    alone = ta == "N" and tb == "N" and nc > nr and 2 * nc * es > 4 << 20
    if not cplx and ((tb == "N" and cols == 1) or alone or (ta == "N" and A.info()["kernel"] == 1)):
        return 0
    blocks = ((nr if ta == "N" else nc) + 255) // 256
    tile = 1024 if es == 16 else 2048
    cus = torch.cuda.get_device_properties(0).multi_processor_count
    few = blocks <= cus * (2 if es == 16 and (ta == "N" or cols <= 2) else 1) and nnz > blocks * tile
    return 2 if few or (ta == "N" and A.info()["max_row"] > tile // 4) else 1


MANY = {  # more workgroups than the rule walks, and more than a tile of entries in each; one fewer than it stages
    "27-point 41^3": (lambda: st.convdiff27(41), (np.float64, np.float32)),
    "27-point 40^3": (lambda: st.convdiff27(40), (np.float64, np.float32)),
    "5-point 530^2": (lambda: st.laplace2d(530, 530), (np.float64,)),  # long vectors, parallel rows: not one by one
    "7-point 51^3": (lambda: st.laplace3d(51, 51, 51), (np.complex128,)),
    "7-point 50^3": (lambda: st.laplace3d(50, 50, 50), (np.complex128,)),
}


@pytest.mark.parametrize("mat", sorted(MANY))
def test_spmm_many_tiles(engine, mat):
    gen, types = MANY[mat]
    p, i, v = gen()
    n = len(p) - 1
    rng = np.random.default_rng(2)
    for ct in types:
        cplx = ct == np.complex128
        w = (v * (1 + 0.5j) if cplx else v).astype(ct)
        A = H.make_sparse_matrix(engine, n, engine.load(p), engine.load(i), engine.load(w))
        paths = set()
        for ta in ("N", "T"):
            for cols in (1, 2, 8):
                B = (rng.uniform(-1, 1, (cols, n)) + (1j * rng.uniform(-1, 1, (cols, n)) if cplx else 0)).astype(ct)
                gC = torch.zeros(cols, n, dtype=torch.from_numpy(B).dtype, device="cuda")
                A.gemm(ta, "N", n, cols, 1.5, engine.load(B), n, 0.0, gC, n)
                path = engine.get_option("path_product")
                if ta == "N" or cols > 1:  # (a single real transposed product picks by rules of its own)
                    assert path == product_path(A, ct, n, n, len(i), ta, "N", cols)
                    paths.add(path)
                got = host(gC)
                for c in range(cols):
                    if ct == np.float64:
                        ref = oracle.spmv(ta, n, n, 1.5, p, i, w, B[c], 0.0, np.zeros(n))
                    elif ct == np.float32 and ta == "N":
                        ref = oracle.spmv_f32(p, i, w, B[c], alpha=1.5, beta=0.0, y=np.zeros(n, ct))
                    else:
                        z = ct if cplx else np.complex64
                        ref = np.zeros(n, z)
                        oracle.zspmv(ta, n, n, 1.5 + 0j, p, i, w.astype(z), B[c].astype(z), 0j, ref)
                        ref = ref if cplx else ref.real.astype(np.float32)
                    assert np.array_equal(raw(got[c]), raw(ref)), (ct, ta, cols, c)
        assert (1 if mat in ("27-point 41^3", "5-point 530^2", "7-point 51^3") else 2) in paths


def test_transposed_product_of_few_long_rows(engine):
    # a few workgroups of rows of several tiles: the single transposed product walks them too
    rng = np.random.default_rng(11)
    n, k = 600, 45
    i = np.concatenate([np.sort(rng.choice(n, k, replace=False)) for _ in range(n)]).astype(np.int32)
    p = np.arange(0, n * k + 1, k, dtype=np.int32)
    for ct in (np.float64, np.float32):
        v = rng.uniform(-1, 1, n * k).astype(ct)
        A = H.make_sparse_matrix(engine, n, engine.load(p), engine.load(i), engine.load(v))
        x, y = rng.uniform(-1, 1, n).astype(ct), rng.uniform(-1, 1, n).astype(ct)
        for beta in (0.0, 0.5):
            gy = engine.load(y)
            A.gemv("T", 1.5, engine.load(x), beta, gy)
            if ct == np.float64:
                assert engine.get_option("path_product") == 2
                ref = oracle.spmv("T", n, n, 1.5, p, i, v, x, beta, y.copy())
            else:
                ref = y.astype(np.complex64)
                oracle.zspmv("T", n, n, 1.5 + 0j, p, i, v.astype(np.complex64), x.astype(np.complex64), complex(beta), ref)
                ref = ref.real.astype(ct)
            assert np.array_equal(raw(host(gy)), raw(ref))


TRI = {
    "grid3": lambda: st.laplace3d(21, 9, 10),
    "grid2": lambda: st.laplace2d(30, 66),
    "column": lambda: st.convdiff27(12, seed=3),
    "pool": lambda: st.laplace2d(10, 6),
}


@pytest.mark.parametrize("name", sorted(TRI))
@pytest.mark.parametrize("uplo", ["L", "U"])
def test_trsm_many_columns(engine, name, uplo):
    p, i, v = TRI[name]()
    n = len(p) - 1
    row = np.repeat(np.arange(n), np.diff(p))
    keep = i <= row if uplo == "L" else i >= row
    q = np.zeros(n + 1, np.int32)
    q[1:] = np.cumsum(np.bincount(row[keep], minlength=n))
    i, v = i[keep].copy(), v[keep] * np.linspace(0.2, 0.3, keep.sum())
    T = H.make_triangular_matrix(engine, uplo, "N", engine.load(q), engine.load(i), engine.load(v))
    T32 = H.make_triangular_matrix(engine, uplo, "N", T.pntr, T.indx, T.vals.float())
    Tz = H.make_triangular_matrix(engine, uplo, "N", T.pntr, T.indx, engine.load(v * (1 + 0.25j)))
    saved = engine.get_option("tri_grid"), engine.get_option("tri_col")
    try:
        if name == "pool":
            engine.set_option("tri_col", 0)
        for ta in "NT":
            for tb, nrhs, pad in (("N", 1, 0), ("N", 3, 5), ("T", 4, 2), ("N", 9, 0)):
                rng = np.random.default_rng(nrhs)
                shape = (nrhs, n + pad) if tb == "N" else (n, nrhs + pad)
                B = rng.uniform(-1, 1, shape)
                for M, w in ((T, np.float64), (T32, np.float32), (Tz, np.complex128)):
                    g = engine.load(B.astype(w))
                    M.trsm(ta, tb, nrhs, 1.5, g, shape[1])
                    got = host(g)
                    assert np.array_equal(raw(got[:, shape[1] - pad:]), raw(B.astype(w)[:, shape[1] - pad:]))
                    for c in range(nrhs):
                        b = np.ascontiguousarray((B[c, :n] if tb == "N" else B[:, c]).astype(w))
                        ref = {np.float64: lambda: oracle.trsv(uplo, ta, "N", 1.5, q, i, v, b),
                               np.float32: lambda: oracle.trsv_f32(uplo, ta, "N", 1.5, q, i, v.astype(w), b),
                               np.complex128: lambda: oracle.ztrsv(uplo, ta, "N", 1.5, q, i, v * (1 + 0.25j), b)}[w]()
                        col = got[c, :n] if tb == "N" else got[:, c]
                        assert np.array_equal(raw(col), raw(ref)), (name, ta, tb, nrhs, w, c)
    finally:
        engine.set_option("tri_grid", saved[0])
        engine.set_option("tri_col", saved[1])


@pytest.mark.parametrize("name", ["grid", "columns"])
@pytest.mark.parametrize("mib", [0, 1, 2])
def test_strips_of_vectors(engine, name, mib):
    # more vectors than a packed copy may hold go in strips, with a remainder, down to one by one: same bits
    p, i, v = st.laplace3d(40, 24, 25)
    n = len(p) - 1
    row = np.repeat(np.arange(n), np.diff(p))
    keep = i <= row
    q = np.zeros(n + 1, np.int32)
    q[1:] = np.cumsum(np.bincount(row[keep], minlength=n))
    li, lv = i[keep].copy(), v[keep].copy()
    gp, gi, gv = engine.load(p), engine.load(i), engine.load(v)
    saved = engine.get_option("tri_grid"), engine.get_option("rhs_mib")
    try:
        engine.set_option("tri_grid", 1 if name == "grid" else 0)
        engine.set_option("rhs_mib", mib)
        T = H.make_triangular_matrix(engine, "L", "N", engine.load(q), engine.load(li), engine.load(lv))
        B = np.stack([st.uniform(70 + k, n) for k in range(11)])
        g = engine.load(B)
        T.trsm("N", "N", 11, 1.5, g)
        for k in range(11):
            assert np.array_equal(bits(host(g[k])), bits(oracle.trsv("L", "N", "N", 1.5, q, li, lv, B[k])))
        M = H.make_ilu(engine, gp, gi, gv)
        X = torch.zeros(11, n, dtype=torch.float64, device="cuda")
        H.solve_batch_cg_ilu(engine, H.stop_criteria(0.0, 4), gp, gi, gv, M, engine.load(B), X)
        assert engine.get_option("path_pcg") == 0  # not fused: the solve's vectors exceed a strip
        dg, _ = oracle.diag(p, i)
        f = oracle.ilu0(p, i, v, dg)
        for k in (0, 4, 10):
            _, x, _ = oracle.cg(p, i, v, B[k], tol=0.0, max_iter=4, prec=oracle.PREC_ILU, mpntr=p, mindx=i, mdiag=dg, mdata=f)
            assert np.array_equal(bits(host(X[k])), bits(x)), k
    finally:
        engine.set_option("tri_grid", saved[0])
        engine.set_option("rhs_mib", saved[1])


@pytest.mark.parametrize("name", ["grid3", "column"])
@pytest.mark.parametrize("nrhs", [1, 2, 3, 5, 8, 9])
def test_multirhs_pcg_grid_and_columns(engine, name, nrhs):
    p, i, v = TRI["grid3"]()
    n = len(p) - 1
    gp, gi, gv = engine.load(p), engine.load(i), engine.load(v)
    saved = engine.get_option("tri_grid")
    try:
        engine.set_option("tri_grid", 1 if name == "grid3" else 0)
        M = H.make_ilu(engine, gp, gi, gv)
        B = np.stack([st.uniform(40 + k, n) for k in range(nrhs)])
        tol = 1e-9 * max(oracle.cnrm2(b) for b in B)
        X = torch.zeros(nrhs, n, dtype=torch.float64, device="cuda")
        it = H.solve_batch_cg_ilu(engine, tol, gp, gi, gv, M, engine.load(B), X)
        dg, _ = oracle.diag(p, i)
        f = oracle.ilu0(p, i, v, dg)
        for k in range(nrhs):  # each column is the single solve stopped after the same number of passes
            _, x, _ = oracle.cg(p, i, v, B[k], tol=0.0, max_iter=it, prec=oracle.PREC_ILU, mpntr=p, mindx=i, mdiag=dg,
                                mdata=f)
            assert np.array_equal(bits(host(X[k])), bits(x)), k
    finally:
        engine.set_option("tri_grid", saved)


def spd(n, extra, full_row, seed):
    """Symmetric, diagonally dominant: `extra` random couplings per row, with full_row one row coupled to all."""
    rng = np.random.default_rng(seed)
    a, b = rng.integers(0, n, n * extra // 2), rng.integers(0, n, n * extra // 2)
    if full_row:
        a, b = np.concatenate([a, np.full(n, n // 3)]), np.concatenate([b, np.arange(n)])
    d = np.arange(n, dtype=np.int64)
    key = np.unique(np.concatenate([a * np.int64(n) + b, b * np.int64(n) + a, d * n + d]))
    row, col = key // n, (key % n).astype(np.int32)
    p = np.zeros(n + 1, np.int32)
    p[1:] = np.cumsum(np.bincount(row, minlength=n))
    v = np.where(row == col, 2.0 * np.diff(p)[row], -1.0 / (1 + (row + col) % 5))
    return p, col, v


MULTI = {  # name: (matrix, path of the product of several columns, of one column)
    "grid": (lambda: st.laplace3d(17, 18, 19), 1, 1),
    "a long row": (lambda: spd(3000, 3, True, 5), 2, 0),
    "few workgroups of long rows": (lambda: spd(700, 30, False, 6), 2, 2),
    "random, groups of four": (lambda: spd(70000, 4, False, 7), 1, 1),
    "random, pairs": (lambda: spd(270000, 4, False, 8), 1, 1),
}


@pytest.mark.parametrize("name", sorted(MULTI))
def test_multirhs_cg_products(engine, name):
    mat, path, path1 = MULTI[name]
    p, i, v = mat()
    n = len(p) - 1
    gp, gi, gv = engine.load(p), engine.load(i), engine.load(v)
    A = H.make_sparse_matrix(engine, n, gp, gi, gv)
    passes = 5
    for nrhs in (1, 2, 3, 5, 8, 9):
        B = np.stack([st.uniform(60 + k, n) for k in range(nrhs)])
        X = torch.zeros(nrhs, n, dtype=torch.float64, device="cuda")
        it = H.solve_batch_cg(engine, H.stop_criteria(0.0, passes), gp, gi, gv, None, engine.load(B), X, matrix=A)
        # of the last group: nine columns leave one over a group of eight, four or two, three one over two
        last = nrhs == 1 or nrhs == 9 or (name.endswith("pairs") and nrhs in (3, 5)) or (name.endswith("four") and nrhs == 5)
        assert engine.get_option("path_product") == (path1 if last else path)
        assert it == passes
        for k in sorted({0, nrhs // 2, nrhs - 1}):
            _, x, _ = oracle.cg(p, i, v, B[k], tol=0.0, max_iter=passes)
            assert np.array_equal(bits(host(X[k])), bits(x)), (nrhs, k)


def test_large_strips_are_given_back():
    # the packed copies of many right-hand sides go back at the end of the call once they pass a gibibyte
    eng = H.gpu_engine(0)
    p, i, v = st.laplace3d(96, 96, 96)
    n = len(p) - 1
    row = np.repeat(np.arange(n), np.diff(p))
    keep = i <= row
    q = np.zeros(n + 1, np.int32)
    q[1:] = np.cumsum(np.bincount(row[keep], minlength=n))
    T = H.make_triangular_matrix(eng, "L", "N", eng.load(q), eng.load(i[keep].copy()), eng.load(v[keep].copy()))
    B = torch.rand(100, n, dtype=torch.float64, device="cuda")
    for k, most in ((4, 100), (100, 0)):  # MiB that stay: a few vectors' buffers, then none of the large ones
        T.trsm("N", "N", 1, 1.0, B)
        held = eng.get_option("held_mib")
        T.trsm("N", "N", k, 1.0, B)
        assert eng.get_option("held_mib") - held <= most, k
