"""ILU applied by Jacobi sweeps over columns of 256 rows: bit for bit the
oracle's at the edges of a block of rows and of the seven entries loaded at
once, and on rows too unequal for the columns (packed rows as before)."""
import numpy as np
import pytest

import hala_amd as H
import oracle
from hala_amd import stencils as st
from tests.conftest import bits

pytestmark = pytest.mark.gpu


def band(n, half, keep, seed):
    """Symmetric pattern of the given half width; off the diagonal a row keeps all, or one in `keep` holds any."""
    rng = np.random.default_rng(seed)
    r, c = np.meshgrid(np.arange(n), np.arange(-half, half + 1), indexing="ij")
    col = (r + c).ravel()
    row = r.ravel()
    ok = (col >= 0) & (col < n) & ((row == col) | (np.minimum(row, col) % keep == 0))
    row, col = row[ok], col[ok]
    p = np.zeros(n + 1, np.int32)
    p[1:] = np.cumsum(np.bincount(row, minlength=n))
    return p, col.astype(np.int32), np.where(row == col, 2.0 * half + 1.0, rng.uniform(-1.0, -0.2, len(row)))


@pytest.mark.parametrize("prec", ["f32", "f64"])
@pytest.mark.parametrize("n,half,keep", [(1, 1, 1), (255, 4, 1), (256, 5, 1), (256, 6, 1), (257, 7, 1), (1000, 8, 1), (770, 13, 1),
                                         (513, 14, 1), (600, 15, 1), (700, 5, 9)])
def test_jacobi_columns_bitexact(engine, n, half, keep, prec):
    p, i, v = band(n, half, keep, n + half)
    opt = "ilu32_jacobi" if prec == "f32" else "ilu64_jacobi"
    saved = engine.get_option(opt)
    # columns for triangles of rows of five and more entries, padded by at most a quarter
    row = np.repeat(np.arange(n), np.diff(p))
    low = np.bincount(row[i < row], minlength=n)
    width, blocks = int(low.max()), (n + 255) // 256
    columns = width >= 5 and blocks * 256 * width * 4 <= int(low.sum()) * 5
    try:
        dg, _ = oracle.diag(p, i)
        f = oracle.ilu0(p, i, v, dg)
        M = H.make_ilu(engine, engine.load(p), engine.load(i), engine.load(v), want_f32=True)
        x = st.uniform(5, n)
        x[::3] = -0.0
        gr = engine.vector(n)
        for k in (1, 3):
            engine.set_option(opt, k)
            if prec == "f32":
                M.apply_f32x64(engine.load(x), gr)
                ref = oracle.ilu_apply_f32_jacobi(p, i, dg, f.astype(np.float32), x.astype(np.float32),
                                                  k).astype(np.float64)
            else:
                M.apply(engine.load(x), gr)
                ref = oracle.ilu_apply_jacobi(p, i, dg, f, x, k)
            assert np.array_equal(bits(gr.cpu().numpy()), bits(ref))
            assert (engine.get_option("path_jacobi") % 4 == 2) == columns
    finally:
        engine.set_option(opt, saved)
