"""Batched PCG with the systems held in registers: solutions and iteration
counts bit for bit the oracle's for every team size, at the edges of the rows
per thread (one row, a full and a just started last round, the two register
classes and the step to the general loop), rows of up to 5, 7 and 9 entries,
ragged rows, a start that is not zero and an iteration cap."""
import numpy as np
import pytest
import torch

import hala_amd as H
import oracle
from tests.conftest import bits

pytestmark = pytest.mark.gpu


def banded(n, longest, rng):
    """Symmetric, diagonally dominant, rows of 1 .. longest entries at a few offsets."""
    offs = [1, max(2, int(n ** 0.5)), max(3, n // 2), max(4, n // 3)][: (longest - 1) // 2]
    row, col = [np.arange(n)], [np.arange(n)]
    for o in offs:
        a = np.nonzero(rng.random(max(n - o, 0)) < 0.9)[0]
        row += [a, a + o]
        col += [a + o, a]
    row, col = np.concatenate(row), np.concatenate(col)
    key = np.unique(row * n + col)
    row, col = key // n, key % n
    v = np.where(row == col, longest + 0.25 * (row % 5), -0.5 - 0.125 * ((row + col) % 4))
    p = np.zeros(n + 1, np.int64)
    p[1:] = np.cumsum(np.bincount(row, minlength=n))
    return p, col, v


def sizes_of(team, longest):
    rounds = {64: (4, 10), 128: (4, 10), 256: (4, 10), 512: (4, 10), 1024: (3, 3)}[team] if longest <= 5 else (3, 8)
    s = [1, 2, 63, 65, team - 1, team, team + 1, rounds[0] * team - 5, rounds[0] * team, rounds[0] * team + 1,
         rounds[1] * team]
    return s


@pytest.mark.parametrize("longest,past", [(5, False), (5, True), (7, False), (9, False)])
@pytest.mark.parametrize("team", [64, 128, 256, 512, 1024])
def test_batch_resident_bitexact(engine, team, longest, past):
    rng = np.random.default_rng(team + longest)
    sizes = [min(n, 6000) for n in sizes_of(team, longest)] + ([min(sizes_of(team, longest)[-1] + 1, 6000)] if past else [])
    sizes = [int(n) for n in rng.permutation(sizes)]
    systems = [banded(n, longest, rng) for n in sizes]
    ro = np.concatenate([[0], np.cumsum(sizes)])
    nz = np.concatenate([[0], np.cumsum([len(s[1]) for s in systems])])
    p = np.concatenate([s[0][:-1] + z for s, z in zip(systems, nz)] + [nz[-1:]])
    i, v = np.concatenate([s[1] for s in systems]), np.concatenate([s[2] for s in systems])
    d = rng.uniform(2.0, 9.0, ro[-1])
    b, x0 = rng.uniform(-1, 1, ro[-1]), rng.uniform(-1, 1, ro[-1])
    i32 = lambda a: engine.load(np.ascontiguousarray(a, np.int32))
    bs = H.batch_solver(engine, i32(ro), i32(p), i32(i))
    bs.set_shape(team, 1)
    gv, gd, gb = engine.load(v), engine.load(d), engine.load(b)
    # which kernels: resident, by rows per thread, where every system and row fits; else the general loop
    small, large = ((4, 10) if team < 1024 else (3, 3)) if longest <= 5 else ((3, 8) if team < 1024 else (0, 0))
    if longest > 7 or max(sizes) > large * team:
        want = 1
    else:
        want = (4 if max(sizes) > small * team else 0) + (2 if min(sizes) <= small * team else 0)
    for rtol, cap in ((1e-9, 100000), (1e-30, 6)):
        gx = engine.load(x0)
        iters = torch.zeros(len(sizes), dtype=torch.int32, device="cuda")
        bs.solve(gv, gd, gb, gx, rtol=rtol, max_iter=cap, iters=iters)
        assert engine.get_option("path_batch") == want
        for s, (sp, si, sv) in enumerate(systems):
            r = slice(ro[s], ro[s + 1])
            tol = rtol * np.sqrt(oracle.team_dot(b[r], b[r], team))
            it, x, _ = oracle.cg_team(sp, si, sv, d[r], b[r], tol, team, x0=x0[r], max_iter=cap)
            assert int(iters[s]) == it, (s, sizes[s])
            assert np.array_equal(bits(gx[r].cpu().numpy()), bits(x)), (s, sizes[s])


@pytest.mark.parametrize("team,wg,n,path", [(512, 4, 204, 1), (512, 4, 205, 2), (512, 2, 60, 2), (1024, 2, 1023, 1),
                                            (1024, 2, 1024, 2), (1024, 1, 40, 2), (256, 8, 20, 2)])
def test_batch_crowded_shapes(engine, team, wg, n, path):
    # more wavefronts per CU than the resident kernels' registers hold, on systems small for the team: the loop
    rng = np.random.default_rng(team + n)
    systems = [banded(n, 5, rng) for _ in range(3)]
    nz = np.concatenate([[0], np.cumsum([len(s[1]) for s in systems])])
    p = np.concatenate([s[0][:-1] + z for s, z in zip(systems, nz)] + [nz[-1:]])
    i, v = np.concatenate([s[1] for s in systems]), np.concatenate([s[2] for s in systems])
    d, b = rng.uniform(2.0, 9.0, 3 * n), rng.uniform(-1, 1, 3 * n)
    i32 = lambda a: engine.load(np.ascontiguousarray(a, np.int32))
    bs = H.batch_solver(engine, i32(np.arange(4) * n), i32(p), i32(i))
    bs.set_shape(team, wg)
    gx, iters = engine.vector(3 * n), torch.zeros(3, dtype=torch.int32, device="cuda")
    bs.solve(engine.load(v), engine.load(d), engine.load(b), gx, rtol=1e-9, max_iter=100000, iters=iters)
    assert engine.get_option("path_batch") == path
    for s, (sp, si, sv) in enumerate(systems):
        r = slice(s * n, (s + 1) * n)
        tol = 1e-9 * np.sqrt(oracle.team_dot(b[r], b[r], team))
        it, x, _ = oracle.cg_team(sp, si, sv, d[r], b[r], tol, team)
        assert int(iters[s]) == it
        assert np.array_equal(bits(gx[r].cpu().numpy()), bits(x))
