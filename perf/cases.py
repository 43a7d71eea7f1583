"""Performance cases of the sparse solve path, through its public Python API.

listed() holds the fixed cases, draw() gives more of the same ranges; prepare()
makes what a program has in hand before the call (matrix, factor, right-hand
sides, all on the GPU), run() is one pass, work() the bytes and operations the
pass cannot do without, exact() the result from plain torch / numpy in 64 bits.

Kinds:
  spmv     y = alpha op(A) x + beta y (sparse_gemv)
  spmm     C = alpha op(A) B + beta C, several columns at once (sparse_gemm)
  trsm     op(T)^-1 (alpha B), several right-hand sides (sparse_trsm)
  cg       plain or ILU(0)-preconditioned CG to a relative residual
  step     a complete solve: ILU(0) analysis, factorisation, ILU-PCG
  multirhs ILU-PCG on several right-hand sides of one matrix
  gmres    restarted GMRES: FP64 with the exact ILU(0), or FP64 refinement
           around an FP32 inner solve
  batch    thousands of independent small systems, Jacobi-PCG
  adjoint  forward solve and gradient of a loss through it (torch autograd)
"""
import math

import numpy as np
import torch

import hala_amd as H
from hala_amd import stencils as st

_REAL = {"f64": torch.float64, "f32": torch.float32}
_TORCH = dict(_REAL, z=torch.complex128, c=torch.complex64)
_SIZE = {"f64": 8, "f32": 4, "z": 16, "c": 8}


def listed():
    return [
        # the product the solvers spend their bandwidth on, at the size of the headline benchmark
        {"name": "spmv_poisson3d_128", "kind": "spmv", "op": "lap3d", "m": 128, "dtype": "f64", "trans": "N",
         "beta": 0.0},
        # a transposed product on a rectangular operator of an unstructured mesh (interpolation
        # transpose, least squares), FP32, accumulating into y
        {"name": "spmv_t_ragged_f32", "kind": "spmv", "op": "ragged", "m": 400009, "dtype": "f32", "trans": "T",
         "beta": 1.0},
        # block Krylov / several load cases: 27-point operator times 16 vectors
        {"name": "spmm_convdiff27_64_x16", "kind": "spmm", "op": "conv27", "m": 64, "dtype": "f64", "trans": "N",
         "cols": 16, "beta": 0.0},
        # a complex (Helmholtz-like) operator times a few vectors
        {"name": "spmm_complex2d_701_x5", "kind": "spmm", "op": "lap2d", "m": 701, "dtype": "z", "trans": "N",
         "cols": 5, "beta": 0.0},
        # a triangular preconditioner (symmetric Gauss-Seidel, a given Cholesky factor) on 8 vectors
        {"name": "trsm_lower3d_64_x8", "kind": "trsm", "op": "lap3d", "m": 64, "dtype": "f64", "uplo": "L",
         "trans": "N", "cols": 8},
        # the smallest solves: plain CG on a small 2D grid, where launches and latency count
        {"name": "cg_poisson2d_64", "kind": "cg", "op": "lap2d", "m": 64, "prec": "none"},
        # the reference's GPU example (ILU(0)-PCG, 2D Poisson) with the factor kept, odd side
        {"name": "pcg_poisson2d_127", "kind": "cg", "op": "lap2d", "m": 127, "prec": "ilu"},
        # the headline benchmark: analysis + factorisation + ILU(0)-PCG, 128^3
        {"name": "step_poisson3d_128", "kind": "step", "op": "lap3d", "m": 128},
        # one matrix, 8 load cases
        {"name": "multirhs_poisson3d_64_x8", "kind": "multirhs", "op": "lap3d", "m": 64, "cols": 8},
        # the mixed-precision benchmark: nonsymmetric 27-point operator, FP32 inner GMRES(30) with the
        # Jacobi-applied ILU(0), FP64 refinement
        {"name": "gmres_mixed_convdiff27_96", "kind": "gmres", "m": 96, "inner": "f32"},
        # the batched benchmark: 4096 independent systems of 14^2 .. 70^2 unknowns
        {"name": "batch_pcg_4096", "kind": "batch", "systems": 4096, "side_hi": 70},
        # the differentiable-solve benchmark: forward, adjoint and coefficient gradient
        {"name": "adjoint_diffusion3d_64", "kind": "adjoint", "m": 64},
    ]


def _logint(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


_GRID = {"lap2d": (24, 1024), "lap3d": (10, 128), "conv27": (8, 72)}


def draw(rng):
    kind = rng.choice(["spmv", "spmm", "trsm", "cg", "step", "multirhs", "gmres", "batch", "adjoint"])
    if kind in ("spmv", "spmm"):
        op = rng.choice(["lap2d", "lap3d", "conv27", "ragged"])
        c = {"kind": kind, "op": op, "m": _logint(rng, 2000, 400000) if op == "ragged" else _logint(rng, *_GRID[op]),
             "dtype": rng.choice(["f64", "f64", "f32"] if kind == "spmv" else ["f64", "f64", "f32", "z", "c"]),
             "trans": rng.choice(["N", "N", "T"]), "beta": rng.choice([0.0, 1.0])}
        if kind == "spmm":
            c["cols"] = rng.randint(2, 24)
            c["m"] = c["m"] if op == "ragged" else max(8, c["m"] // 2)
        return c
    if kind == "trsm":
        op = rng.choice(["lap2d", "lap3d", "conv27"])
        return {"kind": kind, "op": op, "m": _logint(rng, *{"lap2d": (24, 400), "lap3d": (8, 64),
                                                            "conv27": (8, 40)}[op]),
                "dtype": rng.choice(["f64", "f64", "f32"]), "uplo": rng.choice(["L", "U"]),
                "trans": rng.choice(["N", "N", "T"]), "cols": rng.randint(1, 16)}
    if kind == "cg":
        op = rng.choice(["lap2d", "lap3d"])
        return {"kind": kind, "op": op, "m": _logint(rng, *{"lap2d": (16, 260), "lap3d": (8, 72)}[op]),
                "prec": rng.choice(["none", "jacobi", "ilu", "ilu"])}
    if kind == "step":
        op = rng.choice(["lap2d", "lap3d"])
        return {"kind": kind, "op": op, "m": _logint(rng, *{"lap2d": (32, 260), "lap3d": (12, 112)}[op])}
    if kind == "multirhs":
        return {"kind": kind, "op": "lap3d", "m": _logint(rng, 10, 64), "cols": rng.randint(2, 8)}
    if kind == "gmres":
        inner = rng.choice(["f64", "f32"])
        return {"kind": kind, "m": _logint(rng, 10, 48 if inner == "f64" else 88), "inner": inner}
    if kind == "batch":
        return {"kind": kind, "systems": _logint(rng, 100, 4096), "side_hi": rng.randint(20, 70)}
    return {"kind": kind, "m": _logint(rng, 10, 64)}


# ---------------------------------------------------------------------------
# inputs (host arrays, from the seed)
# ---------------------------------------------------------------------------
def _ragged(nr, rng):
    """Rows of 0 to about 60 entries (12 on average) around the diagonal of a rectangular matrix."""
    nc = nr * 4 // 5 + 7
    length = np.minimum(rng.geometric(1.0 / 12.0, nr) - (rng.random(nr) < 0.05) * 60, 60).clip(0)
    row = np.repeat(np.arange(nr, dtype=np.int64), length)
    col = row * nc // nr + (rng.laplace(0.0, 0.01 * nc, row.size)).astype(np.int64)
    col = np.abs(col)  # reflected at both ends
    col = np.minimum(col, 2 * (nc - 1) - col).clip(0)
    key = np.unique(row * nc + col)
    row, col = key // nc, key % nc
    p = np.zeros(nr + 1, np.int32)
    p[1:] = np.cumsum(np.bincount(row, minlength=nr))
    return p, col.astype(np.int32), rng.standard_normal(col.size), nc


def _matrix(case, seed):
    """(pntr, indx, vals, ncols); vals float64 or complex128."""
    rng = np.random.default_rng([seed, 1])
    op, m = case.get("op", "conv27"), case.get("m")
    if op == "ragged":
        p, i, v, nc = _ragged(m, rng)
    else:
        if op == "lap2d":
            p, i, v = st.laplace2d(m, m)
        elif op == "lap3d":
            p, i, v = st.laplace3d(m, m, m)
        else:
            p, i, v = st.convdiff27(m, seed=seed % 1000)
        nc = len(p) - 1
    if case["kind"] in ("spmv", "spmm"):  # products: values of an assembled operator, not of one stencil
        v = v * rng.uniform(0.5, 1.5, v.size)
    if case.get("dtype") in ("z", "c"):
        v = v + 1j * rng.uniform(-0.2, 0.2, v.size)
    return p, i, v, nc


def _vectors(seed, rows, cols, dtype):
    """cols vectors of rows entries, U[-1, 1], as a (cols, rows) tensor (column-major for the library)."""
    rng = np.random.default_rng([seed, 2])
    a = rng.uniform(-1.0, 1.0, (cols, rows))
    if dtype in ("z", "c"):
        a = a + 1j * rng.uniform(-1.0, 1.0, (cols, rows))
    return torch.from_numpy(a).to(_TORCH[dtype])


def _typed(v, dtype):
    return torch.from_numpy(np.ascontiguousarray(v)).to(_TORCH[dtype])


def _triangle(p, i, v, uplo):
    """One triangle with its diagonal, scaled as a well-conditioned factor has it."""
    n = len(p) - 1
    row = np.repeat(np.arange(n), np.diff(p))
    keep = i <= row if uplo == "L" else i >= row
    row, col, val = row[keep], i[keep], v[keep].copy()
    val[col == row] = np.abs(val[col == row]) + 1.0
    q = np.zeros(n + 1, np.int32)
    q[1:] = np.cumsum(np.bincount(row, minlength=n))
    return q, col.astype(np.int32), val


def _spmx_inputs(case, seed):
    p, i, v, nc = _matrix(case, seed)
    nr, cols, dt = len(p) - 1, case.get("cols", 1), case["dtype"]
    k, m = (nc, nr) if case["trans"] == "N" else (nr, nc)
    x = _vectors(seed, k, cols, dt)
    y = _vectors(seed + 1, m, cols, dt) if case["beta"] else torch.zeros(cols, m, dtype=_TORCH[dt])
    return p, i, _typed(v, dt), nc, k, m, x, y


def _trsm_inputs(case, seed):
    p, i, v, _ = _matrix(case, seed)
    p, i, v = _triangle(p, i, v, case["uplo"])
    return p, i, _typed(v, case["dtype"]), _vectors(seed, len(p) - 1, case["cols"], case["dtype"])


# ---------------------------------------------------------------------------
# prepare / run
# ---------------------------------------------------------------------------
def prepare(case, seed):
    eng = H.gpu_engine(0)
    kind = case["kind"]
    s = {"case": case, "eng": eng}
    if kind in ("spmv", "spmm"):
        p, i, v, nc, k, m, x, y = _spmx_inputs(case, seed)
        v = v.cuda()
        s.update(A=H.make_sparse_matrix(eng, nc, eng.load(p), eng.load(i), v), k=k, m=m, x=x.cuda(), y0=y.cuda())
        s["y"] = s["y0"].clone()
        if case["trans"] != "N":  # the transposed pattern is built with the first transposed product and kept
            s["A"].gemm("T", "N", k, 1, 1.0, s["x"], k, 0.0, torch.empty_like(s["y"]), m)
    elif kind == "trsm":
        p, i, v, b = _trsm_inputs(case, seed)
        s.update(T=H.make_triangular_matrix(eng, case["uplo"], "N", eng.load(p), eng.load(i), v.cuda()), b=b.cuda())
        s["x"] = torch.empty_like(s["b"])
    elif kind in ("cg", "step", "multirhs"):
        p, i, v, nc = _matrix(case, seed)
        b = _vectors(seed, nc, case.get("cols", 1), "f64")
        s.update(p=eng.load(p), i=eng.load(i), v=eng.load(v), b=b.cuda(), prec=None)
        s["stop"] = H.stop_criteria(1e-10 * float(b.norm(dim=1).max()))
        s["x"] = torch.empty_like(s["b"])
        s["A"] = H.make_sparse_matrix(eng, nc, s["p"], s["i"], s["v"])
        if kind == "multirhs" or case.get("prec") == "ilu":
            s["prec"] = H.make_ilu(eng, s["p"], s["i"], s["v"])
        elif case.get("prec") == "jacobi":
            row = np.repeat(np.arange(nc), np.diff(p))
            s["prec"] = ("jacobi", eng.load(v[row == i]))
    elif kind == "gmres":
        p, i, v, nc = _matrix(case, seed)
        b = _vectors(seed, nc, 1, "f64")
        mixed = case["inner"] == "f32"
        s.update(p=eng.load(p), i=eng.load(i), v=eng.load(v), b=b[0].cuda())
        s["v32"] = s["v"].float()
        s["A"] = H.make_sparse_matrix(eng, nc, s["p"], s["i"], s["v"])
        s["prec"] = H.make_ilu(eng, s["p"], s["i"], s["v"], want_f32=mixed)
        s["x"] = torch.empty_like(s["b"])
        if mixed:
            eng.set_option("ilu32_jacobi", 3)
        else:  # HALA stops on the preconditioned estimate
            r = torch.empty_like(s["b"])
            s["prec"].apply(s["b"], r)
            s["stop"] = H.stop_criteria(1e-12 * float(r.norm()))
    elif kind == "batch":
        d = _batch_inputs(case, seed)
        s.update({k: eng.load(d[k]) for k in ("row_off", "pntr", "indx", "vals", "dvals")})
        s["b"] = _vectors(seed, len(d["dvals"]), 1, "f64")[0].cuda()
        s["x"] = torch.empty_like(s["b"])
        s["it"] = torch.zeros(case["systems"], dtype=torch.int32, device="cuda")
        s["solver"] = H.batch_solver(eng, s["row_off"], s["pntr"], s["indx"])
        s["solver"].set_shape(512, 2)  # what the tuner settles on for these sizes
    else:
        from hala_amd.autograd import SparseLinearProblem

        d, f, kappa, w = _adjoint_inputs(case, seed)
        s["problem"] = SparseLinearProblem(eng, d["pntr"], d["indx"], d["cptr"], d["cnnz"], d["ccoef"], f, rtol=1e-10)
        s["kappa"], s["w"] = eng.load(kappa), eng.load(w)
    torch.cuda.synchronize()
    return s


def _batch_inputs(case, seed):
    """The systems' sizes are the case's own; every system's values are scaled by the seed."""
    d = st.batch_laplace(case["systems"], seed=4, side_lo=14, side_hi=case["side_hi"])
    scale = np.random.default_rng([seed, 4]).uniform(0.5, 2.0, case["systems"])
    rows = np.repeat(scale, np.diff(d["row_off"]))
    d["vals"] *= np.repeat(rows, np.diff(d["pntr"]))
    d["dvals"] *= rows
    return d


def _adjoint_inputs(case, seed):
    d = st.diffusion3d(case["m"], seed=seed % 1000)
    rng = np.random.default_rng([seed, 3])
    n = len(d["pntr"]) - 1
    return d, st.gaussian_source(case["m"]) + 0.1 * rng.uniform(-1, 1, n), d["kappa"], rng.uniform(-1, 1, n)


def run(s):
    case, kind, eng = s["case"], s["case"]["kind"], s["eng"]
    if kind == "spmv":
        y = s["y"]
        if case["beta"]:
            y.copy_(s["y0"])
        s["A"].gemv(case["trans"], 1.0, s["x"][0], case["beta"], y[0])
        return y
    if kind == "spmm":
        y = s["y"]
        if case["beta"]:
            y.copy_(s["y0"])
        s["A"].gemm(case["trans"], "N", s["k"], case["cols"], 1.0, s["x"], s["k"], case["beta"], y, s["m"])
        return y
    if kind == "trsm":
        s["x"].copy_(s["b"])
        return s["T"].trsm(case["trans"], "N", case["cols"], 1.0, s["x"])
    if kind == "cg":
        s["x"].zero_()
        it = H.solve_cg(eng, s["stop"], s["p"], s["i"], s["v"], s["prec"], s["b"][0], s["x"][0], matrix=s["A"])
        return s["x"], it
    if kind == "step":
        s["x"].zero_()
        s["prec"] = None  # the previous step's factor is released first
        s["prec"] = H.make_ilu(eng, s["p"], s["i"], s["v"])
        it = H.solve_cg_ilu(eng, s["stop"], s["p"], s["i"], s["v"], s["prec"], s["b"][0], s["x"][0], matrix=s["A"])
        return s["x"], it
    if kind == "multirhs":
        s["x"].zero_()
        it = H.solve_batch_cg_ilu(eng, s["stop"], s["p"], s["i"], s["v"], s["prec"], s["b"], s["x"], matrix=s["A"])
        return s["x"], it
    if kind == "gmres":
        s["x"].zero_()
        if case["inner"] == "f32":
            tot, _ = H.solve_gmres_ir(eng, s["A"], s["v"], s["v32"], s["prec"], s["b"], s["x"], rtol=1e-10,
                                      inner_rtol=1e-4, restart=30, max_refine=40)
        else:
            tot, _ = H.solve_gmres_ilu(eng, s["stop"], 30, s["p"], s["i"], s["v"], s["prec"], s["b"], s["x"],
                                       matrix=s["A"])
        return s["x"], tot
    if kind == "batch":
        s["x"].zero_()
        s["solver"].solve(s["vals"], s["dvals"], s["b"], s["x"], rtol=1e-10, iters=s["it"])
        return s["x"], s["it"]
    from hala_amd.autograd import sparse_solve

    kappa = s["kappa"].detach().requires_grad_(True)
    x = sparse_solve(kappa, s["problem"])
    (x * s["w"]).sum().backward()
    return x.detach(), kappa.grad


# ---------------------------------------------------------------------------
# work: every input read once, every output written once, per iteration where the method iterates
# ---------------------------------------------------------------------------
def _counts(case):
    """(rows, nonzeros) of the case's operator, from its dimensions."""
    op, m = case.get("op", "conv27"), case["m"]
    if op == "lap2d":
        return m * m, 5 * m * m - 4 * m
    if op == "lap3d":
        return m ** 3, 7 * m ** 3 - 6 * m * m
    if op == "conv27":
        return m ** 3, (3 * m - 2) ** 3
    return m, 11.4 * m


def work(case):
    kind = case["kind"]
    if kind == "batch":
        side2 = (14 * 14 + 14 * case["side_hi"] + case["side_hi"] ** 2) / 3.0  # mean of side^2
        n = case["systems"] * side2
        it = 0.7 * case["side_hi"]  # measured mean iterations at 70: 49
        # a system fits on chip: matrix, diagonal, b read once, x written once
        return {"bytes": n * (4.9 * 12 + 4 + 24), "flops": it * n * (2 * 4.9 + 13)}
    if kind == "adjoint":
        n, z = case["m"] ** 3, 7 * case["m"] ** 3
        it = 2 * 1.9 * case["m"]  # forward and adjoint iterations (measured at 64: 122 each)
        return {"bytes": it * _pcg_bytes(n, z, True, 1), "flops": it * (4 * z + 12 * n)}
    n, z = _counts(case)
    cols = case.get("cols", 1)
    if kind in ("spmv", "spmm"):
        sz = _SIZE[case["dtype"]]
        mul = 8 if case["dtype"] in ("z", "c") else 2
        k = 1.8 * n if case["op"] == "ragged" else 2 * n
        acc = (0.8 if case["op"] == "ragged" and case["trans"] == "T" else 1.0) * n if case["beta"] else 0
        return {"bytes": z * (sz + 4) + 4 * n + cols * sz * (k + acc), "flops": mul * z * cols}
    if kind == "trsm":
        sz, zt = _SIZE[case["dtype"]], (z + n) / 2
        return {"bytes": zt * (sz + 4) + 4 * n + 2 * cols * sz * n, "flops": 2 * zt * cols}
    if kind == "gmres":
        mixed = case["inner"] == "f32"
        it = (3.4 if mixed else 2.0) * case["m"]  # measured at 96: 323 and 189 preconditioner applies
        vb = 4 if mixed else 8
        # product, one apply of the factor, and the basis read twice at the mean width of a GMRES(30) cycle
        return {"bytes": it * (2 * z * (vb + 4) + 12 * n + 2 * 15 * 8 * n + 40 * n), "flops": it * (4 * z + 62 * n)}
    ilu = kind in ("step", "multirhs") or case["prec"] == "ilu"
    if case["op"] == "lap2d":  # measured: 152 ILU and 853/256 plain iterations per unit side
        it = (1.19 if ilu else 3.33) * case["m"]
    else:
        it = (1.42 if ilu else 3.0) * case["m"]
    return {"bytes": it * _pcg_bytes(n, z, ilu, cols), "flops": it * cols * ((4 if ilu else 2) * z + 12 * n)}


def _pcg_bytes(n, z, ilu, cols):
    """One PCG pass: the matrix (and the factor) once for all columns, the fused vector work per column."""
    return (12 * z + 4 * n) * (2 if ilu else 1) + cols * n * (88 + (32 if ilu else 0))


# ---------------------------------------------------------------------------
# exact: the same result from torch and numpy in 64 bits
# ---------------------------------------------------------------------------
def _csr(p, i, v, nc, dev):
    return torch.sparse_csr_tensor(torch.from_numpy(p.astype(np.int64)), torch.from_numpy(i.astype(np.int64)), v,
                                   size=(len(p) - 1, nc)).to(dev)


def _spmx_exact(case, seed):
    p, i, v, nc, k, m, x, y = _spmx_inputs(case, seed)
    wide = torch.complex128 if case["dtype"] in ("z", "c") else torch.float64
    v, x, y = v.to(wide), x.to(wide), y.to(wide)
    row = torch.from_numpy(np.repeat(np.arange(len(p) - 1), np.diff(p)))
    col = torch.from_numpy(i.astype(np.int64))
    if case["trans"] != "N":
        row, col = col, row
    out = y * case["beta"]
    for c in range(x.shape[0]):
        out[c].index_add_(0, row, v * x[c][col])
    return out


def _trsm_exact(case, seed):
    p, i, v, b = _trsm_inputs(case, seed)
    n = len(p) - 1
    v, x = v.double().numpy(), np.ascontiguousarray(b.double().numpy().T)
    pl = p.tolist()
    lower, trans = case["uplo"] == "L", case["trans"] != "N"
    for r in range(n) if lower != trans else range(n - 1, -1, -1):
        a, e = pl[r], pl[r + 1]
        d, (a, e) = (e - 1, (a, e - 1)) if lower else (a, (a + 1, e))
        if not trans:
            x[r] = (x[r] - v[a:e] @ x[i[a:e]]) / v[d]
        else:
            x[r] /= v[d]
            x[i[a:e]] -= np.outer(v[a:e], x[r])
    return torch.from_numpy(np.ascontiguousarray(x.T))


def _cg64(A, b, dinv, passes=3, cap=4000):
    """Jacobi-CG restarted on its own residual until the 64-bit residual stalls."""
    x = torch.zeros_like(b)
    for _ in range(passes):
        r = b - A @ x
        d = torch.zeros_like(b)
        z = dinv * r
        q, rz, r0 = z.clone(), torch.dot(r, z), r.norm()
        for k in range(cap):
            aq = A @ q
            alpha = rz / torch.dot(q, aq)
            d += alpha * q
            r -= alpha * aq
            if k % 16 == 0 and r.norm() <= 1e-13 * r0:
                break
            z = dinv * r
            rz, old = torch.dot(r, z), rz
            q = z + (rz / old) * q
        x = x + d
    return x


def _bicgstab64(A, b, dinv, passes=3, cap=2000):
    x = torch.zeros_like(b)
    for _ in range(passes):
        r = b - A @ x
        rh, d, q = r.clone(), torch.zeros_like(b), r.clone()
        rho, r0 = torch.dot(rh, r), r.norm()
        for _k in range(cap):
            y = dinv * q
            w = A @ y
            alpha = rho / torch.dot(rh, w)
            s = r - alpha * w
            t = dinv * s
            u = A @ t
            omega = torch.dot(u, s) / torch.dot(u, u)
            d += alpha * y + omega * t
            r = s - omega * u
            if r.norm() <= 1e-11 * r0:
                break
            rho, old = torch.dot(rh, r), rho
            q = r + (rho / old) * (alpha / omega) * (q - omega * w)
        x = x + d
    return x


def _diag(p, i, v):
    row = np.repeat(np.arange(len(p) - 1), np.diff(p))
    return v[row == i]


def exact(case, seed):
    kind = case["kind"]
    if kind in ("spmv", "spmm"):
        return _spmx_exact(case, seed)
    if kind == "trsm":
        return _trsm_exact(case, seed)
    dev = "cuda" if torch.cuda.is_available() else "cpu"
    if kind in ("cg", "step", "multirhs", "gmres"):
        p, i, v, nc = _matrix(case, seed)
        A = _csr(p, i, torch.from_numpy(v), nc, dev)
        dinv = torch.from_numpy(1.0 / _diag(p, i, v)).to(dev)
        b = _vectors(seed, nc, case.get("cols", 1), "f64").to(dev)
        if kind == "gmres":
            return _bicgstab64(A, b[0], dinv), None
        return torch.stack([_cg64(A, c, dinv) for c in b]), None
    if kind == "batch":
        d = _batch_inputs(case, seed)
        ro = d["row_off"]
        n = int(ro[-1])
        base = np.repeat(ro[:-1], np.diff(ro))  # columns are local to their system
        cols = d["indx"] + np.repeat(base, np.diff(d["pntr"]))
        A = _csr(d["pntr"], cols, torch.from_numpy(d["vals"]), n, dev)
        b = _vectors(seed, n, 1, "f64")[0].to(dev)
        return _cg64(A, b, torch.from_numpy(1.0 / d["dvals"]).to(dev)), None
    d, f, kappa, w = _adjoint_inputs(case, seed)
    p, i = d["pntr"], d["indx"]
    vals = np.zeros(len(i))
    coef = np.repeat(np.arange(len(kappa)), np.diff(d["cptr"]))
    np.add.at(vals, d["cnnz"], d["ccoef"] * kappa[coef])
    n = len(p) - 1
    A = _csr(p, i, torch.from_numpy(vals), n, dev)
    dinv = torch.from_numpy(1.0 / _diag(p, i, vals)).to(dev)
    x = _cg64(A, torch.from_numpy(f).to(dev), dinv).cpu()
    lam = _cg64(A, torch.from_numpy(w).to(dev), dinv).cpu()  # the operator is symmetric
    row = torch.from_numpy(np.repeat(np.arange(n), np.diff(p)))
    gv = -lam[row] * x[torch.from_numpy(i.astype(np.int64))]
    g = torch.zeros(len(kappa), dtype=torch.float64)
    g.index_add_(0, torch.from_numpy(coef), torch.from_numpy(d["ccoef"]) * gv[torch.from_numpy(d["cnnz"]).long()])
    return x, g
