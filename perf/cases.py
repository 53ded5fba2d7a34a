"""The work that users of this library have it do, as cases that can be timed and checked.

Users drive the eigensolver in three ways, and the cases follow them: through the slots of the
operation table (a driver of their own, or the reference's, over OPS_HIP_Set), through one call per
problem (solver.solve, gcge_eps_solve), and through the solve service.  Sizes are those of the
problems in gcge_amd.problems: 2D 5-point grids of 2 K to 65 K rows with blocks of a few columns, 3D
7-point grids up to 128^3, 27-point variable-coefficient grids up to 160^3, and the block sizes of
slepc_block_policy.

A case is a dict with "kind" and the sizes of that kind:

product  MatDotMultiVec and MultiVecInnerProd 'D': w = A p and p . w over k columns, the product of a
         driver's own BlockPCG and of its residual checks (op "diff2d", "lap3d", "diff27")
project  MultiVecQtAP: V^T A W and A W for m columns of V and k of W, the projection of Rayleigh-Ritz
ritz     MultiVecLinearComb: X = V C, m columns into k, the Ritz vectors
block    the B-orthonormalization of a new k-column block against m columns: MultiVecAxpby,
         MultiVecQtAP, MultiVecLinearComb and HIP_MultiVecCholQR, as the block method runs them
columns  the same block orthonormalized column by column (the reference's OrthSelf): MultiVecQtAP,
         MultiVecAxpby and MultiVecLinearComb with one column against the rest
pcg      the single-precision BlockPCG of the MultiLinearSolver slot on k columns
solve    solver.solve in mixed precision, 3D 7-point problem, matrices on the device; the whole
         solves return eigenvalues (eigenvectors of a multiple eigenvalue are any basis)
eps      gcge_eps_solve in double precision, 2D 5-point problem, from host CCS arrays
serve    a batch of 2D variable-coefficient problems through the solve service
"""
import ctypes as C
import math

import numpy as np
import torch

from gcge_amd import abi, problems, solver
from gcge_amd.service import Service

F64 = torch.float64


# ------------------------------------------------------------------ cases
def listed():
    return [
        # served requests' products: a small general matrix and a narrow block, where a call is
        # its launches and the way back to the host
        {"name": "product_2d_17k_x12", "kind": "product", "op": "diff2d", "n": 130, "k": 12},
        # the largest general sparse product: 27 points, 4.1 M rows, the SLEPc block of nev = 200
        {"name": "product_27pt_4.1M_x40", "kind": "product", "op": "diff27", "n": 160, "k": 40},
        # served requests' projections: small Gram with its result on the host
        {"name": "project_2d_17k_60x12", "kind": "project", "op": "diff2d", "n": 130, "m": 60,
         "k": 12},
        # the headline problem's projection: 128^3, 340 + 120 columns against the new 120
        {"name": "project_7pt_2.1M_460x120", "kind": "project", "op": "lap3d", "n": 128, "m": 460,
         "k": 120},
        # Ritz vectors on an odd grid (odd leading dimension), SLEPc block sizes of nev = 150
        {"name": "ritz_1.03M_300x141", "kind": "ritz", "n": 101, "m": 300, "k": 141},
        # a new 40-column block against 200 columns at 128^3 (block Cholesky QR)
        {"name": "block_2.1M_200+40", "kind": "block", "n": 128, "m": 200, "k": 40},
        # a 40-column block column by column at 80^3, as the reference's driver does it
        {"name": "columns_512k_40", "kind": "columns", "n": 80, "k": 40},
        # the inner solves of the headline problem: matrix-free, 120 columns
        {"name": "pcg_7pt_2.1M_x120", "kind": "pcg", "op": "lap3d", "n": 128, "k": 120},
        # the inner solves of the 27-point problem: general matrix, 40 columns
        {"name": "pcg_27pt_4.1M_x40", "kind": "pcg", "op": "diff27", "n": 160, "k": 40},
        # a whole mixed-precision solve of a served size
        {"name": "solve_3d_48_nev50", "kind": "solve", "n": 48, "nev": 50},
        # a whole double-precision solve from host arrays: 2D 128 x 128, nev = 20
        {"name": "eps_2d_128_nev20", "kind": "eps", "n": 128, "nev": 20},
        # twelve requests of 2 K to 40 K rows served together
        {"name": "serve_12_to_200", "kind": "serve", "count": 12, "n": 200, "nev": 40},
    ]


def draw(rng):
    def log_int(lo, hi):
        return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))

    kind = rng.choice(["product", "product", "project", "project", "ritz", "block", "columns", "pcg",
                       "pcg", "solve", "eps", "serve"])
    op = rng.choice(["diff2d", "lap3d", "diff27"])
    side = {"diff2d": (45, 256), "lap3d": (16, 128), "diff27": (16, 128)}[op]
    if kind == "product":
        return {"kind": kind, "op": op, "n": log_int(*side), "k": log_int(1, 64)}
    if kind == "project":
        k = log_int(4, 120)
        return {"kind": kind, "op": op, "n": log_int(side[0], min(side[1], 200)),
                "m": min(460, k * rng.randint(1, 10)), "k": k}
    if kind == "ritz":
        k = log_int(8, 220)
        return {"kind": kind, "n": log_int(16, 112), "m": min(460, k + rng.randint(4, 240)), "k": k}
    if kind == "block":
        k = log_int(4, 100)
        return {"kind": kind, "n": log_int(20, 112), "m": min(340, k * rng.randint(3, 9)), "k": k}
    if kind == "columns":
        return {"kind": kind, "n": log_int(16, 96), "k": log_int(4, 60)}
    if kind == "pcg":
        return {"kind": kind, "op": op, "n": log_int(*side), "k": log_int(2, 100)}
    if kind == "solve":
        return {"kind": kind, "n": rng.randint(20, 56), "nev": rng.randint(10, 64)}
    if kind == "eps":
        return {"kind": kind, "n": rng.randint(32, 150), "nev": rng.randint(8, 32)}
    return {"kind": kind, "count": rng.randint(4, 12), "n": rng.randint(60, 220),
            "nev": rng.randint(12, 40)}


# ----------------------------------------------------- handles and their memory
class _MV(C.Structure):
    # the head of a multivector handle: where its column-major device block lies
    _fields_ = [("magic", C.c_uint32), ("nrows", C.c_int64), ("ncols", C.c_int64),
                ("ldd", C.c_int64), ("d", C.c_void_p)]


class _Table(solver.HipTable):
    """An operation table that gives its workspaces back when it is dropped."""

    def __init__(self):
        super().__init__()
        self._slots = {}

    def slot(self, name):
        if name not in self._slots:
            self._slots[name] = super().slot(name)
        return self._slots[name]

    def __del__(self):
        self.lib.HIPGCG_MultiLinearSolverFree_BlockPCG32(self.ops)
        self.lib.OPS_HIP_Clear(self.ops)


class _Block:
    """A multivector and its device memory: tensor() shows it as (columns, rows)."""

    def __init__(self, table, mat, cols):
        self.table, self.mat, self.cols = table, mat, cols
        self.h = table.create_multivec(cols, mat)
        mv = C.cast(self.h, C.POINTER(_MV)).contents
        assert mv.magic == 0x484D5631 and mv.nrows == mat.n and mv.ncols == cols
        self.__cuda_array_interface__ = {"shape": (cols, mat.n), "typestr": "<f8", "version": 2,
                                         "data": (mv.d, False), "strides": (8 * mv.ldd, 8)}

    def tensor(self):
        return torch.as_tensor(self, device="cuda")

    def __del__(self):
        self.table.destroy_multivec(self.h, self.cols)


def _ints(a, b):
    return (C.c_int * 2)(a, b)


def _dbl(a):
    return a.ctypes.data_as(abi.c_dbl_p)


# ------------------------------------------------------------------ inputs
def _rng(seed):
    return torch.Generator(device="cuda").manual_seed(seed)


def _normal(shape, g):
    return torch.randn(shape, generator=g, device="cuda", dtype=F64)


def _dim(case):
    return 2 if case.get("op") == "diff2d" or case["kind"] in ("eps", "serve") else 3


def _rows(case):
    return case["n"] ** _dim(case)


def _coef(case, seed):
    """Lognormal node coefficients (sigma 1 in 3D, 0.5 in 2D, as the problems have)."""
    s = 0.5 if case["op"] == "diff2d" else 1.0
    return np.exp(s * np.random.default_rng([seed, 1]).standard_normal(_rows(case)))


def _matrix(case, seed, fp32=False):
    n = case["n"]
    kind = problems.GRID_KINDS
    if case["op"] == "diff2d":
        return solver.DeviceMatrix.grid(kind["diffusion"], 2, 5, n, _coef(case, seed), 0.0, fp32)
    if case["op"] == "diff27":
        return solver.DeviceMatrix.grid(kind["diffusion"], 3, 27, n, _coef(case, seed), 1e-8, fp32)
    return solver.DeviceMatrix.grid(kind["laplace"], 3, 7, n, None, 0.0, fp32)


def _sines(n, m):
    """m lowest eigenvectors of the 7-point pair, B-orthonormal, as (m, n^3)."""
    k = torch.arange(1, n + 1, dtype=F64, device="cuda")
    s = torch.sin(k[:, None] * k[None, :] * (math.pi / (n + 1))) * math.sqrt(2.0 / (n + 1))
    c = 2.0 * np.cos(np.arange(1, n + 1) * math.pi / (n + 1))
    mu = (c[:, None, None] + c[None, :, None] + c[None, None, :]).ravel()
    low = np.argsort(-mu, kind="stable")[:m]
    out = torch.empty((m, n ** 3), dtype=F64, device="cuda")
    for i, at in enumerate(low):
        z, y, x = int(at) // (n * n), int(at) // n % n, int(at) % n
        v = s[z][:, None, None] * s[y][None, :, None] * s[x][None, None, :]
        out[i] = v.reshape(-1) / math.sqrt((12.0 + mu[at]) / 18.0)
    return out


def _smooth(case, k, g):
    """k columns made of a few low sine modes: what the vectors of a solve look like."""
    n, dim = case["n"], _dim(case)
    j = torch.arange(1, n + 1, dtype=F64, device="cuda")
    f = torch.arange(1, 7, dtype=F64, device="cuda")
    s = torch.sin(f[:, None] * j[None, :] * (math.pi / (n + 1))) * math.sqrt(2.0 / (n + 1))
    out = torch.empty((k, n ** dim), dtype=F64, device="cuda")
    for i in range(k):
        w = _normal((6,) * dim, g)
        if dim == 2:
            out[i] = (s.T @ w @ s).reshape(-1)
        else:
            v = torch.tensordot(s.T, w, dims=1)           # n 6 6
            v = torch.tensordot(v, s, dims=([1], [0]))    # n 6 n
            out[i] = torch.tensordot(v, s, dims=([1], [0])).reshape(-1)
    return out


# ------------------------------------------------------------------ states
class _State:
    pass


def prepare(case, seed):
    s = _State()
    s.case, kind, n = case, case["kind"], case["n"]
    if kind in ("solve", "eps", "serve"):
        return _prepare_whole(s, case, seed)
    s.table = t = _Table()
    g = _rng(seed)
    if kind == "product":
        k = case["k"]
        s.A = _matrix(case, seed)
        s.x, s.y = _Block(t, s.A, k), _Block(t, s.A, k)
        s.x.tensor().copy_(_normal((k, s.A.n), g))
        s.out = s.y.tensor()
        s.call, s.dots = t.slot("MatDotMultiVec"), t.slot("MultiVecInnerProd")
    elif kind == "project":
        m, k = case["m"], case["k"]
        s.A = _matrix(case, seed)
        s.v, s.ws = _Block(t, s.A, m), _Block(t, s.A, k)
        s.v.tensor().copy_(_normal((m, s.A.n), g) / math.sqrt(s.A.n))
        s.out = s.ws.tensor()
        s.call = t.slot("MultiVecQtAP")
    elif kind == "ritz":
        m, k = case["m"], case["k"]
        s.A = _matrix({**case, "op": "lap3d"}, seed)
        s.v, s.x = _Block(t, s.A, m), _Block(t, s.A, k)
        s.v.tensor().copy_(_normal((m, s.A.n), g) / math.sqrt(s.A.n))
        s.coef = _ritz_coef(case, seed)
        s.out = s.x.tensor()
        s.call = t.slot("MultiVecLinearComb")
    elif kind in ("block", "columns"):
        m, k = case.get("m", 0), case["k"]
        s.B = solver.DeviceMatrix.grid(problems.GRID_KINDS["mass"], 3, 7, n)
        s.v, s.w, s.ws = _Block(t, s.B, m + k), _Block(t, s.B, k), _Block(t, s.B, k)
        v, w = _new_block(case, seed)
        if m:
            s.v.tensor()[:m].copy_(v)
        s.w.tensor().copy_(w)
        s.out = s.v.tensor()[m:]
    elif kind == "pcg":
        k = case["k"]
        s.A = _matrix(case, seed, fp32=True)
        s.b, s.x0, s.x = _Block(t, s.A, k), _Block(t, s.A, k), _Block(t, s.A, k)
        # right-hand sides of smooth solutions, and a start that is 1e-3 off, rough and smooth:
        # a Ritz vector on its way to an eigenvector
        want = _smooth(case, k, g)
        s.x.tensor().copy_(want)
        torch.cuda.synchronize()
        t.slot("MatDotMultiVec")(s.A.handle, s.x.h, s.b.h, _ints(0, 0), _ints(k, k), t.ops)
        want += 1e-3 * _smooth(case, k, g)
        want += (1e-4 / math.sqrt(s.A.n)) * _normal(want.shape, g)
        s.x0.tensor().copy_(want)
        t.lib.HIPGCG_MultiLinearSolverSetup_BlockPCG32(30, 1e-2, 1e-14, None, 0.0, t.ops)
        s.out = s.x.tensor()
        s.call = t.slot("MultiLinearSolver")
    else:
        raise ValueError(kind)
    torch.cuda.synchronize()  # torch's stream and the library's do not wait for each other
    return s


def _ritz_coef(case, seed):
    m, k = case["m"], case["k"]
    q = np.random.default_rng([seed, 2]).standard_normal((m, k)) / math.sqrt(m)
    return np.asfortranarray(q)


def _new_block(case, seed):
    """The columns that are there (B-orthonormal) and a new block with parts along them."""
    n, m, k = case["n"], case.get("m", 0), case["k"]
    g = _rng(seed)
    w = _normal((k, n ** 3), g) / math.sqrt(n ** 3)
    v = None
    if m:
        v = _sines(n, m)
        w += (_normal((k, m), g) / math.sqrt(m)) @ v
    return v, w


def _served(case, seed):
    """Requests of sizes from 45 x 45 to n x n with 8 to nev pairs each."""
    got, count = [], case["count"]
    for i in range(count):
        side = int(round(45 * (case["n"] / 45) ** (i / max(1, count - 1))))
        nev = 8 + (13 * i) % (case["nev"] - 7)
        A, B = problems.varcoef_pair_2d(side, 0.5, np.random.default_rng([seed, 3, i]))
        bs, ni, nm = problems.slepc_block_policy(nev)
        got.append(problems.CCSProblem("request%d" % i, A, B, nev, bs, ni, nm))
    return got


def _prepare_whole(s, case, seed):
    kind, n = case["kind"], case["n"]
    s.seed = seed
    if kind == "solve":
        bs, ni, nm = problems.slepc_block_policy(case["nev"])
        s.problem = problems.stencil_grid_problem(n, 3, case["nev"], bs, ni, nm, "solve")
        s.mats = (solver.device_operator(s.problem.A, True),
                  solver.device_operator(s.problem.B, True))
    elif kind == "eps":
        s.A, s.B = problems.stencil_pair(n, 2)
    elif kind == "serve":
        s.requests = _served(case, seed)
        s.service = Service(workers=8)
    else:
        raise ValueError(kind)
    return s


# ------------------------------------------------------------------ passes
def run(s):
    return _RUN[s.case["kind"]](s)


def _run_product(s):
    k = s.case["k"]
    d = np.empty(k)
    s.call(s.A.handle, s.x.h, s.y.h, _ints(0, 0), _ints(k, k), s.table.ops)
    s.dots(b"D", s.x.h, s.y.h, 0, _ints(0, 0), _ints(k, k), _dbl(d), 1, s.table.ops)
    return {"product": s.out, "dots": d}


def _run_project(s):
    m, k = s.case["m"], s.case["k"]
    q = np.empty((m, k), order="F")
    s.call(b"S", b"N", s.v.h, s.A.handle, s.v.h, 0, _ints(0, m - k), _ints(m, m), _dbl(q), m,
           s.ws.h, s.table.ops)
    return {"projected": q, "A_w": s.out}


def _run_ritz(s):
    m, k = s.case["m"], s.case["k"]
    s.call(s.v.h, s.x.h, 0, _ints(0, 0), _ints(m, k), _dbl(s.coef), m, None, 0, s.table.ops)
    return s.out


def _run_block(s):
    m, k, t = s.case["m"], s.case["k"], s.table
    qtap, comb = t.slot("MultiVecQtAP"), t.slot("MultiVecLinearComb")
    one = np.ones(1)
    t.slot("MultiVecAxpby")(1.0, s.w.h, 0.0, s.v.h, _ints(0, m), _ints(k, m + k), t.ops)
    for removals in (2, 1):
        for _ in range(removals):
            q = np.empty((m, k), order="F")
            qtap(b"S", b"N", s.v.h, s.B.handle, s.v.h, 0, _ints(0, m), _ints(m, m + k), _dbl(q), m,
                 s.ws.h, t.ops)
            np.negative(q, out=q)
            comb(s.v.h, s.v.h, 0, _ints(0, m), _ints(m, m + k), _dbl(q), m, _dbl(one), 0, t.ops)
        if t.lib.HIP_MultiVecCholQR(s.v.h, m, m + k, s.B.handle, s.ws.h, 4.4e-16, 1e-10) != 1:
            raise RuntimeError("dependent block")
    return s.out


def _run_columns(s):
    k, t = s.case["k"], s.table
    qtap, comb, axpby = (t.slot(x) for x in ("MultiVecQtAP", "MultiVecLinearComb", "MultiVecAxpby"))
    one, r = np.ones(1), np.empty(k)
    axpby(1.0, s.w.h, 0.0, s.v.h, _ints(0, 0), _ints(k, k), t.ops)
    for c in range(k):
        qtap(b"S", b"N", s.v.h, s.B.handle, s.v.h, 0, _ints(c, c), _ints(k, c + 1), _dbl(r), k - c,
             s.ws.h, t.ops)
        inv = 1.0 / math.sqrt(r[0])
        axpby(0.0, None, inv, s.v.h, _ints(c, c), _ints(c + 1, c + 1), t.ops)
        if c + 1 < k:
            q = -inv * r[1:k - c]
            comb(s.v.h, s.v.h, 0, _ints(c, c + 1), _ints(c + 1, k), _dbl(q), 1, _dbl(one), 0, t.ops)
    return s.out


def _run_pcg(s):
    k, t = s.case["k"], s.table
    t.slot("MultiVecAxpby")(1.0, s.x0.h, 0.0, s.x.h, _ints(0, 0), _ints(k, k), t.ops)
    s.call(s.A.handle, s.b.h, s.x.h, _ints(0, 0), _ints(k, k), t.ops)
    return s.out


def _run_solve(s):
    got = solver.solve_problem(s.problem, mode="mixed", shift=0, rand="device", seed=s.seed,
                               mats=s.mats)
    return got.eval[:s.case["nev"]].copy()


def _run_eps(s):
    return solver.eps_solve(s.A, s.B, s.case["nev"], device_random=True, seed=s.seed).eigr


def _run_serve(s):
    tickets = [s.service.submit(p, seed=s.seed + i, shift=0) for i, p in enumerate(s.requests)]
    got = [s.service.wait(t) for t in tickets]
    return [r.eval[:p.nev].copy() for r, p in zip(got, s.requests)]


_RUN = {"product": _run_product, "project": _run_project, "ritz": _run_ritz, "block": _run_block,
        "columns": _run_columns, "pcg": _run_pcg, "solve": _run_solve, "eps": _run_eps,
        "serve": _run_serve}


# ------------------------------------------------------------------ work
def _nnz(op, n):
    return {"diff2d": 5 * n * n - 4 * n, "lap3d": 0, "diff27": (3 * n - 2) ** 3}[op]


def work(case):
    """Each input read once and each output written once; a constant-coefficient operator has no
    matrix to read.  The iterative kinds count one product per vector and direction."""
    kind, n, N = case["kind"], case["n"], _rows(case)
    points = {"diff2d": 5, "lap3d": 7, "diff27": 27}
    if kind == "product":
        k = case["k"]
        return {"bytes": 12.0 * _nnz(case["op"], n) + 16.0 * N * k,
                "flops": 2.0 * (points[case["op"]] + 1) * N * k}
    if kind == "project":
        m, k = case["m"], case["k"]
        return {"bytes": 12.0 * _nnz(case["op"], n) + 8.0 * N * (m + k) + 8.0 * m * k,
                "flops": 2.0 * N * m * k + 2.0 * points[case["op"]] * N * k}
    if kind == "ritz":
        m, k = case["m"], case["k"]
        return {"bytes": 8.0 * N * (m + k), "flops": 2.0 * N * m * k}
    if kind == "block":
        m, k = case["m"], case["k"]
        return {"bytes": 8.0 * N * (m + 2 * k), "flops": 2.0 * N * k * (2 * m + 2 * k + 7)}
    if kind == "columns":
        k = case["k"]
        return {"bytes": 16.0 * N * k, "flops": 2.0 * N * k * (k + 7)}
    if kind == "pcg":
        k = case["k"]
        return {"bytes": 8.0 * _nnz(case["op"], n) + 24.0 * N * k,
                "flops": 2.0 * points[case["op"]] * N * k}
    if kind == "serve":
        N = sum(int(round(45 * (n / 45) ** (i / max(1, case["count"] - 1)))) ** 2
                for i in range(case["count"]))
        return {"bytes": 12.0 * 10 * N + 8.0 * N * case["nev"], "flops": 4.0 * N * case["nev"]}
    nnz = 12.0 * 2 * 5 * N if kind == "eps" else 0.0
    return {"bytes": nnz + 8.0 * N * case["nev"], "flops": 4.0 * N * case["nev"] ** 2}


# ------------------------------------------------------------------ in 64 bits
def _apply(case, seed, X, mass=False):
    """A X (or B X of the 7-point pair) for X of shape (columns, rows), from the formulas."""
    n, dim = case["n"], _dim(case)
    X = X.reshape((X.shape[0],) + (n,) * dim)
    op = "mass" if mass else case["op"]
    steps = [-1, 0, 1]
    offs = [(a, b, c) for a in (steps if dim == 3 else [0]) for b in steps for c in steps]
    offs = [o[3 - dim:] for o in offs if any(o)]
    if op != "diff27":
        offs = [o for o in offs if sum(abs(v) for v in o) == 1]
    kappa = None
    if op in ("diff2d", "diff27"):
        kappa = torch.from_numpy(_coef(case, seed)).to("cuda").reshape((n,) * dim)
    out = torch.zeros_like(X)
    diag = torch.zeros((n,) * dim, dtype=F64, device="cuda")
    for o in offs:
        at = tuple(slice(max(0, -v), n - max(0, v)) for v in o)
        to = tuple(slice(max(0, v), n + min(0, v)) for v in o)
        if kappa is None:
            w = {"lap3d": -1.0, "mass": 1.0 / 18.0}[op]
        else:
            gd = 1.0 / sum(v * v for v in o)
            a, b = kappa[at], kappa[to]
            h = gd * (2.0 * a * b / (a + b))
            add = gd * kappa
            add[at] = h
            diag += add
            w = -h
        out[(slice(None),) + at] += w * X[(slice(None),) + to]
    if kappa is None:
        diag += {"lap3d": 6.0, "mass": 12.0 / 18.0}[op]
    elif op == "diff27":
        diag += 1e-8 * diag.max()
    out += diag * X
    return out.reshape(out.shape[0], -1)


def exact(case, seed):
    kind, n = case["kind"], case["n"]
    if kind == "solve":
        return _spectrum(n, 3, case["nev"])
    if kind == "eps":
        return _spectrum(n, 2, case["nev"])
    if kind in ("pcg", "serve"):
        return None  # an iterate stopped by its residual; a spectrum without a formula
    g = _rng(seed)
    if kind == "product":
        x = _normal((case["k"], _rows(case)), g)
        y = _apply(case, seed, x)
        return {"product": y, "dots": (x * y).sum(dim=1).cpu().numpy()}
    if kind == "project":
        m, k, N = case["m"], case["k"], _rows(case)
        v = _normal((m, N), g) / math.sqrt(N)
        aw = _apply(case, seed, v[m - k:])
        return {"projected": (v @ aw.T).cpu().numpy(), "A_w": aw}
    if kind == "ritz":
        m, N = case["m"], _rows(case)
        v = _normal((m, N), g) / math.sqrt(N)
        return torch.from_numpy(np.ascontiguousarray(_ritz_coef(case, seed).T)).to("cuda") @ v
    v, w = _new_block(case, seed)
    for p in range(2):
        if v is not None:
            for _ in range(2 - p):
                w = w - (_apply(case, seed, w, mass=True) @ v.T) @ v
        gram = w @ _apply(case, seed, w, mass=True).T
        low = torch.linalg.cholesky(0.5 * (gram + gram.T))
        w = torch.linalg.solve_triangular(low, torch.eye(len(low), dtype=F64, device="cuda"),
                                          upper=False) @ w
    return w


def _spectrum(n, dim, count):
    """Eigenvalues of the constant-coefficient pair: the closed form, by its sine modes."""
    c = 2.0 * np.cos(np.arange(1, n + 1) * math.pi / (n + 1))
    mu = c[:, None] + c[None, :] if dim == 2 else c[:, None, None] + c[None, :, None] + c
    mu = mu.ravel()
    lam = (2 * dim - mu) * (12.0 if dim == 2 else 18.0) / ((8.0 if dim == 2 else 12.0) + mu)
    lam.sort()
    return lam[:count]
