"""The work that users of this library have it do, as cases that can be timed.

A case names a matrix family of workloads.py with its size, the factor's precision, the
number of right-hand sides and how the library is called (`call`):

  step      refactor a resident plan and solve to the tolerance, right-hand sides and
            solutions in HBM (sogl_factor_run + sogl_solve_refined_device): one time or
            Newton step, and the step that bench.py times
  resident  solve with a factor that is kept in HBM (sogl_solve_refined_device)
  hit       the same from host arrays, as the serving loop answers a request whose
            matrix it holds (permute, sogl_solve, unpermute)
  request   factor and then `hit`: a request whose matrix is new to the server
  dropin    sogl_solveLU: plan, load, factor and solve in one call on host arrays

FP64 cases solve once (max_iter 0 where the call has one), FP32 ones are refined in FP64.
The families whose solutions an FP32 factor's refinement reaches to all digits (diagonally
dominant or convection-dominated) appear in FP32; variable-coefficient diffusion, whose
condition grows with the grid, in FP64.
"""
import ctypes
import math
import os
import sys

import numpy as np
import torch

_PKG = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "sparse-operator-graph-lu_amd")
if _PKG not in sys.path:
    sys.path.insert(0, _PKG)

import sogl  # noqa: E402
import workloads as W  # noqa: E402

#: Refinement tolerance of the FP32 cases (the benchmark's, by family).
_TOL = {"convdiff2d": 1e-10}
_MAX_ITER = 30


def listed():
    return [
        # the smallest: a repeated solve on a kept factor of the 64 x 64 Poisson problem
        dict(name="resident_poisson2d_64", call="resident", family="poisson2d", m=64, prec="fp64", nrhs=1),
        # and its refactorisation with one solve (the smoke test's size)
        dict(name="step_poisson2d_64", call="step", family="poisson2d", m=64, prec="fp64", nrhs=1),
        # the reference's own use: a matrix and a right-hand side in, x out; an odd grid
        dict(name="dropin_poisson2d_101", call="dropin", family="poisson2d", m=101, prec="fp64", nrhs=1),
        # serving: a repeat of a matrix the server holds, a few right-hand sides
        dict(name="hit_diffusion2d_253_rhs5", call="hit", family="diffusion2d", m=253, prec="fp64", nrhs=5),
        # serving: the first request of a mid-sized matrix
        dict(name="request_diffusion2d_128", call="request", family="diffusion2d", m=128, prec="fp64", nrhs=1),
        # serving's most right-hand sides on a 3D grid
        dict(name="resident_diffusion3d_31_rhs16", call="resident", family="diffusion3d", m=31, prec="fp64", nrhs=16),
        # the 3D benchmark, FP32 factor with FP64 refinement, one workgroup per CU (what the
        # autotuner picks for it)
        dict(name="step_laplace3d_48_fp32", call="step", family="laplace3d", m=48, prec="fp32", nrhs=1, one_per_cu=True),
        # the same in FP64 with the default executor settings
        dict(name="step_laplace3d_48_fp64", call="step", family="laplace3d", m=48, prec="fp64", nrhs=1),
        # many right-hand sides on a nearly dense factor: a kept FP64 factor, ragged sizes
        dict(name="resident_random_4099_rhs100", call="resident", family="random", m=4099, prec="fp64", nrhs=100),
        # the many-right-hand-side benchmark (random band matrix, 128 columns)
        dict(name="step_random_16384_rhs128", call="step", family="random", m=16384, prec="fp32", nrhs=128),
        # symmetric input: an L L^T factor
        dict(name="step_symmetric3d_37", call="step", family="symmetric3d", m=37, prec="fp64", nrhs=1),
        # the largest, the headline benchmark: 1M unknowns of 2D convection-diffusion
        dict(name="step_convdiff2d_1000", call="step", family="convdiff2d", m=1000, prec="fp32", nrhs=1, one_per_cu=True),
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    """One more case of the ranges above: grids from 16 x 16 up, 1 to 128 right-hand sides."""
    call = rng.choice(["step", "step", "resident", "resident", "hit", "request", "dropin"])
    if call == "dropin":
        family = rng.choice(["poisson2d", "diffusion2d", "laplace3d"])
    elif call in ("hit", "request"):
        family = rng.choice(["diffusion2d", "diffusion3d"])
    else:
        family = rng.choice(["poisson2d", "diffusion2d", "diffusion3d", "laplace3d", "random", "symmetric3d", "convdiff2d"])
    m = {
        "poisson2d": lambda: _log_int(rng, 16, 300),
        "diffusion2d": lambda: _log_int(rng, 32, 400),
        "diffusion3d": lambda: rng.randint(12, 36),
        "laplace3d": lambda: rng.randint(12, 44),
        "random": lambda: _log_int(rng, 1000, 10000),
        "symmetric3d": lambda: rng.randint(12, 38),
        "convdiff2d": lambda: _log_int(rng, 64, 640),
    }[family]()
    if call == "dropin":
        m = min(m, 160 if family != "laplace3d" else 24)
        return dict(call=call, family=family, m=m, prec="fp64", nrhs=1)
    prec = rng.choice(["fp32", "fp64"]) if family in ("laplace3d", "random", "convdiff2d") else "fp64"
    if call in ("hit", "request"):
        nrhs = rng.randint(1, 16)
    elif family == "random":
        nrhs = _log_int(rng, 1, 128)
    else:
        nrhs = rng.choice([1, 1, rng.randint(2, 16), _log_int(rng, 16, 64)])
    case = dict(call=call, family=family, m=m, prec=prec, nrhs=nrhs)
    if call == "step" and family in ("laplace3d", "convdiff2d") and rng.random() < 0.5:
        case["one_per_cu"] = True
    return case


def _problem(case, seed):
    """Matrix and right-hand sides (n, nrhs) of a case; every family draws from the seed."""
    family, m, nrhs = case["family"], case["m"], case["nrhs"]
    s = int(seed) % (1 << 31)
    if family == "poisson2d":
        p = W.poisson2d(m, seed=s)
    elif family in ("diffusion2d", "diffusion3d"):
        p = W.diffusion_varcoef(m, 2 if family == "diffusion2d" else 3, seed=s)
    elif family == "symmetric3d":
        p = W.symmetric_lower(W.diffusion_varcoef(m, 3, seed=s))
    elif family == "laplace3d":
        p = W.laplace3d_dominant(m, seed=s, rhs_seed=s + 1000)
    elif family == "random":
        p = W.random_band(m, seed=s, nrhs=1, rhs_seed=s + 1000)
    else:  # cell Peclet numbers around the benchmark's 10
        p = W.convdiff2d(m, pe=9.0 + 2.0 * W.uniform01(s, 1)[0], vel=(1.0, 0.5), seed=s)
    b = W.uniform_pm1(s + 2000, p.n * nrhs).reshape(nrhs, p.n)
    return p, b


_device = None


def _dev():
    """The program's device context, made once."""
    global _device
    if _device is None:
        _device = sogl.Device(0)
    return _device


class _State:
    """A resident factor with its plan and vectors; the factor is released with it."""

    def __init__(self, case, seed):
        self.case = case
        self.p, b = _problem(case, seed)
        self.fid = None
        if case["call"] == "dropin":
            self.b = b[0].copy()
            return
        dev = _dev()
        self.plan = sogl.Plan(self.p.n, self.p.row, self.p.col, self.p.val, symmetric=self.p.symmetric)
        serving = case["call"] in ("hit", "request")
        dev.set_pool_reuse(sogl.REUSE_ON if serving else sogl.REUSE_AUTO)  # as the server sets it
        self.fid = dev.load(self.plan, sogl.FP32 if case["prec"] == "fp32" else sogl.FP64)
        if serving:
            self.b = b.T if case["nrhs"] > 1 else b[0]  # (n, nrhs), column-major
        else:
            dev.attach_refine(self.fid, self.plan)
            self.b = torch.from_numpy(b).cuda()
            self.x = torch.zeros_like(self.b)
            torch.cuda.synchronize()
        if case["call"] in ("resident", "hit"):
            _factor(self)

    def __del__(self):
        if self.fid is not None:
            _dev().release(self.fid)
            self.fid = None


def prepare(case, seed):
    return _State(case, seed)


def _factor(s):
    if s.case.get("one_per_cu"):
        _dev().factor_config(s.fid, sogl.EXEC_PERSISTENT, 1, 1)
    else:
        _dev().factor(s.fid, sogl.EXEC_PERSISTENT)


def run(state):
    s, case = state, state.case
    call = case["call"]
    if call == "dropin":
        p, x = s.p, np.empty(s.p.n)
        i32, f64 = ctypes.POINTER(ctypes.c_int32), ctypes.POINTER(ctypes.c_double)
        lib = sogl.load()
        rc = lib.sogl_solveLU(p.n, p.nnz, 0, p.row.ctypes.data_as(i32), p.col.ctypes.data_as(i32),
                              p.val.ctypes.data_as(f64), s.b.ctypes.data_as(f64), x.ctypes.data_as(f64))
        if rc != sogl.OK:
            raise sogl.SoglError(rc, lib.sogl_last_error().decode())
        return x
    dev = _dev()
    if call in ("step", "request"):
        _factor(s)
    if call in ("hit", "request"):
        return s.plan.unpermute(dev.solve(s.fid, s.plan.permute_rhs(s.b)))
    fp32 = case["prec"] == "fp32"
    _, resid, rc = dev.solve_refined_device(s.fid, s.b.data_ptr(), s.x.data_ptr(), case["nrhs"],
                                            _TOL.get(case["family"], 1e-12), _MAX_ITER if fp32 else 0)
    if rc != sogl.OK:
        raise sogl.SoglError(rc, f"residual {resid}")
    return s.x


def _shape(case):
    """(unknowns, matrix entries, entries of L and U, operations of the factorisation) of a
    banded elimination: half bandwidth m on an m x m grid, 3/4 m^2 on an m^3 grid (the
    largest level set), the whole matrix for the random family."""
    family, m = case["family"], case["m"]
    if family == "random":
        return m, 69 * m, m * m, 2 * m ** 3 / 3
    if family in ("poisson2d", "diffusion2d", "convdiff2d"):
        n, nnz, w = m * m, 5 * m * m, m
    else:
        n, nnz, w = m ** 3, 7 * m ** 3, 0.75 * m * m
    sym = 0.5 if family == "symmetric3d" else 1.0
    return n, nnz, 2 * n * w * sym, 2 * n * w * w * sym


def work(case):
    n, nnz, lu, fact = _shape(case)
    el, r = (4 if case["prec"] == "fp32" else 8), case["nrhs"]
    solves = 2 if case["prec"] == "fp32" else 1  # the first solve and one correction
    # a solve reads L and U once and b, and writes x; the residual reads the matrix
    b = solves * (el * lu + 16 * n * r) + (0 if case["call"] in ("hit", "request", "dropin") else 12 * nnz)
    f = solves * 2 * lu * r + 2 * nnz * r
    if case["call"] in ("step", "request", "dropin"):  # the matrix read, the factor written
        b += 12 * nnz + el * lu
        f += fact
    return {"bytes": b, "flops": f}


def _solve_grid(n, size, row, col, val, b):
    """x of A x = b (b: (n, k)) for a matrix whose couplings reach at most the next block of
    `size` unknowns: block elimination with pivoted dense solves."""
    k = n // size
    order = np.argsort(row // size, kind="stable")
    row, col, val = row[order].astype(np.int64), col[order].astype(np.int64), val[order]
    start = np.searchsorted(row // size, np.arange(k + 1))
    carry_u, carry_y, ups, ys = None, None, [], []
    for i in range(k):
        q = slice(start[i], start[i + 1])
        wide = torch.zeros(size, 3 * size, dtype=torch.float64)
        wide[torch.from_numpy(row[q] - i * size), torch.from_numpy(col[q] - (i - 1) * size)] = torch.from_numpy(val[q])
        low, d, up = wide[:, :size], wide[:, size:2 * size], wide[:, 2 * size:]
        y = b[i * size:(i + 1) * size]
        if i:
            nz = low.abs().sum(1) > 0  # the rows that reach back
            d[nz] -= low[nz] @ carry_u
            y = y - low @ carry_y
        z = torch.linalg.solve(d, torch.cat([up, y], 1))
        carry_u, carry_y = z[:, :size].contiguous(), z[:, size:].contiguous()
        ups.append(carry_u)
        ys.append(carry_y)
    x = [ys[-1]]
    for i in range(k - 2, -1, -1):
        x.append(ys[i] - ups[i] @ x[-1])
    return torch.cat(x[::-1])


def exact(case, seed):
    p, b = _problem(case, seed)
    row, col, val = W.full_matrix(p)
    bt = torch.from_numpy(b.T.copy())
    family, m = case["family"], case["m"]
    if family == "random":
        a = torch.zeros(p.n, p.n, dtype=torch.float64)
        a[torch.from_numpy(row.astype(np.int64)), torch.from_numpy(col.astype(np.int64))] = torch.from_numpy(val)
        x = torch.linalg.solve(a, bt)
    elif family == "convdiff2d" and m > 700:
        return None  # takes too long
    else:
        x = _solve_grid(p.n, m if family in ("poisson2d", "diffusion2d", "convdiff2d") else m * m, row, col, val, bt)
    if case["call"] in ("step", "resident"):
        return x.T.contiguous()
    return x.numpy() if case["call"] != "dropin" and case["nrhs"] > 1 else x[:, 0].numpy()
