"""Performance cases: the work that programs using this framework have it do.

A case is one call sequence through symPACKMatrix2D on one matrix family:

  step   new values on an analysed structure: DistributeMatrix, Factorize,
         Solve, GetSolution (a time step, a Newton step, a request for a new
         factor in a solver service)
  solve  Solve and GetSolution on a resident factor

with values and right-hand sides resident on the GPU, or (host) in numpy
arrays, as the drop-in interface and the solver service pass them.

Matrices come from sympack_amd.matrices with the values rounded to multiples
of 2^-26, solutions are uniform on [-1, 1] in multiples of 2^-12: every
product and partial sum of b = A x is then exact in FP64, so x is the exact
solution of the system that the framework is given.
"""
import functools
import math

import numpy as np
import torch

import sympack_amd as sp

VALUE_BITS = 26
X_BITS = 12


def listed():
    def case(name, family, k, mode, nrhs, fact="LL", precision="FP64", ordering="NDBOX", max_size=150, host=False):
        return dict(name=name, family=family, k=k, mode=mode, nrhs=nrhs, fact=fact, precision=precision,
                    ordering=ordering, max_size=max_size, host=host)

    return [
        # the smallest system of the tests and of run_sympack2D's first
        # example: one right-hand side on a resident factor, launch-bound
        case("solve_2d_64_mmd", "2d", 64, "solve", 1, ordering="MMD", max_size=0),
        # the same system through host buffers with run_sympack2D's defaults
        # (MMD, no width limit): the driver's whole numeric sequence
        case("host_step_2d_64_mmd", "2d", 64, "step", 1, ordering="MMD", max_size=0, host=True),
        # the large 2D systems of the serving mix (n about 1e5): many levels
        # of small supernodes, odd edge
        case("step_2d_315", "2d", 315, "step", 4, ordering="NDGRID"),
        # the small 3D systems of the serving mix, odd edge and an odd number
        # of right-hand sides
        case("step_3d_17", "3d", 17, "step", 3),
        # 3D with run_sympack2D's defaults: supernodes of any width
        case("step_3d_24_mmd", "3d", 24, "step", 1, ordering="MMD", max_size=0),
        # a batch of follow-up solves merged by the solver service, host buffers
        case("host_solve_3d_37", "3d", 37, "solve", 19, host=True),
        # the benchmark's headline system: factor + solve, and the solve alone
        case("step_3d_48", "3d", 48, "step", 1),
        case("solve_3d_48", "3d", 48, "solve", 1),
        # the precision comparison's system: 27-point stencil, 16 right-hand
        # sides, FP64 and FP32 factor + FP64 refinement
        case("step_27pt_60", "27pt", 60, "step", 16),
        case("step_27pt_60_fp32ir", "27pt", 60, "step", 16, precision="FP32_IR"),
        # the largest: indefinite static LDL^T, 64 right-hand sides; solves
        # on its FP32 factor at half the edge
        case("step_ldl_80", "ldl", 80, "step", 64, fact="LDL"),
        case("solve_ldl_40_fp32ir", "ldl", 40, "solve", 8, fact="LDL", precision="FP32_IR"),
    ]


def _log_int(rng, lo, hi):
    return min(hi, max(lo, int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))))


def draw(rng):
    family = rng.choice(["2d", "2d", "3d", "3d", "3d", "27pt", "27pt", "ldl"])
    lo, hi = {"2d": (24, 447), "3d": (8, 48), "27pt": (8, 60), "ldl": (12, 80)}[family]
    k = _log_int(rng, lo, hi)
    nrhs = _log_int(rng, 1, 64)
    mode = rng.choice(["step", "step", "solve"])
    host = rng.random() < 0.25
    fact = "LDL" if family == "ldl" else "LL"
    precision = "FP32_IR" if family in ("27pt", "ldl") and rng.random() < 0.4 else "FP64"
    ordering, max_size = ("NDGRID" if family == "2d" else "NDBOX"), 150
    if (family == "2d" and k <= 128 or family == "3d" and k <= 24) and rng.random() < 0.4:
        ordering, max_size = "MMD", 0
    return dict(family=family, k=k, mode=mode, nrhs=nrhs, fact=fact, precision=precision, ordering=ordering,
                max_size=max_size, host=host)


def _matrix(case, seed):
    family, k = case["family"], case["k"]
    if family == "2d":
        n, cp, ri, v = sp.matrices.random_laplacian("2d", k, seed)
    elif family == "3d":
        n, cp, ri, v = sp.matrices.diffusion_3d_7pt(k, seed=seed)
    elif family == "27pt":
        n, cp, ri, v = sp.matrices.stencil_3d_27pt(k, seed=seed)
    else:
        n, cp, ri, v = sp.matrices.shifted_laplacian_3d_7pt(k, 0.3)
    return sp.DistSparseMatrix(n, cp, ri, np.round(v * 2.0 ** VALUE_BITS) / 2.0 ** VALUE_BITS)


def _solution(case, seed, n):
    """nrhs x n (columns of the right-hand side contiguous)."""
    rng = np.random.default_rng([seed, 1])
    q = 2 ** X_BITS
    return rng.integers(-q, q + 1, size=(case["nrhs"], n)).astype(np.float64) / q


def _product(A, x):
    """A x per row of x; exact, so the order of the sums does not matter."""
    rows = torch.from_numpy(A.rowind.astype(np.int64)).to(x.device)
    counts = torch.from_numpy(np.diff(A.colptr)).to(x.device)
    cols = torch.repeat_interleave(torch.arange(A.size, device=x.device), counts)
    v = torch.from_numpy(A.nzval).to(x.device)
    off = rows != cols
    ro, co, vo = rows[off], cols[off], v[off]
    b = torch.zeros_like(x)
    for j in range(x.shape[0]):
        b[j].index_add_(0, rows, v * x[j, cols])
        b[j].index_add_(0, co, vo * x[j, ro])
    return b


def _analysed(case, A):
    relax = sp.RelaxationParameters()
    relax.SetMaxSize(case["max_size"])
    M = sp.symPACKMatrix2D()
    M.Init(sp.symPACKOptions(ordering=case["ordering"], decomposition=case["fact"], relax=relax,
                             precision=case["precision"]))
    M.SymbolicFactorization(A)
    return M


def prepare(case, seed):
    A = _matrix(case, seed)
    x = torch.from_numpy(_solution(case, seed, A.size)).cuda()
    b = _product(A, x)
    M = _analysed(case, A)
    state = dict(M=M, nrhs=case["nrhs"], step=case["mode"] == "step", host=case["host"], A=A)
    if case["host"]:
        state["b"] = np.asfortranarray(b.cpu().numpy().T)  # n x nrhs, column-major
    else:
        state["vals"] = torch.from_numpy(A.nzval).cuda()
        state["b"] = b
        state["x"] = torch.empty_like(b)
    torch.cuda.synchronize()
    if case["mode"] == "solve":
        M.DistributeMatrix(A)
        M.Factorize()
    return state


def run(state):
    M, nrhs = state["M"], state["nrhs"]
    if state["host"]:
        if state["step"]:
            M.DistributeMatrix(state["A"])
            M.Factorize()
        M.Solve(state["b"], nrhs)
        return M.GetSolution(nrhs).reshape(-1, nrhs)
    if state["step"]:
        M.DistributeMatrixDevice(state["vals"].data_ptr())
        M.Factorize()
    M.SolveDevice(state["b"].data_ptr(), nrhs)
    M.GetSolutionDevice(state["x"].data_ptr(), nrhs)
    return state["x"]


def exact(case, seed):
    n = case["k"] ** (2 if case["family"] == "2d" else 3)
    x = _solution(case, seed, n)
    return np.ascontiguousarray(x.T) if case["host"] else torch.from_numpy(x)


@functools.lru_cache(maxsize=64)
def _structure(family, k, ordering, max_size):
    case = dict(family=family, k=k, ordering=ordering, max_size=max_size, fact="LL", precision="FP64")
    A = _matrix(case, 0)
    M = _analysed(case, A)
    # unrelaxed column counts: the factor of this ordering without any padding
    flops, nnz = M.stats()["flops"], M.stats()["nnz_l"]
    return A.size, A.nnz, flops, nnz


def work(case):
    """Factor: sum of the squared column counts, the values read and the
    factor written; solve: 4 flops per factor entry and right-hand side, the
    factor, the right-hand sides read and the solutions written."""
    n, nnz, flops, nnz_l = _structure(case["family"], case["k"], case["ordering"], case["max_size"])
    size = 8 if case["precision"] == "FP64" else 4
    vec = 16 * n * case["nrhs"]
    w = dict(bytes=nnz_l * size + vec, flops=4 * nnz_l * case["nrhs"])
    if case["mode"] == "step":
        w["bytes"] += 8 * nnz
        w["flops"] += flops
    return w
