"""Performance cases of the two-level Schwarz PCG path.

Each case is one call (or, for `time_to_solve` and `train`, the few calls of one
step) of the package's public entry points, on the workloads that this
repository benchmarks and tests: the 2-D Laplacian, the 3-D diffusion field
decomposed over several processes, and the locally refined P1 FEM mesh with uneven
subdomains.  `listed()` names the cases that are followed, `draw()` gives
others of the same ranges, odd sizes and ragged partitions among them.

kinds
  spmv            y = A x with the solver's matrix (device pointers)
  apply           z = M^-1 r, one preconditioner apply, FP64 factors
  solve           PCG to rtol 1e-8 with the set-up in hand
  batch           PCG for nrhs right-hand sides at once, set-up in hand
  time_to_solve   doug_setup and PCG, the matrix already handed over
  train           forward and backward of the differentiable solve, from the
                  cells' log-coefficients to their gradient

problems
  lap2d   5-point Laplacian on size^2 points, boxes of edge `block`
  diff3d  7-point diffusion on size^3 cells, kappa = exp(g), boxes of edge
          `block`, each owned by a process of its own (`ranks`) or all by one
  fem2d   P1 diffusion on the Delaunay mesh of `size` points, 2 % of them near
          a circle, block x block cells of growing width, overlap 2
"""
from __future__ import annotations

import functools
import math

import numpy as np
import torch

import doug_amd as D
from doug_amd import problems as P
from doug_amd.autograd import DougSolve, PatternSolver, diffusion3d_pattern, diffusion3d_values

DEV = "cuda:0"

# control values of the repository's benchmark and tests
CTL = {
    "lap2d": dict(radius1=2, strong1=0.08, smoothers=1, overlap=1, symmstruct=1, symmnumeric=1),
    "diff3d": dict(radius1=4, minasize1=100, maxasize1=343, strong1=0.08, smoothers=1, overlap=1,
                   symmstruct=1, symmnumeric=1),
    "fem2d": dict(radius1=5, minasize1=60, maxasize1=121, strong1=0.08, smoothers=1, overlap=2,
                  symmstruct=1, symmnumeric=1),
}
TRAIN_CTL = dict(radius1=2, strong1=0.08, smoothers=1, overlap=1, symmstruct=1, symmnumeric=1)


def _case(name, kind, problem, size, block, precision=0, nrhs=1, ranks=False):
    c = dict(kind=kind, problem=problem, size=size, block=block, precision=precision, nrhs=nrhs, ranks=ranks)
    return c if name is None else dict(name=name, **c)


def listed():
    return [
        # the smallest calls: one operator of a small 2-D system inside a
        # caller's own loop, where launches and latency count
        _case("spmv_128sq", "spmv", "lap2d", 128, 64),
        _case("apply_128sq", "apply", "lap2d", 128, 64),
        # the small system solved: hundreds of short launches
        _case("solve_128sq", "solve", "lap2d", 128, 64),
        # one operator of the large 3-D system inside a caller's own Krylov loop
        _case("spmv_128cube", "spmv", "diff3d", 128, 16, ranks=True),
        # the same for the preconditioner, on a size that boxes do not divide:
        # 343 subdomains of 64 to 4096 cells and their layers, one process
        _case("apply_100cube", "apply", "diff3d", 100, 16),
        # an unstructured system with uneven subdomains, fewer than the GPU has CUs
        _case("solve_fem250k", "solve", "fem2d", 250_000, 8),
        # the benchmarked system, plain FP64 and with FP32 subdomain factors
        _case("solve_128cube_fp64", "solve", "diff3d", 128, 16, precision=0, ranks=True),
        _case("solve_128cube_fp32", "solve", "diff3d", 128, 16, precision=1, ranks=True),
        # many load cases at once, the full batch and a small odd one
        _case("batch32_128cube", "batch", "diff3d", 128, 16, precision=1, nrhs=32, ranks=True),
        _case("batch5_fem100k", "batch", "fem2d", 100_000, 6, precision=1, nrhs=5),
        # new matrix values at every step: the headline time to solve
        _case("time_to_solve_128cube", "time_to_solve", "diff3d", 128, 16, precision=1, ranks=True),
        # one step of a coefficient inversion, forward and backward, to 1e-10
        _case("train_64cube", "train", "diff3d", 64, 16),
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["spmv", "apply", "solve", "solve", "batch", "batch", "time_to_solve", "train"])
    if kind == "train":
        return _case(None, kind, "diff3d", _log(rng, 16, 60), rng.randint(8, 16))
    if kind == "time_to_solve":
        return _case(None, kind, "diff3d", _log(rng, 24, 120), rng.randint(9, 18), rng.randint(0, 1), ranks=True)
    problem = rng.choice(["lap2d", "diff3d", "fem2d"])
    prec = 0 if kind in ("spmv", "apply") else rng.randint(0, 1)
    nrhs = rng.randint(1, 32) if kind == "batch" else 1
    if problem == "lap2d":
        return _case(None, kind, problem, _log(rng, 48, 600), rng.randint(24, 72), prec, nrhs)
    if problem == "diff3d":
        ranks = rng.random() < 0.5
        top = 120 if kind == "spmv" else 64 if kind == "batch" else 96
        return _case(None, kind, problem, _log(rng, 20, top), rng.randint(8, 18), prec, nrhs, ranks)
    size = _log(rng, 8_000, 120_000)
    return _case(None, kind, problem, size, max(2, round(math.sqrt(size / rng.uniform(1500, 5000)))), prec, nrhs)


# --------------------------------------------------------------------------
# problems: padded rows (n, width) of columns and values; the pattern of a
# size is kept, the values follow from the seed

@functools.lru_cache(maxsize=2)
def _stencil(size, dims):
    """Columns of each cell's row in ascending order, and which of them exist."""
    n = size ** dims
    coords = np.indices((size,) * dims).reshape(dims, -1)
    ok = []
    steps = [size ** (dims - 1 - a) for a in range(dims)]
    order = [(-steps[a], a, -1) for a in range(dims)] + [(0, -1, 0)] + [(steps[a], a, 1) for a in reversed(range(dims))]
    cols = np.empty((n, len(order)), np.int32)
    for k, (o, a, s) in enumerate(order):
        cols[:, k] = np.arange(n) + o
        ok.append(np.ones(n, bool) if a < 0 else coords[a] > 0 if s < 0 else coords[a] < size - 1)
    return cols, np.stack(ok, 1), order


@functools.lru_cache(maxsize=2)
def _mesh(npoints):
    """The mesh of this many points: matrix rows, padded, and the points."""
    n, i, j, v, pts = P.fem_p1_square(npoints, 8)
    ptr = np.searchsorted(i, np.arange(1, n + 2))
    width = int(np.diff(ptr).max())
    ok = np.arange(width)[None, :] < np.diff(ptr)[:, None]
    cols = np.zeros((n, width), np.int32)
    vals = np.zeros((n, width))
    cols[ok], vals[ok] = j - 1, v
    return cols, vals, ok, pts


def _rows(case, seed):
    """(columns, values, which entries exist), the values of this seed."""
    size, problem = case["size"], case["problem"]
    if problem == "fem2d":
        cols, v0, ok, _ = _mesh(size)
        n = len(cols)
        # element stiffness times a nodal conductivity: harmonic means on the
        # edges, the row's boundary share with the node's own
        kappa = np.exp(0.5 * np.random.default_rng(seed).standard_normal(n))
        diag = cols == np.arange(n)[:, None]
        kj = kappa[cols]
        v = np.where(ok & ~diag, v0 * (2.0 * kappa[:, None] * kj / (kappa[:, None] + kj)), 0.0)
        share = np.maximum(v0.sum(1), 0.0) * kappa
        v = np.where(diag & ok, (share - v.sum(1))[:, None], v)
        return cols, v, ok
    dims = 2 if problem == "lap2d" else 3
    cols, ok, order = _stencil(size, dims)
    n = len(cols)
    if problem == "lap2d":
        v = np.where(np.array([o[1] < 0 for o in order])[None, :], 4.0, -1.0) * ok
        return cols, v, ok
    kappa = np.exp(P.smoothed_gaussian(size, seed, dims=dims))
    v = np.zeros(kappa.shape + (len(order),))
    mid = len(order) // 2
    for a in range(dims):
        k = a  # the column of the lower neighbour along this axis; the upper one mirrors it
        lo, hi = [slice(None)] * dims, [slice(None)] * dims
        lo[a], hi[a] = slice(0, size - 1), slice(1, size)
        lo, hi = tuple(lo), tuple(hi)
        f = 2.0 * kappa[lo] * kappa[hi] / (kappa[lo] + kappa[hi])
        v[hi + (k,)] = -f
        v[lo + (2 * mid - k,)] = -f
        v[lo + (mid,)] += f
        v[hi + (mid,)] += f
        for end in (0, size - 1):
            e = [slice(None)] * dims
            e[a] = end
            v[tuple(e) + (mid,)] += kappa[tuple(e)]
    return cols, v.reshape(n, len(order)), ok


@functools.lru_cache(maxsize=2)
def _entries(problem, size):
    """0-based rows and columns of the entries, row by row."""
    cols, ok = _mesh(size)[0:3:2] if problem == "fem2d" else _stencil(size, 2 if problem == "lap2d" else 3)[:2]
    return np.repeat(np.arange(len(cols), dtype=np.int32), ok.sum(1)), cols[ok]


def _partition(case):
    if case["problem"] == "fem2d":
        return P.graded_partition(_mesh(case["size"])[3], case["block"])
    return _boxes(case["size"], 2 if case["problem"] == "lap2d" else 3, case["block"])


@functools.lru_cache(maxsize=4)
def _boxes(size, dims, block):
    return P.block_partition((size,) * dims, block)


def _unknowns(case):
    if case["problem"] == "fem2d":
        return len(_mesh(case["size"])[0])
    return case["size"] ** (2 if case["problem"] == "lap2d" else 3)


def _vector(n, seed, cols=None):
    g = torch.Generator(device=DEV).manual_seed(seed)
    shape = (n,) if cols is None else (n, cols)
    return torch.rand(shape, generator=g, dtype=torch.float64, device=DEV) * 2.0 - 1.0


def _theta(case, seed):
    t = 0.5 * P.smoothed_gaussian(case["size"], seed).ravel()
    return torch.tensor(t, dtype=torch.float64, device=DEV)


# --------------------------------------------------------------------------

def prepare(case, seed):
    n = _unknowns(case)
    if case["kind"] == "train":
        N = case["size"]
        ps = PatternSolver(*diffusion3d_pattern(N), TRAIN_CTL, partition=_partition(case), tol=1e-10)
        return dict(kind="train", N=N, ps=ps, theta=_theta(case, seed), b=_vector(n, seed + 1),
                    target=_vector(n, seed + 2))
    _, v, ok = _rows(case, seed)
    s = D.Solver(0)
    s.set_params(**CTL[case["problem"]])
    s.set_matrix(n, *_entries(case["problem"], case["size"]), v[ok], 0)
    part = _partition(case)
    if case["ranks"]:
        rank = np.empty(n, np.int32)
        rank[part[1] - 1] = np.repeat(np.arange(len(part[0]) - 1), np.diff(part[0]))
        s.set_ranks(len(part[0]) - 1, rank, 0)
    else:
        s.set_partition(*part)
    s.setup(case["precision"])
    many = case["nrhs"] if case["kind"] == "batch" else None
    if many:
        s.prepare_batch()
    if n >= 50_000:  # a program of many solves tunes the launch shapes once
        s.autotune(5)
    return dict(kind=case["kind"], s=s, precision=case["precision"], nrhs=case["nrhs"],
                b=_vector(n, seed + 1, many), x=torch.zeros((n,) if many is None else (n, many),
                                                            dtype=torch.float64, device=DEV))


def run(st):
    kind = st["kind"]
    if kind == "train":
        th = st["theta"].clone().requires_grad_(True)
        b = st["b"].clone().requires_grad_(True)
        x = DougSolve.apply(diffusion3d_values(th, st["N"]), b, st["ps"])
        loss = 0.5 * torch.sum((x - st["target"]) ** 2)
        loss.backward()
        return dict(x=x.detach(), grad_theta=th.grad, grad_b=b.grad)
    s, b, x = st["s"], st["b"], st["x"]
    if kind == "spmv":
        s.spmv_device(b.data_ptr(), x.data_ptr())
        return x
    if kind == "apply":
        s.prec_device(b.data_ptr(), x.data_ptr())
        return x
    x.zero_()
    if kind == "batch":
        its = s.pcg_batch_device(st["nrhs"], b.data_ptr(), x.data_ptr(), 1e-8, 2000)
        return dict(x=x, iterations=its)
    if kind == "time_to_solve":
        s.setup(st["precision"])
    it, cond, _ = s.pcg_device(b.data_ptr(), x.data_ptr(), 1e-8, 2000)
    # with FP32 factors the condition estimate carries the factors' rounding
    # (1e-7), as the solution does not
    if st["precision"] == 0:
        return dict(x=x, iterations=it, cond=cond)
    return dict(x=x, iterations=it)


# --------------------------------------------------------------------------

# iterations of a solve to 1e-8 on these problems (1e-10 in training, twice)
ITERATIONS = {"lap2d": 25, "diff3d": 60, "fem2d": 70}


def work(case):
    n = _unknowns(case)
    problem, kind, k = case["problem"], case["kind"], case["nrhs"]
    nnz = {"lap2d": 5, "diff3d": 7, "fem2d": 7}[problem] * n
    spmv = dict(bytes=12 * nnz + 4 * (n + 1) + 16 * n * k, flops=2 * nnz * k)
    if kind == "spmv":
        return spmv
    # one apply reads each subdomain's factor at least once; a factor of s
    # unknowns has about 5 s^(4/3) entries in 3-D and 1.75 s log2(s) in 2-D
    # under nested dissection (A. George, SIAM J. Numer. Anal. 10 (1973) 345-363)
    if problem == "fem2d":
        nsub = case["block"] ** 2
        s = n / nsub + 4 * 2 * math.sqrt(n / nsub)
    elif problem == "lap2d":
        nsub = math.ceil(case["size"] / case["block"]) ** 2
        s = min(case["size"], case["block"] + 2) ** 2
    else:
        nsub = math.ceil(case["size"] / case["block"]) ** 3
        s = min(case["size"], case["block"] + 2) ** 3
    s = min(s, n)
    entries = nsub * (5.0 * s ** (4.0 / 3.0) if problem == "diff3d" else 1.75 * s * math.log2(max(s, 2)))
    size = 4 if case["precision"] == 1 else 8
    apply = dict(bytes=size * entries + 16 * n * k, flops=4 * entries * k)
    if kind == "apply":
        return apply
    its = ITERATIONS[problem] * (2 if kind == "train" else 1)
    return dict(bytes=its * (spmv["bytes"] + apply["bytes"]), flops=its * (spmv["flops"] + apply["flops"]))


# --------------------------------------------------------------------------
# the exact solution: Jacobi-preconditioned CG in 64 bits on the padded rows,
# to a residual far below the cases' tolerance

def _mul(cols, v, x):
    y = torch.zeros_like(x)
    for k in range(cols.shape[1]):
        vk = v[:, k]
        y += (vk[:, None] if x.ndim == 2 else vk) * x[cols[:, k]]
    return y


def _cg(cols, v, b, tol=2e-14, maxit=6000):
    n = len(cols)
    diag = (v * (cols == torch.arange(n, device=DEV)[:, None])).sum(1)
    inv = 1.0 / (diag[:, None] if b.ndim == 2 else diag)
    x = torch.zeros_like(b)
    r = b.clone()
    z = inv * r
    p = z.clone()
    rz = (r * z).sum(0)
    r0 = (r * r).sum(0)
    for it in range(maxit):
        q = _mul(cols, v, p)
        a = rz / (p * q).sum(0)
        x += a * p
        r -= a * q
        z = inv * r
        new = (r * z).sum(0)
        if it % 25 == 24 and bool(((r * r).sum(0) <= tol * tol * r0).all()):
            break
        p = z + (new / rz) * p
        rz = new
    return x


def _faces(theta, N):
    """Padded values of the 7-point rows for kappa = exp(theta), differentiable."""
    cols, ok, order = _stencil(N, 3)
    kappa = torch.exp(theta)
    out, diag = [None] * len(order), torch.zeros_like(kappa)
    for k, o in enumerate(order):
        if o[1] < 0:
            mid = k
            continue
        m = torch.as_tensor(ok[:, k], device=DEV)
        kj = kappa[torch.as_tensor(np.where(ok[:, k], cols[:, k], 0), device=DEV).long()]
        f = torch.where(m, 2.0 * kappa * kj / (kappa + kj), kappa)
        diag = diag + f
        out[k] = torch.where(m, -f, torch.zeros_like(f))
    out[mid] = diag
    return torch.stack(out, 1)


def exact(case, seed):
    kind = case["kind"]
    if kind == "apply":  # needs the aggregates and index sets: no plain form
        return None
    n = _unknowns(case)
    if kind == "train":
        cols, ok, _ = _stencil(case["size"], 3)
        cols = torch.as_tensor(np.where(ok, cols, 0), device=DEV).long()
        th = _theta(case, seed).requires_grad_(True)
        v = _faces(th, case["size"])
        b, target = _vector(n, seed + 1), _vector(n, seed + 2)
        x = _cg(cols, v.detach(), b)
        lam = _cg(cols, v.detach(), x - target)
        (g,) = torch.autograd.grad((lam * _mul(cols, v, x)).sum(), th)
        return dict(x=x, grad_theta=-g, grad_b=lam)
    cols, v, ok = _rows(case, seed)
    cols = torch.as_tensor(np.where(ok, cols, 0), device=DEV).long()
    v = torch.as_tensor(np.where(ok, v, 0.0), device=DEV)
    b = _vector(n, seed + 1, case["nrhs"] if kind == "batch" else None)
    if kind == "spmv":
        return _mul(cols, v, b)
    x = _cg(cols, v, b)
    if kind == "batch" or case["precision"] == 1:
        return dict(x=x, iterations=None)
    return dict(x=x, iterations=None, cond=None)
