"""Frontal subdomain factors: the host's patterns and schedules run on the
CPU, and the GPU's factor and solve against the assembled subdomains."""
import os
import subprocess

import numpy as np
import pytest
import scipy.sparse as sp
import scipy.sparse.linalg as spl

import doug_amd as D
from doug_amd import problems as P

P1 = dict(levels=1, radius1=2, strong1=0.08, smoothers=1, overlap=0, symmstruct=1, symmnumeric=1)
ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))


def test_patterns_and_schedules(tmp_path):
    src = os.path.join(ROOT, "doug_amd", "csrc")
    exe = str(tmp_path / "fronts_check")
    subprocess.run(["g++", "-O1", "-std=c++17", "-pthread", "-I", src, "-o", exe,
                    os.path.join(ROOT, "tests", "fronts_check.cpp"), os.path.join(src, "doug_fronts.cpp"),
                    os.path.join(src, "doug_setup.cpp")], check=True)
    r = subprocess.run([exe], capture_output=True, text=True, timeout=300)
    assert r.returncode == 0, r.stdout


def _graph(kind, rng):
    """COO (1-based, both triangles) of a graph's weighted Laplacian plus one:
    symmetric, dominant by 1, so that its condition is at most 2 max(a_ii)."""
    if kind.startswith("box"):
        dims = [int(x) for x in kind[3:].split("x")]
        idx = np.arange(int(np.prod(dims))).reshape(dims)
        pairs = [(np.moveaxis(idx, a, 0)[:-1].ravel(), np.moveaxis(idx, a, 0)[1:].ravel())
                 for a in range(len(dims)) if dims[a] > 1]
        n = idx.size
    else:
        n, deg, parts, hub = {"components": (500, 2, 7, 0), "hub": (400, 1, 5, 1), "dense": (130, 110, 1, 1)}[kind]
        i = np.repeat(np.arange(n), deg)
        j = (i + rng.integers(0, max(2, n // 20) if kind != "dense" else n, i.size)) % n
        j = j - j % parts + i % parts
        pairs = [(i, np.minimum(j, n - 1))]
        if hub:
            pairs.append((np.zeros(n - 1, int), np.arange(1, n)))
    i = np.concatenate([a for a, _ in pairs] or [np.zeros(0, int)])
    j = np.concatenate([b for _, b in pairs] or [np.zeros(0, int)])
    keep = i != j
    lo, hi = np.minimum(i, j)[keep], np.maximum(i, j)[keep]
    e = np.unique(lo * n + hi)
    lo, hi = e // n, e % n
    w = -rng.uniform(0.5, 1.5, lo.size)
    A = sp.coo_matrix((np.r_[w, w], (np.r_[lo, hi], np.r_[hi, lo])), shape=(n, n)).tocsr()
    A = (A + sp.diags(1.0 - np.asarray(A.sum(axis=1)).ravel())).tocoo()
    return n, A.row.astype(np.int32) + 1, A.col.astype(np.int32) + 1, A.data


@pytest.mark.gpu
@pytest.mark.parametrize("precision", [0, 1])
@pytest.mark.parametrize("kind", ["box1", "box3", "box31", "box33", "box4x4x4", "box65", "box9x9", "box7x9x11",
                                  "box16x16x16", "box1500", "components", "hub", "dense"])
def test_solves_the_subdomains(kind, precision):
    # one-level preconditioner: z = sum over subdomains of A_ii^-1 r, with the
    # whole system as one subdomain and cut in three; frontal factors (order 1)
    # and envelopes (order 0), the entries placed by the device and by the host
    rng = np.random.default_rng(7)
    n, i, j, v = _graph(kind, rng)
    A = sp.csr_matrix((v, (i - 1, j - 1)), shape=(n, n))
    r = rng.uniform(-1, 1, n)
    eps = 1.2e-7 if precision else 2.3e-16
    bound = eps * max(n, 64) * 2.0 * A.diagonal().max()
    print(f"fronts {kind} precision={precision} n={n}", flush=True)
    # workgroups per subdomain: eight up to 32 subdomains, four up to 64, two up to 128
    for parts in (1, 3, 50, 100, 150) if n >= 1500 else (1, 3) if n >= 3 else (1,):
        cut = np.linspace(0, n, parts + 1).astype(int)
        sets = [np.arange(cut[p], cut[p + 1]) for p in range(parts)]
        z = np.zeros(n)
        for q in sets:
            z[q] += spl.spsolve(A[np.ix_(q, q)].tocsc(), r[q])
        for order, device in ((1, 1), (1, 0), (0, 1)):
            with D.Solver(0) as s:
                s.set_option(4, order)
                s.set_option(7, device)
                s.set_params(**P1)
                s.set_matrix(n, i, j, v, 1)
                s.set_subdomains(np.r_[0, np.cumsum([len(q) for q in sets])].astype(np.int32),
                                 np.concatenate(sets).astype(np.int32), 0)
                s.setup(precision)
                got = s.prec(r)
            assert np.linalg.norm(got - z) <= bound * np.linalg.norm(z), (parts, order, device)
