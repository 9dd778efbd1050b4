"""PCG's scalars where the vector kernels sum the partials themselves (up to
1024 of 256 unknowns each) and just above, where a launch of its own does."""
import numpy as np
import pytest
import scipy.linalg as sl

import doug_amd as D

P1 = dict(levels=1, radius1=2, strong1=0.08, smoothers=1, overlap=0, symmstruct=1, symmnumeric=1)


def _pcg(mul, prec, b, its):
    x, r, p, rho, hist = np.zeros_like(b), b.copy(), None, 0.0, []
    for _ in range(its):
        z = prec(r)
        rho, old = r @ z, rho
        p = z if p is None else z + rho / old * p
        q = mul(p)
        a = rho / (p @ q)
        x, r = x + a * p, r - a * q
        hist.append(np.linalg.norm(r))
    return x, np.array(hist)


@pytest.mark.gpu
@pytest.mark.parametrize("method", [0, 1])
@pytest.mark.parametrize("n", [300, 1025, 65537, 262144, 262145])
def test_iterates(n, method):
    # a weighted chain plus one (condition at most 7), blocks of 512 as subdomains
    rng = np.random.default_rng(n)
    w = rng.uniform(0.5, 1.5, n - 1)
    d = 1.0 + np.r_[w, 0.0] + np.r_[0.0, w]
    k = np.arange(1, n, dtype=np.int32)
    i = np.r_[np.arange(1, n + 1, dtype=np.int32), k, k + 1]
    j = np.r_[np.arange(1, n + 1, dtype=np.int32), k + 1, k]
    b = rng.uniform(-1, 1, n)
    cut = np.r_[np.arange(0, n, 512), n].astype(np.int32)
    inner = w.copy()
    inner[cut[1:-1] - 1] = 0.0  # no coupling between two subdomains
    band = np.vstack([d, np.r_[-inner, 0.0]])

    def mul(x):
        y = d * x
        y[:-1] -= w * x[1:]
        y[1:] -= w * x[:-1]
        return y

    its = 6
    x, hist = _pcg(mul, (lambda r: sl.solveh_banded(band, r, lower=True)) if method else (lambda r: r.copy()), b, its)
    print(f"folded sums n={n} method={method}", flush=True)
    with D.Solver(0) as s:
        s.set_params(method=method, **P1)
        s.set_matrix(n, i, j, np.r_[d, -w, -w], 1)
        s.set_subdomains(cut, np.arange(n, dtype=np.int32), 0)
        s.setup(0)
        for _ in range(2):  # the second call starts from the first one's scalars
            got, done, _, h = s.pcg(b, 0.0, its)
            assert done == its
            # rounding per iteration: sums of depth 30 and three vector updates,
            # times the condition, and as much again carried on by each
            # iteration: 2 * 6 * 33 * 7 * 6 * 1.1e-16 = 1.8e-12
            assert np.all(np.abs(h - hist) <= 2e-12 * np.linalg.norm(b)), (h, hist)
            assert np.linalg.norm(got - x) <= 2e-12 * np.linalg.norm(x)
