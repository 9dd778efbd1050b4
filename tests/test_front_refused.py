"""Subdomains whose work vector exceeds a workgroup's LDS: fewer workgroups for
all of them, or envelopes for all of them."""
import numpy as np
import pytest
import scipy.sparse as sp
import scipy.sparse.linalg as spl

import doug_amd as D
from doug_amd import problems as P

P1 = dict(levels=1, radius1=2, strong1=0.08, smoothers=1, overlap=0, symmstruct=1, symmnumeric=1)


@pytest.mark.gpu
@pytest.mark.parametrize("precision", [0, 1])
@pytest.mark.parametrize("edge", [18, 20, 22, 24])
def test_one_large_subdomain_beside_small_ones(edge, precision):
    # around the FP64 limit of 19,392 entries, of which 24^3 unknowns leave 5,568
    # for their updates; FP32 holds twice as many
    n0, i0, j0, v0 = P.diffusion3d(edge, 0.5, 11)
    n1, i1, j1, v1 = P.diffusion3d(7, 0.5, 12)
    sizes = [n1, n0, n1]
    off = np.r_[0, np.cumsum(sizes)]
    n = int(off[-1])
    i = np.concatenate([q + o for q, o in zip((i1, i0, i1), off)]).astype(np.int32)
    j = np.concatenate([q + o for q, o in zip((j1, j0, j1), off)]).astype(np.int32)
    v = np.concatenate([v1, v0, v1])
    A = sp.csc_matrix((v, (i - 1, j - 1)), shape=(n, n))
    r = np.random.default_rng(13).uniform(-1, 1, n)
    print(f"refused edge={edge} precision={precision}", flush=True)
    with D.Solver(0) as s:
        s.set_params(**P1)
        s.set_matrix(n, i, j, v, 1)
        s.set_subdomains(off.astype(np.int32), np.arange(n, dtype=np.int32), 0)
        s.setup(precision)
        z = s.prec(r)
    # residual of a backward stable solve: rounding of the factor's entries
    # times the front's depth (64 at most here), in the matrix's norm
    eps = 1.2e-7 if precision else 2.3e-16
    norm = np.abs(A).sum(axis=1).max()
    for a, b in zip(off, off[1:]):
        res = r[a:b] - (A @ z)[a:b]
        assert np.linalg.norm(res) <= 64 * eps * norm * np.linalg.norm(z[a:b]), (a, b)
