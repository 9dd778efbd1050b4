"""Frontal solves subdomain by subdomain, with fronts for every wavefront and
workgroup of each split, and the batch beside them."""
import numpy as np
import pytest
import scipy.sparse as sp
import scipy.sparse.linalg as spl

import doug_amd as D

P1 = dict(levels=1, radius1=2, strong1=0.08, smoothers=1, overlap=0, symmstruct=1, symmnumeric=1)
EPS = {0: 2.3e-16, 1: 1.2e-7}


def _grid(dims, rng):
    """1-based entries of a weighted grid Laplacian plus one."""
    idx = np.arange(int(np.prod(dims))).reshape(dims)
    pairs = [(np.moveaxis(idx, a, 0)[:-1].ravel(), np.moveaxis(idx, a, 0)[1:].ravel()) for a in range(len(dims))]
    lo, hi = (np.concatenate(x) for x in zip(*pairs))
    w = rng.uniform(0.5, 1.5, lo.size)
    n = idx.size
    d = 1.0 + np.bincount(lo, w, n) + np.bincount(hi, w, n)
    i = np.r_[np.arange(n), lo, hi].astype(np.int32) + 1
    j = np.r_[np.arange(n), hi, lo].astype(np.int32) + 1
    return n, i, j, np.r_[d, -w, -w]


def _bound(A, precision):
    # the rows' dominance by one bounds a block's inverse by one in the maximum
    # norm, so its condition is at most twice its largest diagonal entry; each
    # of the front tree's levels (below 24 here) rounds once more
    return 24 * EPS[precision] * 2.0 * A.diagonal().max()


@pytest.mark.gpu
@pytest.mark.parametrize("precision", [0, 1])
@pytest.mark.parametrize("dims,parts", [((21, 20, 20), 3), ((24, 24, 24), 20), ((32, 32, 32), 64), ((40, 28, 30), 100),
                                        ((44, 32, 32), 150), ((33, 32, 32), 300), ((150, 150), 12), ((180, 170), 56),
                                        ((260, 210), 110)])
def test_each_subdomain_in_the_maximum_norm(dims, parts, precision):
    rng = np.random.default_rng(parts)
    n, i, j, v = _grid(dims, rng)
    A = sp.csr_matrix((v, (i - 1, j - 1)), shape=(n, n))
    r = rng.uniform(-1, 1, n)
    side = max(2, int(round((n / parts) ** (1 / len(dims)))))
    cell = np.zeros(dims, np.int64)
    for a, m in enumerate(dims):
        k = np.arange(m) // side
        cell = cell * int(k[-1] + 1) + k.reshape([-1 if q == a else 1 for q in range(len(dims))])
    _, cell = np.unique(cell.ravel(), return_inverse=True)
    order = np.argsort(cell, kind="stable").astype(np.int32)
    starts = np.searchsorted(cell[order], np.arange(cell.max() + 2)).astype(np.int32)
    print(f"accuracy {dims} subdomains={len(starts) - 1} of up to {np.diff(starts).max()} precision={precision}", flush=True)
    with D.Solver(0) as s:
        s.set_params(**P1)
        s.set_matrix(n, i, j, v, 1)
        s.set_subdomains(starts, order, 0)
        s.setup(precision)
        z = s.prec(r)
    bound = _bound(A, precision)
    for a, b in zip(starts, starts[1:]):
        q = order[a:b]
        x = spl.spsolve(A[np.ix_(q, q)].tocsc(), r[q])
        assert np.abs(z[q] - x).max() <= bound * np.abs(x).max(), (a, b)


@pytest.mark.gpu
@pytest.mark.parametrize("precision", [0, 1])
def test_repeated_pairs_and_the_batch(precision):
    # every entry in two parts, some in three: the host's map sums them for the
    # fronts and again for the batch's envelopes
    import torch

    rng = np.random.default_rng(61)
    n, i, j, v = _grid((12, 13, 14), rng)
    A = sp.csr_matrix((v, (i - 1, j - 1)), shape=(n, n))
    pick = np.arange(0, v.size, 3)
    third = np.zeros_like(v)
    third[pick] = 0.25 * v[pick]
    ii, jj, vv = np.r_[i, i, i[pick]], np.r_[j, j, j[pick]], np.r_[0.5 * v, 0.5 * v - third, third[pick]]
    mix = rng.permutation(vv.size)
    starts = np.array([0, 700, 1400, n], np.int32)
    R = rng.uniform(-1, 1, (n, 3))
    with D.Solver(0) as s:
        s.set_params(**P1)
        s.set_matrix(n, ii[mix], jj[mix], vv[mix], 1)
        s.set_subdomains(starts, np.arange(n, dtype=np.int32), 0)
        s.setup(precision)
        s.prepare_batch()
        dR = torch.tensor(R, device="cuda:0")
        dZ = torch.zeros_like(dR)
        s.prec_batch_device(3, dR.data_ptr(), dZ.data_ptr())
        Z = dZ.cpu().numpy()
        single = np.stack([s.prec(R[:, k]) for k in range(3)], axis=1)
    bound = _bound(A, precision)
    # (the envelopes round along rows of up to 700 entries instead of a tree)
    loose = bound * 700 / 24
    for a, b in zip(starts, starts[1:]):
        lu = spl.splu(A[a:b, a:b].tocsc())
        for k in range(3):
            x = lu.solve(R[a:b, k])
            assert np.abs(single[a:b, k] - x).max() <= bound * np.abs(x).max()
            assert np.abs(Z[a:b, k] - x).max() <= loose * np.abs(x).max()
