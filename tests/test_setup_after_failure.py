"""A set-up after one that failed on the same context."""
import numpy as np
import pytest

import doug_amd as D
from doug_amd import problems as P

CTL = dict(radius1=2, strong1=0.08, smoothers=1, overlap=1, symmstruct=1, symmnumeric=1)
N = 16


def _ranks():
    st, nd = P.block_partition((N,) * 3, 8)
    rank = np.zeros(N ** 3, np.int32)
    for r in range(len(st) - 1):
        rank[nd[st[r] - 1:st[r + 1] - 1] - 1] = r + 1
    return len(st) - 1, rank


@pytest.mark.gpu
@pytest.mark.parametrize("precision", [0, 1])
def test_same_bits_as_a_new_context(precision):
    # a decomposition over processes whose subdomains are not positive definite
    # leaves its work on other streams than the one-process set-up that follows
    n, i, j, v = P.diffusion3d(N, 1.0, 51)
    bad = np.where((i == j) & (i % 64 == 0), -v, v)
    r = np.random.default_rng(52).uniform(-1, 1, n)
    part = P.block_partition((N,) * 3, 8)

    def good(s):
        s.set_params(**CTL)
        s.set_matrix(n, i, j, v, 1)
        s.set_partition(*part)
        s.setup(precision)
        return s.prec(r)

    with D.Solver(0) as s:
        z = good(s)
    with D.Solver(0) as s:
        for _ in range(3):
            s.set_params(**CTL)
            s.set_matrix(n, i, j, bad, 1)
            s.set_partition(np.ones(1, np.int32), np.zeros(0, np.int32))
            s.set_ranks(*_ranks())
            with pytest.raises(D.DougError):
                s.setup(precision)
            s.set_ranks(0, None)
            assert np.array_equal(good(s), z)
