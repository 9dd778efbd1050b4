"""Frontal solves of several contexts that live side by side."""
import numpy as np
import pytest

import doug_amd as D
from doug_amd import problems as P

P1 = dict(levels=1, radius1=2, strong1=0.08, smoothers=1, overlap=0, symmstruct=1, symmnumeric=1)


def _one_subdomain(N):
    n, i, j, v = P.diffusion3d(N, 1.0, 3)
    s = D.Solver(0)
    s.set_params(**P1)
    s.set_matrix(n, i, j, v, 1)
    s.set_subdomains(np.array([0, n], np.int32), np.arange(n, dtype=np.int32), 0)
    return s, np.random.default_rng(N).uniform(-1, 1, n)


@pytest.mark.gpu
@pytest.mark.parametrize("order", [0, 1])
@pytest.mark.parametrize("precision", [0, 1])
def test_a_smaller_context_leaves_the_larger_one_its_lds(precision, order):
    # work vectors of 18^3 and 16^3 unknowns (FP64: 108 and 74 KB, envelopes
    # 47 and 33 KB): the second set-up must not lower what the first may take
    print(f"contexts precision={precision} order={order}", flush=True)
    large, r = _one_subdomain(18)
    small, q = _one_subdomain(16)
    with large, small:
        for s in (large, small):
            s.set_option(4, order)
        large.setup(precision)
        z = large.prec(r)
        small.setup(precision)
        y = small.prec(q)
        assert np.array_equal(large.prec(r), z)
        assert np.array_equal(small.prec(q), y)
        assert np.linalg.norm(z) > 0 and np.linalg.norm(y) > 0
