"""doug_autotune's dispatch orders where equal unknown counts hide unequal work."""
import numpy as np
import pytest

import doug_amd as D
from doug_amd import problems as P

P1 = dict(levels=1, radius1=2, strong1=0.08, smoothers=1, overlap=0, symmstruct=1, symmnumeric=1)
N = 8


@pytest.mark.gpu
@pytest.mark.parametrize("chain_first", [True, False])
def test_largest_first_goes_by_the_factors(chain_first):
    # a chain and a box of 512 unknowns each: the box's fronts hold several
    # times the chain's entries, so largest first differs from chain, box only
    m = N ** 3
    _, i, j, v = P.diffusion3d(N, 1.0, 4)
    k = np.arange(1, m + 1, dtype=np.int32)
    ci = np.r_[k, k[1:], k[:-1]]
    cj = np.r_[k, k[:-1], k[1:]]
    cv = np.r_[np.full(m, 3.0), np.full(2 * (m - 1), -1.0)]
    a, b = (m, 0) if not chain_first else (0, m)  # offsets of the chain, of the box
    with D.Solver(0) as s:
        s.set_params(**P1)
        s.set_matrix(2 * m, np.r_[ci + a, i + b], np.r_[cj + a, j + b], np.r_[cv, v], 1)
        s.set_subdomains(np.array([0, m, 2 * m], np.int32), np.arange(2 * m, dtype=np.int32), 0)
        s.setup()
        tune = s.autotune(4)
        r = np.random.default_rng(5).uniform(-1, 1, 2 * m)
        z = s.prec(r)
        assert (tune["trsv_ms"][1] > 0) == chain_first
        for order in (0, 1):  # either order gives the same bits
            s.set_option(3, order)
            assert np.array_equal(s.prec(r), z)
