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


@pytest.mark.gpu
@pytest.mark.parametrize("precision", [0, 1])
def test_batch_keeps_its_bits(precision):
    # uneven subdomains, smallest first: both dispatch orders are timed for the
    # fronts and for the batch's own factors
    import torch

    n, i, j, v = P.diffusion3d(16, 1.0, 6)
    cut = np.array([0, 256, 1024, 2048, n], np.int32)
    with D.Solver(0) as s:
        s.set_params(**P1)
        s.set_matrix(n, i, j, v, 1)
        s.set_subdomains(cut, np.arange(n, dtype=np.int32), 0)
        R = torch.tensor(np.random.default_rng(7).uniform(-1, 1, (n, 5)), device="cuda:0")
        Z = []
        for step in range(3):
            if step != 1:  # set-up, tuned, set up again with the choice kept
                s.setup(precision)
                s.prepare_batch()
            else:
                s.autotune(4)
            Z.append(torch.zeros_like(R))
            s.prec_batch_device(5, R.data_ptr(), Z[-1].data_ptr())
        assert torch.equal(Z[0], Z[1]) and torch.equal(Z[0], Z[2])
        z = s.prec(R[:, 2].cpu().numpy())
        # rounding of one application: n terms, the blocks' condition below 2e3
        assert np.linalg.norm(Z[0][:, 2].cpu().numpy() - z) <= (1.2e-7 if precision else 2.3e-16) * 64 * 2e3 * np.linalg.norm(z)
