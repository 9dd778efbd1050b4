"""The batched apply and solve of every fine level and method they accept,
column by column against the single-vector ones."""
import numpy as np
import pytest

import doug_amd as D
from doug_amd import problems as P

N = 8
CTL = dict(radius1=2, strong1=0.08, smoothers=1, overlap=1, symmstruct=1, symmnumeric=1)


def _compare(variant, nrhs):
    import torch

    n, i, j, v = P.diffusion3d(N, 1.0, 31)
    part = P.block_partition((N,) * 3, 4)
    R = np.random.default_rng(32).uniform(-1, 1, (n, nrhs))
    A = np.zeros((n, n))
    A[i - 1, j - 1] = v
    its, eps = 4, 1.1e-16
    # the two orders of summation: n terms at most, and the iterates carry
    # them on by the matrix's condition in each of the iterations
    bound = 2 * n * eps * its * np.linalg.cond(A)
    print(f"batch {variant} nrhs={nrhs} bound={bound:.1e}", flush=True)
    with D.Solver(0) as s:
        # the context's batch of another fine level comes first
        for ctl in (CTL, dict(CTL, **variant)):
            s.set_params(**ctl)
            s.set_matrix(n, i, j, v, 1)
            s.set_partition(*part)
            s.setup()
            s.prepare_batch()
        dR = torch.tensor(R, device="cuda:0")
        dZ = torch.full_like(dR, np.nan)
        s.prec_batch_device(nrhs, dR.data_ptr(), dZ.data_ptr())
        Z = dZ.cpu().numpy()
        X, count, hist = s.pcg_batch(R, 0.0, its)
        for k in range(nrhs):
            z = s.prec(R[:, k])
            assert np.linalg.norm(Z[:, k] - z) <= bound * np.linalg.norm(z)
            x, it, _, h = s.pcg(R[:, k], 0.0, its)
            assert it == count[k] == its
            assert np.all(np.abs(hist[:, k] - h) <= bound * np.linalg.norm(R[:, k]))
            assert np.linalg.norm(X[:, k] - x) <= bound * np.linalg.norm(x)


@pytest.mark.gpu
@pytest.mark.parametrize("nrhs", [1, 2, 5])
@pytest.mark.parametrize("variant", [dict(fine_method=0), dict(fine_method=0, levels=1), dict(levels=1),
                                     dict(method=5)])
def test_columns_equal_the_single_vector_path(variant, nrhs):
    _compare(variant, nrhs)


@pytest.mark.gpu
@pytest.mark.parametrize("nrhs", [1, 2, 5])
def test_without_a_preconditioner(nrhs):
    _compare(dict(method=0), nrhs)
