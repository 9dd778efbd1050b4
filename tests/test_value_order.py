"""The differentiable assembly's entry order without a sort."""
import numpy as np
import pytest
import torch

from doug_amd.autograd import _diffusion_order, _diffusion_pattern, diffusion3d_values
from doug_amd import problems as P


@pytest.mark.parametrize("N", [1, 2, 3, 4, 7, 16])
def test_order_equals_the_sort(N):
    rows, cols, order = _diffusion_pattern(N)
    got = _diffusion_order(N, torch.device("cpu")).numpy()
    # entries of a matrix without repeated pairs: the sort has one answer
    assert np.array_equal(got, order)
    assert np.array_equal(rows[got], np.sort(rows))


def test_values_equal_the_generator():
    N = 6
    theta = torch.tensor(P.smoothed_gaussian(N, 3), dtype=torch.float64)
    _, _, _, v = P.diffusion3d(N, kappa=np.exp(P.smoothed_gaussian(N, 3)))
    np.testing.assert_allclose(diffusion3d_values(theta, N).numpy(), v, rtol=4e-16 * 8)
