"""The differentiable assembly on tensors without data, and under transforms."""
import pytest
import torch
from torch._subclasses.fake_tensor import FakeTensorMode

from doug_amd.autograd import diffusion3d_values

N = 3


def _fake(t):
    with FakeTensorMode() as mode:
        return diffusion3d_values(mode.from_tensor(t), N)


@pytest.mark.parametrize("call", [_fake, lambda t: diffusion3d_values(t.to("meta"), N)], ids=["fake", "meta"])
def test_shapes_without_data(call):
    out = call(torch.zeros(N ** 3, dtype=torch.float64))
    assert out.shape == (7 * N ** 3 - 6 * N * N,) and out.dtype == torch.float64


def test_transforms_agree():
    f = lambda t: diffusion3d_values(t, N)
    theta = torch.linspace(-1, 1, N ** 3, dtype=torch.float64)
    rev = torch.func.jacrev(f)(theta)
    # the same derivative by another order of the same few operations
    torch.testing.assert_close(torch.func.jacfwd(f)(theta), rev, rtol=1e-14, atol=1e-14)
    many = torch.stack([theta, -theta])
    assert torch.equal(torch.func.vmap(f)(many), torch.stack([f(t) for t in many]))
    assert torch.equal(torch.compile(f, backend="eager", fullgraph=True)(theta), f(theta))
