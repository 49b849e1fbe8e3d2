"""The FC-fit loss's gradient at many nodes, against the float64 loss: the
kernel in both orders of its workgroups, with remainders of the samples,
nodes and instances, and the batched product where few instances of many
nodes take it."""

import pytest
import torch

from test_gpu_fc_loss import _case
from tvb_hpc import autograd as AG

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize('M,N,P,bmm', [
    (37, 110, 70, False),     # node groups of a sample tile together
    (37, 111, 70, False),     # sample tiles of a node group together
    (50, 117, 65, False),
    (33, 200, 130, False),
    (40, 300, 3, True),
    (35, 257, 1, True)])
def test_gradient_matches_float64_torch(M, N, P, bmm):
    assert AG._grad_by_bmm(M, N, P) == bmm
    x, tgt, gout = _case(M, N, P, False, seed=M + N + P)
    xr = x.double().requires_grad_(True)
    (AG.fc_loss(xr, tgt) * gout).sum().backward()
    xd = x.clone().requires_grad_(True)
    (AG.fc_loss_device(xd, tgt).double() * gout).sum().backward()
    torch.cuda.synchronize()
    err = (xd.grad.double() - xr.grad).abs().max() / xr.grad.abs().max()
    # float32 products of the gradient against float64 autograd
    assert err.item() <= 1e-4
