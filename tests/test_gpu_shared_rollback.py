"""Reverse sweep: the signature is taken back inside the adjoint of a step; fp32 rows of more than 4096 increments take it back
in a pass of its own.  Both sides of that length, against the CPU checker."""
import pytest
import torch

from oracle import tensor_oracle as TO

from .helpers import brownian_path, randn, rel_err

pytestmark = pytest.mark.gpu


# A gradient of the path is the difference of sums that are rounded to 6e-8 of themselves and sqrt(L) times larger:
# 6e-8 * sqrt(2) * sqrt(4097) = 5.4e-6, and a few roundings of that size per sum.
@pytest.mark.parametrize("d,depth", [(2, 3), (3, 4), (4, 6)])
@pytest.mark.parametrize("L", [4096, 4097, 4098])
def test_both_sides_of_the_length(d, depth, L):
    import pathsig_amd as ps
    path = brownian_path(1, L, d, seed=77 + d).float().double()
    want = TO.signature(path, depth)
    G = randn(tuple(want.shape), seed=78).float().double()
    x = path.float().cuda().requires_grad_(True)
    out = ps.Signature(depth=depth)(x)
    (grad,) = torch.autograd.grad(out, x, G.float().cuda())
    want_grad = TO.signature_vjp(path, G, depth)
    assert rel_err(out, want) < 1e-5
    diff = (grad.cpu().double() - want_grad).norm() / want_grad.norm()
    assert float(diff) < 2.5e-5
