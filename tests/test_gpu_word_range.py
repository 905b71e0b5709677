"""Per-word kernels: what fits fp32 comes out in fp32, whatever the size of the increments and of the upstream gradient, also
where the factorials of the recurrences are what makes it fit.  Paths of one increment x, whose coefficient of the word
w_1 .. w_N is x_(w_1) .. x_(w_N) / N!."""
import math

import pytest
import torch

from .helpers import strict_rel_err

pytestmark = pytest.mark.gpu


# One increment of the same size in every letter and the word of all letters in turn: every place of a letter in the word has
# the gradient upstream * size^(N-1) / N!, which fits, while upstream * size^(N-1) does not.
# Two paths take the lanes on words, sixteen the lanes on paths (up to and above sixteen letters).
@pytest.mark.parametrize("B,d", [(2, 3), (16, 3), (16, 20)])
@pytest.mark.parametrize("depth,size,upstream", [(8, 1e5, 3e6), (6, 1e6, 1e10), (4, 1e8, 1e15)])
def test_gradient_of_large_increments(set_option, B, d, depth, size, upstream):
    import pathsig_amd as ps
    set_option("tiled", 0)
    word = tuple(k % d for k in range(depth))
    proj = ps.projections.words([word], depth=depth, path_dim=d)
    x = torch.zeros(B, 2, d)
    x[:, 1] = size
    x = x.cuda().requires_grad_(True)
    out = ps.Signature(depth=depth, projection=proj)(x)
    (grad,) = torch.autograd.grad(out, x, torch.full_like(out, upstream))
    one = upstream * size ** (depth - 1) / math.factorial(depth)
    assert upstream * size ** (depth - 1) > torch.finfo(torch.float32).max
    letters = torch.tensor([float(word.count(k)) for k in range(d)], dtype=torch.float64) * one
    want = torch.stack([-letters, letters]).expand(B, 2, d)
    # taking the step back leaves 2^-24 of each prefix value, which weighs binomial(N, m) in a gradient; 4 N roundings
    assert strict_rel_err(grad, want) < (2 ** depth + 4 * depth) * 2 ** -23
