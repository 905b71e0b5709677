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


# A word that begins with an increment close to the smallest normal float, the others large: its value is an ordinary number,
# and the values on the way to it are not smaller than that increment over the first two divisors of the recurrence,
# 1.2e-38 / 56 = 1.5e5 steps of the smallest float: relative 3e-6, and 1e-6 of ordinary roundings.
@pytest.mark.parametrize("depth,size", [(8, 1e4), (6, 1e5)])
def test_value_of_a_word_that_begins_small(set_option, depth, size):
    import pathsig_amd as ps
    set_option("tiled", 0)
    B, d = 40, 3
    proj = ps.projections.words([(0,) + (1,) * (depth - 1)], depth=depth, path_dim=d)
    path = torch.zeros(B, 2, d)
    path[:, 1, 0] = torch.logspace(math.log10(1.2e-38), -36, B, dtype=torch.float64).float()
    path[:, 1, 1] = size
    out = ps.Signature(depth=depth, projection=proj)(path.cuda())[:, 0].double().cpu()
    want = path[:, 1, 0].double() * size ** (depth - 1) / math.factorial(depth)
    assert float(((out - want).abs() / want).max()) < 1e-5
