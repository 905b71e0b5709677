"""Backward of word projections with lanes on paths over at most sixteen letters (batch_lists.hip): the entries of an
increment sorted by letter into rows, against the oracle."""
import random

import pytest
import torch

from oracle import tensor_oracle as TO

from .helpers import brownian_path, randn, rel_err

pytestmark = pytest.mark.gpu
TOL = {torch.float32: 1e-5, torch.float64: 1e-12}


@pytest.fixture(scope="module")
def ps():
    import pathsig_amd
    return pathsig_amd


def _words(kind, d, depth, count):
    rng = random.Random(31 * d + depth)
    if kind == "one_letter":  # every entry of a block falls to one letter: the most rows that a letter can take
        return [(d - 1,) * depth] * count
    words = [tuple(rng.randrange(d) for _ in range(rng.randint(max(1, depth - 2), depth))) for _ in range(count)]
    return sorted(words, key=len)


# paths: one short of a group, a group, one more, several; points: a single increment, tiles of two and stages of eight
# increments with and without a remainder; words: one, less than a lane's, more than a block's, at every number of
# words to a lane; one letter, sixteen, and numbers in between
@pytest.mark.parametrize("dtype", [torch.float64, torch.float32])
@pytest.mark.parametrize("kind,d,depth,B,L,count,windows", [
    ("random", 16, 4, 16, 17, 130, None), ("random", 16, 3, 17, 18, 200, None), ("random", 15, 2, 33, 9, 120, None),
    ("random", 5, 6, 15, 8, 67, None), ("random", 4, 5, 16, 10, 33, None), ("random", 3, 8, 12, 19, 40, None),
    ("random", 2, 12, 16, 25, 20, None), ("random", 9, 1, 40, 2, 9, None), ("random", 16, 2, 16, 3, 1, None),
    ("one_letter", 16, 3, 16, 27, 70, None), ("one_letter", 2, 6, 31, 11, 100, None), ("one_letter", 2, 4, 16, 70, 50, None),
    ("random", 6, 4, 18, 30, 90, [(0, 30), (3, 4), (5, 14), (9, 30), (7, 7)])])
def test_letter_rows(ps, set_option, dtype, kind, d, depth, B, L, count, windows):
    set_option("tiled", 0)
    proj = ps.projections.words(_words(kind, d, depth, count), depth=depth, path_dim=d)
    path = brownian_path(B, L, d, seed=860 + d)
    want = TO.compute_signature(path, depth, proj.level_sizes, proj._codes, windows)
    G = randn(tuple(want.shape), seed=86)
    want_grad = TO.signature_vjp(path, G, depth, proj.level_sizes, proj._codes, windows)
    module = ps.Signature(depth=depth, projection=proj,
                          windows=None if windows is None else torch.tensor(windows, device="cuda"))
    x = path.to(dtype).cuda().requires_grad_(True)
    out = module(x)
    (grad,) = torch.autograd.grad(out, x, G.to(dtype).cuda())
    assert rel_err(out, want) < TOL[dtype] and rel_err(grad, want_grad) < TOL[dtype]
    # without the chains that the forward kept
    alone = torch.ops.pathsig.signature_backward(
        x.detach(), out.detach(), G.to(dtype).cuda(), depth, True, module._encoded_words, module._level_sizes,
        windows is not None, module._windows)
    assert rel_err(alone, want_grad) < TOL[dtype]


@pytest.mark.parametrize("dtype", [torch.float64, torch.float32])
def test_infinite_points_stay_with_their_letter_and_path(ps, set_option, dtype):
    set_option("tiled", 0)
    d, depth, B = 4, 3, 20
    proj = ps.projections.words([(0, 1, 0), (2, 3, 3), (3, 2, 2), (1, 0, 1), (2, 2, 3)],
                                depth=depth, path_dim=d)
    module = ps.Signature(depth=depth, projection=proj)
    path = brownian_path(B, 21, d, seed=870).to(dtype).cuda()
    spoilt = path.clone()
    spoilt[5, 9, 0] = float("inf")
    G = randn((B, proj.sig_size), seed=87).to(dtype).cuda()
    grads = []
    for p in (path, spoilt):
        x = p.requires_grad_(True)
        grads.append(torch.autograd.grad(module(x), x, G)[0])
    assert rel_err(grads[1][..., 2:], grads[0][..., 2:]) < TOL[dtype]
    others = torch.arange(B, device="cuda") != 5
    assert rel_err(grads[1][others], grads[0][others]) < TOL[dtype]
    assert not torch.isfinite(grads[1][5, :, 0]).all()
