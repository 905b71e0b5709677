"""Backward of word projections with lanes on paths over more than sixteen letters (batch_kernels.hip), against the per-word
oracle: every compiled depth, groups of sixteen and of 32 paths, prefixes from the saved signature, kept by the forward
and rebuilt."""
import random

import pytest
import torch

from oracle import words_oracle as WO

from .helpers import brownian_path, randn, random_word_set, rel_err

pytestmark = pytest.mark.gpu
TOL = {torch.float32: 1e-5, torch.float64: 1e-12}


@pytest.fixture(scope="module")
def ps():
    import pathsig_amd
    return pathsig_amd


# paths: groups of sixteen (13, 37, 50) and of 32 (24, 30, 64), full and ragged; words up to every depth that is compiled
# on its own (3, 4, 6, 8, 12), fewer than a lane's and more than a block's; an alphabet that leaves one increment to a tile
WINDOWS = [(0, 25), (3, 5), (7, 7), (2, 19), (23, 25), (5, 24)]  # (the oracle takes them as they are: within every path)


@pytest.mark.parametrize("dtype", [torch.float64, torch.float32])
@pytest.mark.parametrize("d,depth,lo,count,full,B,L,windows,tile", [
    (17, 3, 3, 300, (1, 2), 24, 22, None, 0), (17, 4, 2, 250, (1,), 37, 19, None, 0), (33, 4, 4, 1, (), 13, 9, None, 0),
    (33, 6, 3, 120, (), 24, 12, None, 0), (17, 8, 5, 70, (), 30, 14, None, 0), (17, 12, 7, 40, (1,), 13, 11, None, 0),
    (33, 10, 9, 30, (), 64, 8, None, 0), (65, 5, 2, 80, (), 13, 10, None, 0), (33, 6, 2, 60, (1,), 24, 30, WINDOWS, 0),
    (17, 5, 3, 90, (), 50, 30, WINDOWS, 0), (17, 6, 3, 90, (1,), 24, 25, None, 1), (17, 4, 3, 90, (), 13, 25, WINDOWS, 3)])
def test_words_over_wide_alphabets(ps, set_option, dtype, d, depth, lo, count, full, B, L, windows, tile):
    set_option("tiled", 0)
    if tile:
        set_option("batch_tile", tile)
    words = random_word_set(d, lo, depth, count, seed=71)
    words = sorted([*words, *random.Random(72).sample(words, min(3, count))], key=len)  # (some of them twice)
    proj = ps.projections.words(words, depth=depth, path_dim=d, full_levels=full)
    path = brownian_path(B, L, d, seed=870 + d) * 2.0
    want = WO.sig_forward(path, depth, proj.level_sizes, proj._codes, windows)
    G = randn(tuple(want.shape), seed=87)
    want_grad = WO.sig_backward(path, want, G, depth, proj.level_sizes, proj._codes, windows)
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
