"""Per-word kernels: increments staged in pairs (forward sweep) and twice over (lanes on paths, fp32), against the oracle."""
import random

import pytest
import torch

from oracle import tensor_oracle as TO

from .helpers import brownian_path, randn, rel_err

pytestmark = pytest.mark.gpu
TOL = {torch.float32: 1e-5, torch.float64: 1e-12}


# Forward tiles hold 16 KB of increments: 128 of them at 16 letters, 58 (fp64: 28) at 70, four (fp64: two) at 1024;
# lengths at both sides of a tile, odd and even, the shortest ones, and rows that fill a tile of their own.
@pytest.mark.parametrize("d,depth,L,windows", [
    (5, 4, 2, None), (5, 4, 3, None), (16, 4, 128, None), (16, 4, 129, None), (16, 4, 130, None), (16, 4, 132, None),
    (70, 2, 29, None), (70, 2, 30, None), (70, 2, 59, None), (70, 2, 60, None), (70, 2, 118, None), (2, 5, 10, None),
    (1024, 1, 2, None), (1024, 1, 3, None), (1024, 1, 6, None), (1024, 1, 7, None), (3, 7, 150, None), (2, 12, 40, None),
    (16, 3, 300, [(0, 300), (3, 4), (5, 134), (6, 6), (160, 291)])])
@pytest.mark.parametrize("dtype", [torch.float64, torch.float32])
def test_forward_tiles(set_option, dtype, d, depth, L, windows):
    import pathsig_amd as ps
    set_option("tiled", 0)
    rng = random.Random(d + L)
    words = sorted([tuple(rng.randrange(d) for _ in range(rng.randint(1, depth))) for _ in range(70)], key=len)
    proj = ps.projections.words(words, depth=depth, path_dim=d)
    path = brownian_path(2, L, d, seed=500 + d + L)
    want = TO.compute_signature(path, depth, proj.level_sizes, proj._codes, windows)
    module = ps.Signature(depth=depth, projection=proj,
                          windows=None if windows is None else torch.tensor(windows, device="cuda"))
    assert rel_err(module(path.to(dtype).cuda()), want) < TOL[dtype]


# Lanes on paths stage four increments at a time in fp32 and eight in fp64: lengths around one and two stages of either, around
# one group of sixteen paths, and alphabets whose staged increments fill a wave and do not.
@pytest.mark.parametrize("B", [15, 17])
@pytest.mark.parametrize("d", [2, 7, 16])
@pytest.mark.parametrize("L,dtype", [(L, torch.float32) for L in (2, 4, 5, 6, 9, 10)]
                         + [(L, torch.float64) for L in (2, 8, 9, 10, 16, 17, 18)])
def test_backward_stages(set_option, B, d, L, dtype):
    import pathsig_amd as ps
    set_option("tiled", 0)
    depth = 3
    rng = random.Random(d + L)
    words = sorted([tuple(rng.randrange(d) for _ in range(rng.randint(1, depth))) for _ in range(150)], key=len)
    proj = ps.projections.words(words, depth=depth, path_dim=d)
    path = brownian_path(B, L, d, seed=600 + d + L)
    want = TO.compute_signature(path, depth, proj.level_sizes, proj._codes)
    G = randn(tuple(want.shape), seed=61)
    x = path.to(dtype).cuda().requires_grad_(True)
    out = ps.Signature(depth=depth, projection=proj)(x)
    (grad,) = torch.autograd.grad(out, x, G.to(dtype).cuda())
    assert rel_err(out, want) < TOL[dtype]
    assert rel_err(grad, TO.signature_vjp(path, G, depth, proj.level_sizes, proj._codes)) < TOL[dtype]


# A lane per word (few paths), lanes on paths up to sixteen letters and above: the infinite gradient of one word reaches the
# letters of that word at every point and no others, which other words hold.
@pytest.mark.parametrize("dtype", [torch.float32, torch.float64])
@pytest.mark.parametrize("B,d", [(2, 6), (17, 6), (17, 20)])
def test_an_infinite_gradient_stays_with_its_letters(set_option, B, d, dtype):
    import pathsig_amd as ps
    set_option("tiled", 0)
    depth, L, word = 4, 12, (0, 2, 1, 0)
    rng = random.Random(7)
    others = {tuple(rng.randrange(3, d) for _ in range(rng.randint(2, depth))) for _ in range(60)}
    words = sorted({word, (2, 2, 1), (0,)} | others, key=lambda w: (len(w), w))
    proj = ps.projections.words(words, depth=depth, path_dim=d)
    x = brownian_path(B, L, d, seed=83).to(dtype).cuda().requires_grad_(True)
    out = ps.Signature(depth=depth, projection=proj)(x)
    G = randn(tuple(out.shape), seed=84).to(dtype).cuda()
    G[:, words.index(word)] = float("inf")
    (grad,) = torch.autograd.grad(out, x, G)
    assert torch.isfinite(grad[..., 3:]).all()
    assert not torch.isfinite(grad[..., :3]).any()
