"""Per-increment sums over the letters in the reverse sweep, against the oracle: the lanes leave their terms in a slab
in LDS (fp32 up to fifteen letters, fp64 over the alphabets where that is the faster way) or exchange them."""
import pytest
import torch

from oracle import tensor_oracle as TO

from .helpers import brownian_path, randn, rel_err

pytestmark = pytest.mark.gpu
TOL = {torch.float32: 1e-5, torch.float64: 1e-12}


# Alphabets on both sides of every padding of the slab (2, 4, 8, 16 letters), blocks of one to eight waves; lengths around
# the increments that wait in the slab (1 to 8) and the tiles of 8, 16 and 32 increments; time chunks with a ghost step.
@pytest.mark.parametrize("d,depth,dtype", [(8, 5, torch.float32), (7, 5, torch.float32), (2, 4, torch.float64),
                                           (3, 3, torch.float64), (7, 4, torch.float64), (8, 3, torch.float64),
                                           (8, 5, torch.float64), (10, 3, torch.float64), (12, 2, torch.float64),
                                           (15, 3, torch.float64), (9, 3, torch.float32), (10, 4, torch.float32),
                                           (15, 3, torch.float32), (15, 2, torch.float32), (12, 3, torch.float64),
                                           (9, 2, torch.float64), (2, 8, torch.float64), (11, 5, torch.float32),
                                           (13, 5, torch.float32)])
@pytest.mark.parametrize("L,chunks", [(2, 1), (8, 1), (10, 1), (34, 1), (35, 3), (65, 2)])
def test_lengths_around_the_tiles(set_option, d, depth, dtype, L, chunks):
    import pathsig_amd as ps
    set_option("chunks", chunks)
    B = 2
    path = brownian_path(B, L, d, seed=40 + d + L)
    want = TO.signature(path, depth)
    G = randn(tuple(want.shape), seed=41)
    x = path.to(dtype).cuda().requires_grad_(True)
    out = ps.Signature(depth=depth)(x)
    (grad,) = torch.autograd.grad(out, x, G.to(dtype).cuda())
    assert rel_err(out, want) < TOL[dtype]
    assert rel_err(grad, TO.signature_vjp(path, G, depth)) < TOL[dtype]


# (fp64 over two, nine and twelve letters: windows and rows in one piece exchange, rows in chunks take the slab)
@pytest.mark.parametrize("d,depth,dtype", [(8, 5, torch.float32), (8, 4, torch.float64), (2, 5, torch.float64),
                                           (11, 3, torch.float64), (2, 8, torch.float64), (9, 2, torch.float64),
                                           (12, 3, torch.float64), (14, 4, torch.float32), (15, 4, torch.float32),
                                           (11, 5, torch.float32)])
@pytest.mark.parametrize("chunks", [1, 2])
def test_overlapping_windows(set_option, d, depth, dtype, chunks):
    import pathsig_amd as ps
    set_option("chunks", chunks)
    B, L = 2, 40
    path = brownian_path(B, L, d, seed=60 + d)
    spans = [(0, 40), (3, 20), (5, 5), (7, 8), (11, 29)]
    x = path.to(dtype).cuda().requires_grad_(True)
    out = ps.Signature(depth=depth, windows=torch.tensor(spans, device="cuda"))(x)
    G = randn(tuple(out.shape), seed=61)
    (grad,) = torch.autograd.grad(out, x, G.to(dtype).cuda())
    want = torch.zeros_like(path)
    for w, (start, end) in enumerate(spans):
        if end - start > 1:
            want[:, start:end] += TO.signature_vjp(path[:, start:end], G[:, w], depth)
    assert rel_err(grad, want) < TOL[dtype]


# (Not fp32 shapes whose prefix letters times letters are 24 at most, like (8, 5) and (4, 6): there the terms of a prefix are
# multiplied by zeros and ones to reach their letters, and an infinite one turns the other letters' sums into NaN.)
@pytest.mark.parametrize("d,depth,dtype", [(14, 3, torch.float32), (15, 3, torch.float32), (12, 4, torch.float32),
                                           (8, 4, torch.float64)])
def test_an_infinite_gradient_stays_with_its_letters(d, depth, dtype):
    import pathsig_amd as ps
    L, word = 12, [0, 2, 1, 0][:depth]
    x = brownian_path(1, L, d, seed=80 + d).to(dtype).cuda().requires_grad_(True)
    out = ps.Signature(depth=depth)(x)
    G = randn(tuple(out.shape), seed=81).to(dtype).cuda()
    column = sum(d ** k for k in range(1, depth))
    for k, letter in enumerate(word):
        column += letter * d ** (depth - 1 - k)
    G[0, column] = float("inf")
    (grad,) = torch.autograd.grad(out, x, G)
    # the words of the other letters do not meet this gradient; its own letters all do, at every point
    assert torch.isfinite(grad[..., 3:]).all()
    assert not torch.isfinite(grad[..., :3]).any()
