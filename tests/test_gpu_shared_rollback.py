"""Reverse sweep: the signature is taken back inside the adjoint of a step, or in a pass of its own (rows of more than 4096
increments in time chunks in fp32; shapes whose state would not fit the registers; wide alphabets).  Both sides of that
length and rows that are not cut, against the oracle."""
import pytest
import torch

from oracle import tensor_oracle as TO

from .helpers import brownian_path, randn, rel_err

pytestmark = pytest.mark.gpu


# A gradient of the path is the difference of sums that are rounded to 6e-8 of themselves and sqrt(L) times larger:
# 6e-8 * sqrt(2) * sqrt(4097) = 5.4e-6, and no more than as much again from the roundings that the state gathers.
# In chunks, in one piece and as one window, which is added to the gradient of the path.
@pytest.mark.parametrize("how", ["chunks", "one piece", "window"])
@pytest.mark.parametrize("d,depth", [(2, 3), (3, 4), (4, 6)])
@pytest.mark.parametrize("L", [4096, 4097, 4098])
def test_both_sides_of_the_length(set_option, d, depth, L, how):
    import pathsig_amd as ps
    if how == "one piece":
        set_option("chunks", 1)
    path = brownian_path(1, L, d, seed=77 + d).float().double()
    want = TO.signature(path, depth)
    G = randn(tuple(want.shape), seed=78).float().double()
    x = path.float().cuda().requires_grad_(True)
    windows = torch.tensor([[0, L]], device="cuda") if how == "window" else None
    out = ps.Signature(depth=depth, windows=windows)(x).reshape(want.shape)
    (grad,) = torch.autograd.grad(out, x, G.float().cuda())
    want_grad = TO.signature_vjp(path, G, depth)
    assert rel_err(out, want) < 1e-5
    diff = (grad.cpu().double() - want_grad).norm() / want_grad.norm()
    assert float(diff) < 1.1e-5


# Shapes on either side of the rule, in one piece, in chunks and in overlapping windows.
@pytest.mark.parametrize("d,depth,dtype", [(14, 4, torch.float32), (15, 4, torch.float32), (8, 5, torch.float64),
                                           (8, 6, torch.float64), (11, 5, torch.float64), (17, 3, torch.float32),
                                           (28, 3, torch.float64), (24, 4, torch.float64)])
@pytest.mark.parametrize("how", ["one piece", "chunks", "windows"])
def test_shapes_taken_back_either_way(set_option, d, depth, dtype, how):
    import pathsig_amd as ps
    set_option("chunks", 2 if how == "chunks" else 1)
    B, L = 2, 12
    path = brownian_path(B, L, d, seed=90 + d)
    spans = [(0, 12), (3, 9), (5, 6)] if how == "windows" else [(0, 12)]
    x = path.to(dtype).cuda().requires_grad_(True)
    out = ps.Signature(depth=depth, windows=torch.tensor(spans, device="cuda") if how == "windows" else None)(x)
    G = randn((B, len(spans), out.shape[-1]), seed=91)
    (grad,) = torch.autograd.grad(out, x, G.reshape(out.shape).to(dtype).cuda())
    want = torch.zeros_like(path)
    for w, (start, end) in enumerate(spans):
        if end - start > 1:
            want[:, start:end] += TO.signature_vjp(path[:, start:end], G[:, w], depth)
    assert rel_err(grad, want) < (1e-5 if dtype == torch.float32 else 1e-12)
