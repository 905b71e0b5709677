"""Log-signatures of few rows of large layouts: adjoint in a launch per level, products over the top level split between
blocks, the level below the top shared by blocks."""
import pytest
import torch

from oracle import tensor_oracle as TO

from .helpers import brownian_path, randn, rel_err

pytestmark = pytest.mark.gpu
TOL = {torch.float32: 1e-5, torch.float64: 1e-12}


# words of a level around the groups of lanes (1, 4, .., a wave, the block of 256); layouts whose adjoint does not fit a block's
# LDS in fp64 alone, and in both types; rows that split the products over the top level and rows that do not; depth 12
@pytest.mark.parametrize("dtype", [torch.float64, torch.float32])
@pytest.mark.parametrize("rows,d,depth", [(1, 7, 5), (3, 8, 5), (130, 8, 5), (1, 9, 5), (2, 6, 6), (5, 5, 6), (2, 3, 9), (1, 34, 3),
                                          (70, 6, 6), (1, 2, 12)])
def test_operators(dtype, rows, d, depth):
    import pathsig_amd  # noqa: F401
    sig = TO.signature(brownian_path(rows, 12, d, seed=1200 + d) * 1.5, depth)
    top = d ** depth
    want, powers = TO.sig_to_logsig(sig, depth, d, top, None)
    G = randn(tuple(sig.shape), seed=121)
    want_grad = TO.logsig_vjp(sig, G, depth, d, top, None)
    x = sig.to(dtype).cuda().requires_grad_(True)
    none = torch.empty(0, dtype=torch.int64, device="cuda")
    got = torch.ops.pathsig.sig_to_logsig(x, depth, d, False, none, [0] + [d ** k for k in range(1, depth + 1)])[0]
    assert rel_err(got, want) < TOL[dtype]
    (grad,) = torch.autograd.grad(got, x, G.to(dtype).cuda())
    assert rel_err(grad, want_grad) < TOL[dtype]


@pytest.mark.parametrize("dtype", [torch.float64, torch.float32])
@pytest.mark.parametrize("rows,d,depth,lyndon", [(1, 9, 5, False), (2, 9, 5, True), (64, 8, 5, True), (65, 8, 5, True), (2, 6, 6, True),
                                                 (3, 16, 4, False)])
def test_modules(dtype, rows, d, depth, lyndon):
    import pathsig_amd as ps
    path = brownian_path(rows, 14, d, seed=1250 + d)
    proj = ps.projections.lyndon(depth=depth, path_dim=d) if lyndon else None
    x = path.to(dtype).cuda().requires_grad_(True)
    out = ps.LogSignature(depth=depth, projection=proj)(x)
    sig = TO.signature(path, depth)
    cols = torch.arange(sig.shape[1])
    if lyndon:
        offs, listed, cols = TO.dense_level_offsets(d, depth), iter(proj._codes), []
        for k in range(1, depth + 1):
            size = proj.level_sizes[k]
            cols += [offs[k] + (j if size == d ** k else next(listed)) for j in range(size)]
        cols = torch.tensor(cols)
    full = TO.sig_to_logsig(sig, depth, d, d ** depth, None)[0]
    assert rel_err(out, full[:, cols]) < TOL[dtype]
    G = randn(tuple(out.shape), seed=125)
    dense = torch.zeros_like(full).index_add_(1, cols, G)
    want = TO.signature_vjp(path, TO.logsig_vjp(sig, dense, depth, d, d ** depth, None), depth)
    (grad,) = torch.autograd.grad(out, x, G.to(dtype).cuda())
    assert rel_err(grad, want) < 2 * TOL[dtype]


# The outputs of a product over the top level in parts: two, three, five (fewer than one output to some of a wide alphabet's
# parts), sixteen, and rows that are just too many for any
@pytest.mark.parametrize("dtype", [torch.float64, torch.float32])
@pytest.mark.parametrize("rows,d,depth", [(51, 6, 6), (52, 6, 6), (42, 9, 5), (13, 16, 4), (1, 64, 3), (3, 49, 3)])
def test_parts_of_the_top_products(dtype, rows, d, depth):
    import pathsig_amd  # noqa: F401
    sig = TO.signature(brownian_path(rows, 8, d, seed=1300 + d) * 1.5, depth)
    G = randn(tuple(sig.shape), seed=130)
    x = sig.to(dtype).cuda().requires_grad_(True)
    none = torch.empty(0, dtype=torch.int64, device="cuda")
    got = torch.ops.pathsig.sig_to_logsig(x, depth, d, False, none, [0] + [d ** k for k in range(1, depth + 1)])[0]
    (grad,) = torch.autograd.grad(got, x, G.to(dtype).cuda())
    some = torch.tensor([0, rows - 1]).unique()
    assert rel_err(grad[some], TO.logsig_vjp(sig[some], G[some], depth, d, d ** depth, None)) < TOL[dtype]
