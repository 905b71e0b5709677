"""Long chains of time chunks: the products of a row's chunks in steps of a parallel prefix product
(chain_kernels.hip), against the CPU checker."""
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


# (2, 5) and (4, 6): groups of four chunks in fp32; (8, 5): rows of which six do not fit a block's LDS (radix 2);
# (3, 3): two levels below the top; chunk counts around the powers of the radix, and one that nothing divides
@pytest.mark.parametrize("dtype", [torch.float64, torch.float32])
@pytest.mark.parametrize("d,depth,chunks,L", [(2, 5, 260, 300), (3, 3, 256, 300), (3, 3, 257, 258), (4, 6, 128, 150),
                                              (4, 6, 101, 150), (3, 6, 272, 280), (8, 5, 65, 70), (2, 2, 320, 330)])
def test_many_chunks(ps, set_option, dtype, d, depth, chunks, L):
    set_option("chunks", chunks)
    B = 2
    path = brownian_path(B, L, d, seed=700 + d + chunks)
    want = TO.signature(path, depth)
    G = randn(tuple(want.shape), seed=71)
    want_grad = TO.signature_vjp(path, G, depth)
    x = path.to(dtype).cuda().requires_grad_(True)
    module = ps.Signature(depth=depth)
    with torch.no_grad():
        assert rel_err(module(x), want) < TOL[dtype]
    out = module(x)
    assert rel_err(out, want) < TOL[dtype]
    (grad,) = torch.autograd.grad(out, x, G.to(dtype).cuda())
    assert rel_err(grad, want_grad) < TOL[dtype]
    # the operator that gets no products from the forward
    none = torch.empty(0, dtype=torch.int64, device="cuda")
    alone = torch.ops.pathsig.signature_backward(x.detach(), out.detach(), G.to(dtype).cuda(), depth, False, none, [],
                                                 False, none.int())
    assert rel_err(alone, want_grad) < TOL[dtype]


@pytest.mark.parametrize("dtype,grad", [(torch.float64, True), (torch.float32, True), (torch.float32, False)])
@pytest.mark.parametrize("d,depth,L", [(3, 6, 2801), (7, 5, 1203)])
def test_one_long_path(ps, dtype, grad, d, depth, L):
    """The library's own choice of chunks for a single path."""
    path = brownian_path(1, L, d, seed=720 + d)
    want = TO.signature(path, depth)
    x = path.to(dtype).cuda().requires_grad_(grad)
    out = ps.Signature(depth=depth)(x)
    assert rel_err(out, want) < TOL[dtype]
    if grad:
        G = randn(tuple(want.shape), seed=73)
        (got,) = torch.autograd.grad(out, x, G.to(dtype).cuda())
        assert rel_err(got, TO.signature_vjp(path, G, depth)) < TOL[dtype]
