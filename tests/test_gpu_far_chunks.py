"""Time chunks of the shapes whose kernels sweep a row in one piece (several blocks to a unit, children split between lanes,
fp64 rows that the scan kernel does not take), against the CPU checker."""
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


# (16, 4): split children in one block; (12, 5): split, beyond what the products are compiled for (one piece); (9, 5), (5, 7):
# several blocks; (13, 4): several blocks in fp64; (4, 7): fp64 rows too long for the scan kernel.  Six chunks are the least
# that are multiplied; fewer increments than chunks leave some empty.
@pytest.mark.parametrize("dtype", [torch.float64, torch.float32])
@pytest.mark.parametrize("d,depth,chunks,L", [(16, 4, 6, 40), (16, 4, 9, 7), (12, 5, 6, 20), (9, 5, 7, 31), (5, 7, 17, 35),
                                              (13, 4, 16, 20), (4, 7, 6, 67), (4, 7, 33, 40), (16, 4, 5, 40)])
def test_forced_chunks(ps, set_option, dtype, d, depth, chunks, L):
    set_option("chunks", chunks)
    B = 2 if d ** depth < 70000 else 1
    path = brownian_path(B, L, d, seed=900 + d + chunks)
    want = TO.signature(path, depth)
    G = randn(tuple(want.shape), seed=91)
    want_grad = TO.signature_vjp(path, G, depth)
    x = path.to(dtype).cuda().requires_grad_(True)
    module = ps.Signature(depth=depth)
    with torch.no_grad():
        plain = module(x)
    out = module(x)
    assert rel_err(out, want) < TOL[dtype]
    assert torch.equal(out.detach(), plain)  # whether or not anything is kept
    (grad,) = torch.autograd.grad(out, x, G.to(dtype).cuda())
    assert rel_err(grad, want_grad) < TOL[dtype]
    # the operator that gets no products from the forward
    none = torch.empty(0, dtype=torch.int64, device="cuda")
    alone = torch.ops.pathsig.signature_backward(x.detach(), out.detach(), G.to(dtype).cuda(), depth, False, none, [],
                                                 False, none.int())
    assert rel_err(alone, want_grad) < TOL[dtype]


@pytest.mark.parametrize("dtype", [torch.float64, torch.float32])
@pytest.mark.parametrize("d,depth,L,name", [(14, 4, 600, "lyndon"), (9, 5, 400, "lyndon"), (9, 5, 500, "words"),
                                            (16, 4, 300, None), (14, 4, 500, None), (4, 7, 700, None)])
def test_own_choice(ps, dtype, d, depth, L, name):
    """The library's choice for one path, with projections that are swept in the dense layout."""
    path = brownian_path(1, L, d, seed=930 + d)
    x = path.to(dtype).cuda().requires_grad_(True)
    proj = None
    if name == "lyndon":
        proj = ps.projections.lyndon(depth=depth, path_dim=d)
    elif name == "words":
        words = [tuple((7 * i + 3 * j * j + i // 5) % d for j in range(depth)) for i in range(0, 40000, 5)]
        proj = ps.projections.words(sorted(set(words)), depth=depth, path_dim=d, full_levels=(1, 2, 3, 4))
    module = ps.LogSignature if name == "lyndon" else ps.Signature
    out = module(depth=depth, projection=proj)(x)
    full = (TO.logsignature if name == "lyndon" else TO.signature)(path, depth)
    offs = TO.dense_level_offsets(d, depth)
    cols = torch.arange(full.shape[1])
    if proj is not None:
        listed, cols = iter(proj._codes), []
        for k in range(1, depth + 1):
            size = proj.level_sizes[k]
            cols += [offs[k] + (j if size == d ** k else next(listed)) for j in range(size)]
        cols = torch.tensor(cols)
    assert rel_err(out, full[:, cols]) < TOL[dtype]
    if name != "lyndon":
        G = randn(tuple(out.shape), seed=93)
        dense = torch.zeros_like(full)
        dense.index_add_(1, cols, G)
        (grad,) = torch.autograd.grad(out, x, G.to(dtype).cuda())
        assert rel_err(grad, TO.signature_vjp(path, dense, depth)) < TOL[dtype]


def test_infinite_gradient_after_the_last_chunk(ps, set_option):
    """Nothing follows the last chunk: an infinite upstream gradient is not multiplied with the zeros there."""
    set_option("chunks", 8)
    x = brownian_path(1, 41, 16, seed=950).float().cuda().requires_grad_(True)
    out = ps.Signature(depth=4)(x)
    G = torch.zeros_like(out)
    G[0, 3] = float("inf")  # level 1: the sum of the increments of letter 3
    (grad,) = torch.autograd.grad(out, x, G)
    others = [k for k in range(16) if k != 3]
    assert torch.isfinite(grad[0, -5:, others]).all()
