"""What an upstream gradient of a module's output can be besides a plain tensor: the backward nodes of the direct module
calls hand such tensors to the operators."""
import pytest
import torch
from torch.utils._python_dispatch import TorchDispatchMode

from .helpers import brownian_path, randn, rel_err

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def ps():
    import pathsig_amd
    return pathsig_amd


@pytest.fixture(params=["sig", "sig_windows", "sig_words", "logsig", "lyndon", "lyndon_large"])
def call(ps, request):
    kind, windows, proj = request.param, None, None
    d, depth = (8, 5) if kind == "lyndon_large" else (3, 3)
    if kind == "sig_windows":
        windows = torch.tensor([(0, 12), (3, 9)], device="cuda")
    if kind == "sig_words":
        proj = ps.projections.words([(0,), (1, 2), (2, 0, 1)], depth=depth, path_dim=d)
    if "lyndon" in kind:
        proj = ps.projections.lyndon(depth=depth, path_dim=d)
    module = (ps.Signature if "sig" in kind[:3] else ps.LogSignature)(depth=depth, projection=proj, windows=windows)
    x = brownian_path(2, 12, d, seed=890).cuda().requires_grad_(True)
    out = module(x)
    assert "Direct" in out.grad_fn.name()
    G = randn((3, *out.shape), seed=89).cuda()
    each = torch.stack([torch.autograd.grad(out, x, g, retain_graph=True)[0] for g in G])
    return module, x, out, G, each


def test_batched_gradients(call):
    module, x, out, G, each = call
    (got,) = torch.autograd.grad(out, x, G, is_grads_batched=True, retain_graph=True)
    assert got.shape == each.shape and rel_err(got, each) < 1e-12
    if out.numel() <= 200:
        rows = torch.autograd.functional.jacobian(module, x, vectorize=True)
        assert rel_err(torch.tensordot(G, rows, dims=out.dim()), each) < 1e-12


def test_gradient_with_its_sign_still_to_apply(call):
    _, x, out, G, each = call
    (got,) = torch.autograd.grad(out, x, torch._neg_view(G[0]), retain_graph=True)
    assert rel_err(got, -each[0]) < 1e-12
    # (as it comes out of a complex computation: the imaginary part of a conjugate)
    (got,) = torch.autograd.grad(out, x, torch.complex(G[1], G[0]).conj().imag, retain_graph=True)
    assert rel_err(got, -each[0]) < 1e-12


def test_modes_see_the_backward(call):
    _, x, out, G, each = call
    seen = []

    class Watch(TorchDispatchMode):
        def __torch_dispatch__(self, func, types, args=(), kwargs=None):
            seen.append(str(func))
            return func(*args, **(kwargs or {}))

    with Watch():
        (got,) = torch.autograd.grad(out, x, G[0], retain_graph=True)
    assert rel_err(got, each[0]) < 1e-12
    assert any(name.startswith("pathsig.signature_backward_kept") for name in seen)


def test_gradients_of_other_strides_and_saved_tensors_through_hooks(call):
    module, x, _, G, each = call
    with torch.autograd.graph.save_on_cpu():
        out = module(x)
    spread = torch.empty((*G[0].shape, 2), dtype=G.dtype, device="cuda")[..., 0].copy_(G[0])
    (got,) = torch.autograd.grad(out, x, spread)
    assert rel_err(got, each[0]) < 1e-12
