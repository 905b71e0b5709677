"""Depth 2 in windows: several windows to a wave, against the CPU checker."""
import pytest
import torch

from oracle import tensor_oracle as TO

from .helpers import brownian_path, randn, rel_err

pytestmark = pytest.mark.gpu
TOL = {torch.float32: 1e-5, torch.float64: 1e-12}


# letters around the padded group sizes; windows that are empty, of one point, of one increment, overlapping, of very
# different lengths inside one wave, out of range; more windows than a block holds; a path far from the origin
@pytest.mark.parametrize("dtype", [torch.float64, torch.float32])
# (3000 paths: windows enough to take one increment at a time)
@pytest.mark.parametrize("d,B,far", [(d, B, far) for d in (2, 3, 4, 5, 8, 9, 15, 16, 17, 32, 33)
                                     for B, far in ((1, False), (40, False), (7, True))]
                         + [(4, 3000, False), (9, 3000, False), (17, 3000, False)])
def test_depth_two_windows(dtype, d, B, far):
    import pathsig_amd as ps
    L = 60
    windows = [(0, 60), (5, 5), (7, 8), (9, 11), (3, 40), (30, 60), (58, 60), (59, 60), (0, 2), (20, 50), (25, 33)]
    path = brownian_path(B, L, d, seed=1300 + d)
    if far:
        path = path + 8.0  # (an exact shift up to rounding of the points themselves)
    path = path.to(dtype).double()
    want = TO.compute_signature(path, 2, None, None, windows)
    x = path.to(dtype).cuda().requires_grad_(True)
    out = ps.Signature(depth=2, windows=torch.tensor(windows, device="cuda"))(x)
    assert rel_err(out, want) < TOL[dtype]
    G = randn(tuple(want.shape), seed=131)
    (grad,) = torch.autograd.grad(out, x, G.to(dtype).cuda())
    assert rel_err(grad, TO.signature_vjp(path, G, 2, None, None, windows)) < TOL[dtype]
    log = ps.LogSignature(depth=2, windows=torch.tensor(windows, device="cuda"))(x)
    assert torch.isfinite(log).all() and rel_err(log[..., :d], want[..., :d]) < TOL[dtype]
