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


# 16 rows, and more than the windows that share a wave start from
@pytest.mark.parametrize("B", [2, 2100])
@pytest.mark.parametrize("dtype", [torch.float64, torch.float32])
@pytest.mark.parametrize("d", [3, 9])
def test_points_that_are_not_finite_show(dtype, d, B):
    """A point that is not finite shows in every coefficient of its letter in its windows, level 1 among them, and in the gradient
    of all of these windows; no other window has it."""
    import pathsig_amd as ps
    windows = torch.tensor([(0, 20), (0, 8), (5, 12), (12, 20), (3, 19), (8, 20), (8, 9), (1, 7)])
    holds = torch.tensor([a <= 7 < b and b - a > 1 for a, b in windows.tolist()])
    path = brownian_path(B, 20, d, seed=1340).to(dtype)
    module = ps.Signature(depth=2, windows=windows.cuda())
    of_letter = torch.zeros(d + d * d, dtype=torch.bool)
    of_letter[1] = True
    of_letter[d:].view(d, d)[1, :] = True
    of_letter[d:].view(d, d)[:, 1] = True
    for bad in (float("nan"), float("inf"), -float("inf")):
        x = path.clone()
        x[1, 7, 1] = bad
        x = x.cuda().requires_grad_(True)
        out = module(x)
        finite = torch.isfinite(out.detach()).cpu()
        want = torch.ones_like(finite)
        want[1] = ~(holds[:, None] & of_letter[None, :])
        assert torch.equal(finite, want)
        (grad,) = torch.autograd.grad(out, x, randn(tuple(out.shape), seed=134).to(dtype).cuda())
        finite = torch.isfinite(grad).all(dim=2).cpu()
        assert finite[0].all() and finite[2:].all() and not finite[1].any()
    # the last point of the window (0, 8): what a very large one there gives, at its limit
    x, large = path.clone(), path.double().clone()
    x[1, 7, 1], large[1, 7, 1] = float("inf"), 1e12
    got = module(x.cuda())[1, 1].double().cpu()
    want = TO.compute_signature(large[1:2], 2, None, None, [(0, 8)])[0, 0]
    assert torch.equal(torch.isinf(got), of_letter) and torch.equal(torch.sign(got)[of_letter], torch.sign(want)[of_letter])


# (8800 windows and 25 600, which share waves with four increments and with one to an LDS round trip.  Few windows are swept, where
# the letter sums of small alphabets are products with zeros and ones, which an infinite gradient turns into NaN for all letters.)
@pytest.mark.parametrize("B", [1100, 3200])
@pytest.mark.parametrize("dtype", [torch.float64, torch.float32])
@pytest.mark.parametrize("word", [(1,), (1, 1), (0, 1), (1, 0)])
def test_an_infinite_gradient_stays_with_its_letters(dtype, word, B):
    """The gradient of the first and of the last point of a window (of one increment sum each) has the sign that a finite upstream
    gradient of its coefficient gives it; the other letters get none."""
    import pathsig_amd as ps
    d, windows = 3, [(0, 20), (5, 12), (12, 20), (2, 5), (3, 19), (8, 20), (8, 9), (0, 8)]
    # (all letters grow all the time: no two infinite terms of opposite signs meet)
    path = brownian_path(B, 20, d, seed=1350)
    path[:, 1:] = (path[:, 1:] - path[:, :-1]).abs().cumsum(dim=1)
    x = path.to(dtype).cuda().requires_grad_(True)
    out = ps.Signature(depth=2, windows=torch.tensor(windows, device="cuda"))(x)
    column = word[0] if len(word) == 1 else d + word[0] * d + word[1]
    grads = []
    for value in (1.0, float("inf")):
        G = torch.zeros_like(out)
        G[1, 1, column] = value
        grads.append(torch.autograd.grad(out, x, G, retain_graph=True)[0].cpu())
    one, infinite = grads
    others = [k for k in range(d) if k not in word]
    assert torch.equal(infinite[..., others], torch.zeros_like(infinite[..., others]))
    assert torch.equal(infinite[0], torch.zeros_like(infinite[0]))
    for at in (5, 11):
        for k in set(word):
            assert one[1, at, k] != 0 and infinite[1, at, k] == torch.sign(one[1, at, k]) * float("inf")


# Windows that start at the same point add their sums up before these go to memory: groups of equal starts that end inside a
# wave, at its end and beyond it, with lengths that differ by more than a tile of increments; tiles that are not full
@pytest.mark.parametrize("dtype", [torch.float64, torch.float32])
@pytest.mark.parametrize("d,B", [(d, B) for d in (2, 3, 4, 7, 8, 12, 16, 20, 32) for B in (2, 420)])
def test_windows_with_equal_starts(dtype, d, B):
    import pathsig_amd as ps
    L = 70
    windows = ([(0, n) for n in (2, 70, 18, 17, 33, 34, 1, 50)] + [(1, 70)] * 3 + [(40, 70), (40, 41), (40, 57)]
               + [(0, 70), (69, 70), (0, 16), (0, 0), (0, 49), (1, 10)])
    path = brownian_path(B, L, d, seed=1360 + d).to(dtype).double()
    x = path.to(dtype).cuda().requires_grad_(True)
    out = ps.Signature(depth=2, windows=torch.tensor(windows, device="cuda"))(x)
    some = torch.tensor([0, 1, B // 2, B - 1]).unique()  # (all of a large batch would take the checker a minute)
    assert rel_err(out[some], TO.compute_signature(path[some], 2, None, None, windows)) < TOL[dtype]
    G = randn(tuple(out.shape), seed=136)
    (grad,) = torch.autograd.grad(out, x, G.to(dtype).cuda())
    assert rel_err(grad[some], TO.signature_vjp(path[some], G[some], 2, None, None, windows)) < TOL[dtype]
    assert torch.isfinite(grad).all()


# Both sides of the lines between sweeps (in chunks, where rows are few) and shared waves, 2048, 4096 and 8192 windows, on paths
# longer than a chunk takes
@pytest.mark.parametrize("dtype", [torch.float64, torch.float32])
@pytest.mark.parametrize("d", [2, 4, 8, 15, 17, 32])
@pytest.mark.parametrize("B", [64, 255, 256, 511, 512, 1023, 1024])
def test_rows_on_both_sides_of_the_lines(dtype, d, B):
    import pathsig_amd as ps
    L = 150
    windows = [(0, 150), (0, 150), (0, 90), (33, 150), (60, 69), (61, 132), (149, 150), (100, 150)]
    path = brownian_path(B, L, d, seed=1370 + d).to(dtype).double()
    x = path.to(dtype).cuda().requires_grad_(True)
    some = torch.tensor([0, B - 1])
    module = ps.Signature(depth=2, windows=torch.tensor(windows, device="cuda"))
    out = module(x)
    with torch.no_grad():
        assert torch.equal(module(x), out)
    assert rel_err(out[some], TO.compute_signature(path[some], 2, None, None, windows)) < TOL[dtype]
    G = randn(tuple(out.shape), seed=137)
    (grad,) = torch.autograd.grad(out, x, G.to(dtype).cuda())
    assert rel_err(grad[some], TO.signature_vjp(path[some], G[some], 2, None, None, windows)) < TOL[dtype]
