"""The log-signature in one call (pathsig_logsignature_*), as the `LogSignature` module takes it, against the CPU
checker: what the wanted columns can be, many rows and few, and buffers and tuning switches that change under it."""
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


def _want(path, depth, windows, proj):
    xr = path.clone().requires_grad_(True)
    parts = [xr] if windows is None else [xr[:, s:e] for s, e in windows]
    full = torch.stack([TO.logsignature(p, depth, method="inverse_exp") for p in parts], dim=1)
    full = full[:, 0] if windows is None else full
    if proj is not None:
        cols = torch.tensor(TO.projection_columns(path.shape[2], depth, proj.level_sizes, proj._codes))
        full = full.index_select(-1, cols)
    return xr, full


def _projection(ps, kind, d, depth):
    if kind == "lyndon":
        return ps.projections.lyndon(depth=depth, path_dim=d)
    if kind == "twice":  # outputs asked for twice, on a level below the top and on the top level
        return ps.projections.words([(0,), (1,), (0,), (1, 0), (1, 0), (0,) * depth, (1,) * depth, (0,) * depth],
                                    depth=depth, path_dim=d)
    if kind == "full_top":  # the top level complete, a level below it not
        return ps.projections.words([(0,), (1, 1), (0, 1)][:depth - 1], depth=depth, path_dim=d, full_levels=(depth,))
    return None


# (8, 5): letter bounds; (8, 4): few rows (several blocks of a row share its outputs); (3, 3): many (a block per
# row); (13, 4): swept in one piece; (2, 2): the smallest layout
@pytest.mark.parametrize("dtype", [torch.float64, torch.float32])
@pytest.mark.parametrize("kind", ["dense", "lyndon", "twice", "full_top"])
@pytest.mark.parametrize("d,depth,B,L,windows", [(8, 5, 2, 90, None), (8, 4, 2, 40, None), (2, 2, 3, 2, None),
                                                 (3, 3, 150, 12, [(0, 12), (3, 9), (5, 7)]), (13, 4, 1, 9, None),
                                                 (6, 4, 2, 30, [(0, 30), (4, 20)])])
def test_one_call(ps, dtype, kind, d, depth, B, L, windows):
    proj = _projection(ps, kind, d, depth)
    path = brownian_path(B, L, d, seed=800 + d)
    xr, want = _want(path, depth, windows, proj)
    G = randn(tuple(want.shape), seed=81)
    (want_grad,) = torch.autograd.grad(want, xr, G)
    module = ps.LogSignature(depth=depth, projection=proj,
                             windows=None if windows is None else torch.tensor(windows, device="cuda"))
    x = path.to(dtype).cuda().requires_grad_(True)
    with torch.no_grad():
        plain = module(x)
    out = module(x)
    (grad,) = torch.autograd.grad(out, x, G.to(dtype).cuda())
    if kind in ("dense", "full_top"):  # (whether a list of words runs on the compiled kernels is a matter of cost)
        assert "LogSignatureKeepDirect" in out.grad_fn.name()
    assert torch.equal(plain, out)
    assert rel_err(out, want) < TOL[dtype] and rel_err(grad, want_grad) < 2 * TOL[dtype]


def test_lists_follow_the_buffers_and_switches(ps, set_option):
    d, depth = 4, 4
    first = ps.projections.words([(0, 1, 2, 3), (3, 3, 3, 0)], depth=depth, path_dim=d, full_levels=(1,))
    other = ps.projections.words([(1, 1, 2, 2), (2, 0, 0, 1)], depth=depth, path_dim=d, full_levels=(1,))
    set_option("embed_share", 10 ** 6)
    path = brownian_path(3, 60, d, seed=820)
    G = randn((3, first.sig_size), seed=82)
    module = ps.LogSignature(depth=depth, projection=first)
    module.load_state_dict(ps.LogSignature(depth=depth, projection=other).state_dict())
    xr, want = _want(path, depth, None, other)
    (want_grad,) = torch.autograd.grad(want, xr, G)
    x = path.cuda().requires_grad_(True)
    # the switches of the backward are not those of the forward: other chunks, and no compiled shape at all
    for name, value in (("chunks", 5), ("tiled", 0)):
        out = module(x)
        assert rel_err(out, want) < 1e-12
        set_option(name, value)
        (grad,) = torch.autograd.grad(out, x, G.cuda())
        assert rel_err(grad, want_grad) < 2e-12
        set_option("tiled", 1)


# a block per row compiled for the layout: the longest and the shortest of every depth, those that fit in fp32 only
# ((3, 7), (4, 6)), tiny ones whose rows are less than a wave, more rows than share the device by slices
@pytest.mark.parametrize("kind", ["dense", "lyndon"])
@pytest.mark.parametrize("d,depth", [(2, 2), (16, 2), (2, 3), (16, 3), (7, 4), (2, 5), (5, 5), (3, 6), (4, 6), (2, 7), (3, 7),
                                     (2, 8)])
def test_small_layouts(ps, kind, d, depth):
    proj = _projection(ps, kind, d, depth)
    module = ps.LogSignature(depth=depth, projection=proj)
    for B in (1, 530 if d ** depth < 300 else 5):
        path = brownian_path(B, 7, d, seed=840 + d)
        xr, want = _want(path, depth, None, proj)
        G = randn(tuple(want.shape), seed=83)
        (want_grad,) = torch.autograd.grad(want, xr, G)
        for dtype in (torch.float64, torch.float32):
            x = path.to(dtype).cuda().requires_grad_(True)
            out = module(x)
            (grad,) = torch.autograd.grad(out, x, G.to(dtype).cuda())
            assert rel_err(out, want) < TOL[dtype] and rel_err(grad, want_grad) < 2 * TOL[dtype]


def test_modules_and_tensors_the_direct_call_leaves_to_the_operators(ps):
    """A module from a file without the derived lists, buffers whose writes leave no trace, and tangents."""
    d, depth = 3, 3
    first = ps.projections.words([(0, 1, 2), (2, 2, 0)], depth=depth, path_dim=d)
    other = ps.projections.words([(1, 1, 2), (2, 0, 1)], depth=depth, path_dim=d)
    path = brownian_path(2, 9, d, seed=830)
    older = ps.LogSignature(depth=depth, projection=first)
    del older.__dict__["_lists"]
    assert rel_err(older(path.cuda()), _want(path, depth, None, first)[1]) < 1e-12
    with torch.inference_mode():
        written = ps.LogSignature(depth=depth, projection=first)
        written(path.cuda())
        written._top_words.copy_(ps.LogSignature(depth=depth, projection=other)._top_words)
        assert rel_err(written(path.cuda()), _want(path, depth, None, other)[1]) < 1e-12
    for module in (ps.Signature(depth=depth), ps.LogSignature(depth=depth)):
        with torch.autograd.forward_ad.dual_level():
            x = torch.autograd.forward_ad.make_dual(path.cuda(), path.cuda())
            with pytest.raises(RuntimeError):
                module(x)
