"""Time chunks of the per-word kernels (words_chunks.hip), against the CPU checker."""
import ctypes

import pytest
import torch

from oracle import tensor_oracle as TO

from .helpers import brownian_path, code_of, random_word_set, randn, rel_err

pytestmark = pytest.mark.gpu
TOL = {torch.float32: 1e-5, torch.float64: 1e-12}


@pytest.fixture(scope="module")
def ps():
    import pathsig_amd
    return pathsig_amd


def _chunked(dtype, B, L, d, depth, sizes):
    from pathsig_amd import _load
    host = None if sizes is None else (ctypes.c_int64 * len(sizes))(*sizes)
    return _load.lib().pathsig_sig_forward_scratch(0 if dtype == torch.float32 else 1, B, L, d, depth, host, 0) > 0


# Lanes on words (fewer than a dozen paths) and lists (groups of sixteen paths, the last one with lanes to spare); words of one
# letter to eight; levels without words; more words of a level than a wave holds, which put suffixes of several levels into
# one wave; all words (no list); chunks of unequal length
@pytest.mark.parametrize("dtype", [torch.float64, torch.float32])
@pytest.mark.parametrize("B,L,d,depth,lo,hi,count,full", [
    (1, 130, 3, 4, 3, 4, 10, (1, 2)), (11, 211, 3, 5, 1, 5, 90, ()), (12, 211, 3, 5, 1, 5, 90, ()), (17, 300, 2, 8, 7, 8, 9, ()),
    (3, 150, 2, 8, 1, 8, 60, ()), (2, 97, 6, 4, 4, 4, 200, (2,)), (5, 260, 4, 6, 5, 6, 150, (1, 2, 3)), (20, 400, 4, 3, 3, 3, 5, ()),
    (2, 333, 5, 1, 1, 1, 0, (1,)), (33, 180, 6, 4, 2, 4, 80, (1,)), (1, 4000, 2, 3, 2, 3, 7, (1,))])
def test_words_in_chunks(ps, set_option, dtype, B, L, d, depth, lo, hi, count, full):
    set_option("tiled", 0)
    words = [w for w in random_word_set(d, lo, hi, count, seed=970 + count) if len(w) not in full]
    proj = ps.projections.words(words, depth=depth, path_dim=d, full_levels=full)
    assert _chunked(dtype, B, L, d, depth, proj.level_sizes)
    path = brownian_path(B, L, d, seed=960 + L)
    x = path.to(dtype).cuda().requires_grad_(True)
    module = ps.Signature(depth=depth, projection=proj)
    with torch.no_grad():
        plain = module(x)
    out = module(x)
    offs, listed, cols = TO.dense_level_offsets(d, depth), iter(proj._codes), []
    for k in range(1, depth + 1):
        size = proj.level_sizes[k]
        cols += [offs[k] + (j if size == d ** k else next(listed)) for j in range(size)]
    cols = torch.tensor(cols)
    full_sig = TO.signature(path, depth)
    assert rel_err(out, full_sig[:, cols]) < TOL[dtype]
    assert torch.equal(out.detach(), plain)
    G = randn(tuple(out.shape), seed=97)
    dense = torch.zeros_like(full_sig).index_add_(1, cols, G)
    want = TO.signature_vjp(path, dense, depth)
    (grad,) = torch.autograd.grad(out, x, G.to(dtype).cuda())
    assert rel_err(grad, want) < TOL[dtype]
    # the operator that gets nothing from the forward
    alone = torch.ops.pathsig.signature_backward(x.detach(), out.detach(), G.to(dtype).cuda(), depth, True,
                                                 proj.encoded_words, proj.level_sizes, False,
                                                 torch.empty(0, dtype=torch.int32, device="cuda"))
    assert rel_err(alone, want) < TOL[dtype]


@pytest.mark.parametrize("dtype", [torch.float64, torch.float32])
def test_all_words_in_chunks(ps, set_option, dtype):
    set_option("tiled", 0)
    B, L, d, depth = 2, 170, 3, 4
    assert _chunked(dtype, B, L, d, depth, None)
    path = brownian_path(B, L, d, seed=981)
    x = path.to(dtype).cuda().requires_grad_(True)
    out = ps.Signature(depth=depth)(x)
    want = TO.signature(path, depth)
    assert rel_err(out, want) < TOL[dtype]
    G = randn(tuple(want.shape), seed=98)
    (grad,) = torch.autograd.grad(out, x, G.to(dtype).cuda())
    assert rel_err(grad, TO.signature_vjp(path, G, depth)) < TOL[dtype]


@pytest.mark.parametrize("B", [2, 14])
def test_repeated_words_and_an_infinite_gradient(ps, set_option, B):
    """Entries of one word add up; an infinite gradient reaches the letters of its word and no others, also from the last chunk,
    behind which nothing follows."""
    set_option("tiled", 0)
    L, d, depth, dtype = 200, 4, 4, torch.float64
    words = [(0, 1, 0, 1), (3, 2, 3, 3), (0, 1, 0, 1), (2, 2, 3, 2)]
    codes = torch.tensor([code_of(w, d) for w in words], device="cuda")
    sizes = [0, 0, 0, 0, len(words)]
    none = torch.empty(0, dtype=torch.int32, device="cuda")
    assert _chunked(dtype, B, L, d, depth, sizes)
    path = brownian_path(B, L, d, seed=985)
    x = path.cuda().requires_grad_(True)
    out = torch.ops.pathsig.compute_signature(x, depth, True, codes, sizes, False, none)
    cols = TO.dense_level_offsets(d, depth)[depth] + codes.cpu()
    full = TO.signature(path, depth)
    assert rel_err(out, full[:, cols]) < 1e-12
    G = randn(tuple(out.shape), seed=99)
    (grad,) = torch.autograd.grad(out, x, G.cuda(), retain_graph=True)
    want = TO.signature_vjp(path, torch.zeros_like(full).index_add_(1, cols, G), depth)
    assert rel_err(grad, want) < 1e-12
    G[:, 0] = float("inf")
    (grad,) = torch.autograd.grad(out, x, G.cuda())
    assert not torch.isfinite(grad[..., :2]).any(dim=1).all()
    assert rel_err(grad[..., 2:], want[..., 2:]) < 1e-12


def test_scratch_that_holds_one_piece_only(ps):
    """A plain forward or backward that brings no more scratch than a sweep in one piece takes is swept in one piece."""
    from pathsig_amd import _load
    lib = _load.lib()
    B, L, d, depth = 2, 300, 16, 6
    words = random_word_set(d, 3, depth, 40, seed=990)
    proj = ps.projections.words(words, depth=depth, path_dim=d, full_levels=(1,))
    sizes = (ctypes.c_int64 * len(proj.level_sizes))(*proj.level_sizes)
    need = lib.pathsig_sig_backward_workspace(1, B, L, d, depth, sizes, 0)
    small = B * (L - 1) * d * 8 + 512
    assert lib.pathsig_sig_forward_scratch(1, B, L, d, depth, sizes, 0) > 0 and need > small
    x = brownian_path(B, L, d, seed=991).cuda()
    codes = proj.encoded_words
    S = proj.sig_size
    g = randn((B, S), seed=992).cuda()
    ws = torch.empty(need, dtype=torch.uint8, device="cuda")
    p = lambda t: ctypes.c_void_p(t.data_ptr())
    stream = ctypes.c_void_p(torch.cuda.current_stream().cuda_stream)
    results = []
    for fws, bws in ((lib.pathsig_sig_forward_scratch(1, B, L, d, depth, sizes, 0), need), (0, small)):
        wsf = torch.empty(max(fws, 1), dtype=torch.uint8, device="cuda")
        sig, grad = torch.full((B, S), float("nan"), dtype=torch.float64, device="cuda"), torch.full_like(x, float("nan"))
        assert lib.pathsig_sig_forward(p(x), p(sig), 1, B, L, d, depth, sizes, p(codes), codes.numel(), None, 0,
                                       p(wsf) if fws else None, fws, stream) == 0
        assert lib.pathsig_sig_backward(p(x), p(sig), p(g), p(grad), 1, B, L, d, depth, sizes, p(codes), codes.numel(), None, 0,
                                        p(ws), bws, stream) == 0
        torch.cuda.synchronize()
        results.append((sig, grad))
    assert rel_err(results[0][0], results[1][0]) < 1e-12 and rel_err(results[0][1], results[1][1]) < 1e-12


@pytest.mark.parametrize("dtype", [torch.float64, torch.float32])
def test_a_plain_forward_with_the_scratch_it_asks_for_is_swept_in_chunks(ps, dtype):
    """Words that would be computed through a dense shape: with the workspace that the query asks for, the forward gives the bits of
    one that keeps the table of the chunks; with none it is swept in one piece."""
    from pathsig_amd import _load
    lib = _load.lib()
    B, L, d, depth, code = 2, 1000, 6, 5, 0 if dtype == torch.float32 else 1
    words = random_word_set(d, 3, depth, 16, seed=994)
    proj = ps.projections.words(words, depth=depth, path_dim=d, full_levels=(1, 2))
    sizes = (ctypes.c_int64 * len(proj.level_sizes))(*proj.level_sizes)
    call = (code, B, L, d, depth, sizes, 0)
    need, keeps = lib.pathsig_sig_forward_workspace(*call), lib.pathsig_sig_chunks_bytes(*call)
    assert need > 0 and lib.pathsig_sig_forward_keep_workspace(*call) == 0
    path = brownian_path(B, L, d, seed=995)
    x, codes = path.to(dtype).cuda(), proj.encoded_words
    ws, table = (torch.empty(n, dtype=torch.uint8, device="cuda") for n in (need, keeps))
    p = lambda t: ctypes.c_void_p(t.data_ptr())
    stream = ctypes.c_void_p(torch.cuda.current_stream().cuda_stream)
    sigs = [torch.full((B, proj.sig_size), float("nan"), dtype=dtype, device="cuda") for _ in range(3)]
    words_arg = (sizes, p(codes), codes.numel(), None, 0)
    assert lib.pathsig_sig_forward(p(x), p(sigs[0]), code, B, L, d, depth, *words_arg, p(ws), need, stream) == 0
    assert lib.pathsig_sig_forward_keep(p(x), p(sigs[1]), code, B, L, d, depth, *words_arg, p(table), keeps, None, 0, stream) == 0
    assert lib.pathsig_sig_forward(p(x), p(sigs[2]), code, B, L, d, depth, *words_arg, None, 0, stream) == 0
    torch.cuda.synchronize()
    offs, listed, cols = TO.dense_level_offsets(d, depth), iter(proj._codes), []
    for k in range(1, depth + 1):
        size = proj.level_sizes[k]
        cols += [offs[k] + (j if size == d ** k else next(listed)) for j in range(size)]
    want = TO.signature(path, depth)[:, torch.tensor(cols)]
    assert torch.equal(sigs[0], sigs[1]) and not torch.equal(sigs[0], sigs[2])
    assert all(rel_err(s, want) < TOL[dtype] for s in sigs)
