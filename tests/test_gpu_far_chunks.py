"""Time chunks of the shapes whose kernels sweep a row in one piece (several blocks to a unit, children split between lanes,
fp64 rows that the scan kernel does not take), against the CPU checker."""
import ctypes

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


def _columns(proj, d, depth):
    """Places of a projection's words in the dense layout."""
    if proj is None:
        return torch.arange(sum(d ** k for k in range(1, depth + 1)))
    return torch.tensor(TO.projection_columns(d, depth, proj.level_sizes, proj._codes))


def _kept_chunks(dtype, B, L, d, depth, level_sizes, logarithm):
    """Time chunks whose products a forward of the call hands to its backward (0: none)."""
    from pathsig_amd import _load
    lib, code, elem = _load.lib(), 0 if dtype == torch.float32 else 1, 4 if dtype == torch.float32 else 8
    if logarithm:  # (levels below the top are full in what the call computes; the size counts the chunks, four elements each)
        sizes = None if level_sizes is None else [0, *[d ** k for k in range(1, depth)], level_sizes[depth]]
        host = None if sizes is None else (ctypes.c_int64 * len(sizes))(*sizes)
        out = [ctypes.c_size_t() for _ in range(3)]
        lib.pathsig_logsignature_sizes.argtypes = [ctypes.c_int] + [ctypes.c_int64] * 3 + [
            ctypes.c_int, ctypes.c_void_p, ctypes.c_int64] + [ctypes.POINTER(ctypes.c_size_t)] * 3
        assert lib.pathsig_logsignature_sizes(code, B, L, d, depth, host, 0, *out) == 0
        tag = out[0].value // elem % 4096
        return tag // 4 if tag % 4 == 1 else 0
    host = None if level_sizes is None else (ctypes.c_int64 * len(level_sizes))(*level_sizes)
    low = B * sum(d ** k for k in range(1, depth)) * elem
    kept = lib.pathsig_sig_chunks_bytes(code, B, L, d, depth, host, 0)
    dense = low + B * d ** depth * elem  # (a projection that is swept in one piece keeps its dense rows)
    return 0 if kept == dense else kept // low // 2


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
    """The library's choice for one path is far chunks, with projections that are swept in the dense layout too."""
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
    cols = _columns(proj, d, depth)
    assert _kept_chunks(dtype, 1, L, d, depth, None if proj is None else proj.level_sizes, name == "lyndon") > 1
    assert rel_err(out, full[:, cols]) < TOL[dtype]
    G = randn(tuple(out.shape), seed=93)
    dense = torch.zeros_like(full)
    dense.index_add_(1, cols, G)
    (grad,) = torch.autograd.grad(out, x, G.to(dtype).cuda())
    if name == "lyndon":
        dense = TO.logsig_vjp(TO.signature(path, depth), dense, depth, d, d ** depth, None)
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


# (16, 4): far chunks; (14, 4): the entry with the shorter prefix, for its chunks; (4, 7) fp64: rows that the scan kernel does not
# take; 70 letters at depth 3: on copies over 72; a word projection of (9, 5), through its dense rows
@pytest.mark.parametrize("dtype,B,L,d,depth,listed", [
    (torch.float32, 2, 400, 16, 4, False), (torch.float64, 2, 400, 16, 4, False), (torch.float32, 2, 500, 14, 4, False),
    (torch.float64, 2, 700, 4, 7, False), (torch.float32, 1, 500, 70, 3, False), (torch.float32, 2, 300, 9, 5, True)])
def test_scratch_that_holds_one_piece_only(ps, dtype, B, L, d, depth, listed):
    """Far chunks are there for speed: a forward or backward that hands nothing over and brings what a sweep in one piece takes is
    swept in one piece, and one that brings less is refused."""
    from pathsig_amd import _load
    lib = _load.lib()
    code, elem = (0, 4) if dtype == torch.float32 else (1, 8)
    pad = lambda n: (n + 255) // 256 * 256
    top = d ** depth
    codes = torch.arange(0, top, 3) if listed else torch.empty(0, dtype=torch.int64)
    sizes = (ctypes.c_int64 * (depth + 1))(0, *[d ** k for k in range(1, depth)], len(codes)) if listed else None
    S = sum(d ** k for k in range(1, depth)) + (len(codes) if listed else top)
    wide = (d + 7) // 8 * 8 if d > 64 else d
    copies = [0, 0] if wide == d else [pad(B * L * wide * elem), pad(B * sum(wide ** k for k in range(1, depth + 1)) * elem)]
    dense = pad(B * sum(d ** k for k in range(1, depth + 1)) * elem) if listed else 0
    forward = sum(copies) + dense
    backward = 2 * sum(copies) + 2 * dense + pad(B * (L - 1) * wide * elem)
    call = (code, B, L, d, depth, sizes, 0)
    asked = lib.pathsig_sig_forward_workspace(*call), lib.pathsig_sig_backward_workspace(*call)
    assert asked[0] > forward and asked[1] > backward + 256
    path = brownian_path(B, L, d, seed=960 + d).to(dtype).double()
    x = path.to(dtype).cuda()
    G = randn((B, S), seed=96)
    g, words = G.to(dtype).cuda(), codes.cuda()
    p = lambda t: ctypes.c_void_p(t.data_ptr() if t.numel() else 0)
    stream = ctypes.c_void_p(torch.cuda.current_stream().cuda_stream)
    ws = torch.empty(max(asked), dtype=torch.uint8, device="cuda")
    tail = (code, B, L, d, depth, sizes, p(words) if listed else None, len(codes), None, 0)
    cols = torch.cat([torch.arange(S - len(codes)), S - len(codes) + codes]) if listed else torch.arange(S)
    full = TO.signature(path, depth)
    want_grad = TO.signature_vjp(path, torch.zeros_like(full).index_add_(1, cols, G), depth)
    for fws, bws in (asked, (forward, backward)):
        sig, grad = torch.full((B, S), float("nan"), dtype=dtype, device="cuda"), torch.full_like(x, float("nan"))
        assert lib.pathsig_sig_forward(p(x), p(sig), *tail, p(ws) if fws else None, fws, stream) == 0, lib.pathsig_last_error()
        assert lib.pathsig_sig_backward(p(x), p(sig), p(g), p(grad), *tail, p(ws), bws, stream) == 0, lib.pathsig_last_error()
        torch.cuda.synchronize()
        assert rel_err(sig, full[:, cols]) < TOL[dtype] and rel_err(grad, want_grad) < TOL[dtype]
    if forward:
        assert lib.pathsig_sig_forward(p(x), p(sig), *tail, p(ws), forward - 256, stream) == -3
    assert lib.pathsig_sig_backward(p(x), p(sig), p(g), p(grad), *tail, p(ws), backward - 256, stream) == -3


# In chunks by force and by the library's choice; the last lengths that an fp32 call of a depth has its chunks for, and the first
# that it has not (LogPlan)
@pytest.mark.parametrize("dtype", [torch.float64, torch.float32])
@pytest.mark.parametrize("d,depth,L,chunks,lyndon", [(9, 5, 90, 7, False), (9, 5, 90, 7, True), (16, 4, 90, 7, False), (16, 4, 90, 7, True),
                                                     (9, 5, 300, 0, False), (16, 4, 300, 0, True), (9, 5, 1025, 0, True),
                                                     (9, 5, 1026, 0, True), (16, 4, 2049, 0, False), (16, 4, 2050, 0, False)])
def test_gradient_of_the_logarithm(ps, set_option, dtype, d, depth, L, chunks, lyndon):
    set_option("chunks", chunks)
    path = brownian_path(1, L, d, seed=970 + d + L).to(dtype).double()
    proj = ps.projections.lyndon(depth=depth, path_dim=d) if lyndon else None
    in_chunks = _kept_chunks(dtype, 1, L, d, depth, proj.level_sizes if lyndon else None, True)
    one_piece = dtype == torch.float32 and L - 1 > 2048 >> (depth - 4)
    assert in_chunks == chunks if chunks else (in_chunks > 1) != one_piece
    x = path.to(dtype).cuda().requires_grad_(True)
    out = ps.LogSignature(depth=depth, projection=proj)(x)
    sig, cols = TO.signature(path, depth), _columns(proj, d, depth)
    assert rel_err(out, TO.sig_to_logsig(sig, depth, d, d ** depth, None)[0][:, cols]) < TOL[dtype]
    G = randn(tuple(out.shape), seed=97)
    dense = torch.zeros_like(sig).index_add_(1, cols, G)
    want = TO.signature_vjp(path, TO.logsig_vjp(sig, dense, depth, d, d ** depth, None), depth)
    (grad,) = torch.autograd.grad(out, x, G.to(dtype).cuda())
    assert rel_err(grad, want) < TOL[dtype]
