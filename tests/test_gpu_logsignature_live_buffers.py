"""A `LogSignature` keeps nothing on the device beside its buffers: words and wanted columns may be rewritten in any way
(through `.data`, before a copy or a pickle, between two replays of a captured graph) and every call, copy and replay
follows them, against the CPU checker."""
import copy
import io
import random

import pytest
import torch

from oracle import tensor_oracle as TO

from .helpers import brownian_path, randn, rel_err

pytestmark = pytest.mark.gpu
BUFFERS = ("_encoded_words", "_top_words", "_indices_from_sig")


@pytest.fixture(scope="module")
def ps():
    import pathsig_amd
    return pathsig_amd


# (8, 5): letter bounds, few chosen words above a random letter each; (4, 7): above the layouts of one block per row,
# no bounds; (3, 3): a block per row
SHAPES = [(8, 5, 90), (4, 7, 70), (3, 3, 12)]


def _random_words(ps, d, depth, seed):
    """Makes the projection anew each time: a module's buffer of words is the projection's own tensor."""
    rng = random.Random(seed)
    # (from one letter up, so that the letter bounds of two lists differ)
    low = rng.randrange(d - 1)
    letter = rng.randrange(d)
    words = {tuple(rng.randrange(low, d) for _ in range(depth)) for _ in range(9)}
    while len(words) < 9:
        words.add(tuple(rng.randrange(d) for _ in range(depth)))
    return lambda: ps.projections.words([(letter,)] + sorted(words), depth=depth, path_dim=d)


def _want(path, depth, make, G):
    proj = make()
    x = path.clone().requires_grad_(True)
    full = TO.logsignature(x, depth, method="inverse_exp")
    out = full.index_select(-1, torch.tensor(TO.projection_columns(path.shape[2], depth, proj.level_sizes, proj._codes)))
    return out.detach(), torch.autograd.grad(out, x, G)[0]


def _agrees(module, path, depth, proj, G):
    want, want_grad = _want(path, depth, proj, G)
    x = path.cuda().requires_grad_(True)
    out = module(x)
    (grad,) = torch.autograd.grad(out, x, G.cuda())
    assert "LogSignatureKeepDirect" in out.grad_fn.name()
    assert rel_err(out, want) < 1e-12 and rel_err(grad, want_grad) < 2e-12


@pytest.fixture
def pair(ps, set_option, request):
    d, depth, L = request.param
    set_option("embed_share", 10 ** 6)
    first, other = (_random_words(ps, d, depth, seed) for seed in (3, 11))
    path = brownian_path(2, L, d, seed=880 + d)
    G = randn((2, first().sig_size), seed=88)
    return depth, first, other, path, G


def _rewrite(module, source, how):
    if how == "load":
        module.load_state_dict(source.state_dict())
    else:  # (leaves the version counters where they are)
        for name in BUFFERS:
            getattr(module, name).data.copy_(getattr(source, name))


@pytest.mark.parametrize("pair", SHAPES, indirect=True)
@pytest.mark.parametrize("how", ["load", "data"])
def test_rewritten_buffers_copies_and_pickles(ps, pair, how):
    depth, first, other, path, G = pair
    module = ps.LogSignature(depth=depth, projection=first())
    source = ps.LogSignature(depth=depth, projection=other())
    _rewrite(module, ps.LogSignature(depth=depth, projection=first()), how)
    _agrees(module, path, depth, first, G)
    _rewrite(module, source, how)
    twin = copy.deepcopy(module)
    file = io.BytesIO()
    torch.save(module, file)
    file.seek(0)
    read = torch.load(file, weights_only=False)  # (written three lines above)
    for m in (twin, read, module):
        _agrees(m, path, depth, other, G)
    tensors = {id(b) for b in module.buffers()}
    assert all(id(t) in tensors for t in module.__dict__.values() if isinstance(t, torch.Tensor))


@pytest.mark.parametrize("pair", SHAPES, indirect=True)
def test_captured_graph_follows_the_buffers(ps, pair):
    """Captured before any eager call of the module; an eager call before the first replay; then the lists of words
    are rewritten between replays."""
    depth, first, other, path, G = pair
    module = ps.LogSignature(depth=depth, projection=first())
    x, g = path.cuda().requires_grad_(True), G.cuda()
    warm = ps.LogSignature(depth=depth, projection=other())
    side = torch.cuda.Stream()
    side.wait_stream(torch.cuda.current_stream())
    with torch.cuda.stream(side):
        torch.autograd.grad(warm(x), x, g)
    torch.cuda.current_stream().wait_stream(side)
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        out = module(x)
        (grad,) = torch.autograd.grad(out, x, g)
    _agrees(module, path, depth, first, G)
    for proj in (first, other, first, other):
        want, want_grad = _want(path, depth, proj, G)
        module.load_state_dict(ps.LogSignature(depth=depth, projection=proj()).state_dict())
        out.detach().fill_(float("nan"))
        grad.fill_(float("nan"))
        graph.replay()
        torch.cuda.synchronize()
        assert rel_err(out, want) < 1e-12 and rel_err(grad, want_grad) < 2e-12
        _agrees(module, path, depth, proj, G)


@pytest.mark.parametrize("pair", SHAPES, indirect=True)
def test_calls_on_several_streams_after_a_rewrite(ps, pair):
    depth, first, other, path, G = pair
    module = ps.LogSignature(depth=depth, projection=first())
    want, want_grad = _want(path, depth, other, G)
    x, g = path.cuda().requires_grad_(True), G.cuda()
    module.load_state_dict(ps.LogSignature(depth=depth, projection=other()).state_dict())
    streams = [torch.cuda.Stream() for _ in range(3)]
    results = []
    for stream in streams * 4:
        stream.wait_stream(torch.cuda.default_stream())  # (buffers and inputs; nothing else is shared)
        with torch.cuda.stream(stream):
            out = module(x)
            results.append((out, torch.autograd.grad(out, x, g)[0]))
    torch.cuda.synchronize()
    for out, grad in results:
        assert rel_err(out, want) < 1e-12 and rel_err(grad, want_grad) < 2e-12


@pytest.mark.parametrize("dtype", [torch.float64, torch.float32])
@pytest.mark.parametrize("pair", SHAPES, indirect=True)
def test_columns_and_words_that_are_none(ps, pair, dtype):
    """Wanted columns and words out of range (a damaged state_dict) are NaN and have no gradient; the others are as
    they were."""
    depth, first, _, path, G = pair
    module = ps.LogSignature(depth=depth, projection=first())
    d, columns = path.shape[2], sum(module._ext_level_sizes)
    x, g = path.to(dtype).cuda().requires_grad_(True), G.to(dtype).cuda()
    good = module(x)
    assert "LogSignatureKeepDirect" in good.grad_fn.name()  # (the launches that check)
    picked, words = module._indices_from_sig, module._top_words
    n = picked.numel()
    bad_columns = {0: -1, 2: columns, 3: 2 ** 40}
    bad_words = {4: -1, 6: d ** depth, 8: 2 ** 40}  # of the outputs 5, 7 and 9
    lost = torch.zeros(n, dtype=torch.bool, device="cuda")
    lost[[*bad_columns, *(at + 1 for at in bad_words)]] = True
    (want_grad,) = torch.autograd.grad(good, x, g.masked_fill(lost, 0))
    for at, column in bad_columns.items():
        picked[at] = column
    for at, code in bad_words.items():
        words[at] = code
    with torch.no_grad():
        plain = module(x)
    out = module(x)
    (grad,) = torch.autograd.grad(out, x, g)
    assert torch.equal(out.isnan(), lost.expand_as(out)) and torch.equal(plain.isnan(), out.isnan())
    tol = 1e-12 if dtype == torch.float64 else 1e-5
    assert rel_err(out[:, ~lost], good[:, ~lost].detach().cpu().double()) < tol
    assert rel_err(grad, want_grad.cpu().double()) < 2 * tol
