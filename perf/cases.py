"""Workloads whose time matters: what a program that uses this package has it do, from one short path that is
answered while someone waits to training batches that fill the device.

A case is a dict of plain values:

* `op`: "sig" (`Signature`) or "logsig" (`LogSignature`); `dtype`: "f32" or "f64";
* `B`, `L`, `d`, `depth`: paths, points per path, channels, truncation depth;
* `win`, `stride`: length and stride of sliding windows over the points (0: no windows);
* `proj`: "none", "lyndon", "words" (levels 1 and 2 in full and `words` random words of the lengths above) or
  "aniso" (letter weights spread over [1, 2], threshold 1.25 * depth);
* `grad`: True for a training step (forward and the gradient of the path), False for inference.
"""
import math
import random

import torch

import pathsig_amd as pathsig

_DTYPE = {"f32": torch.float32, "f64": torch.float64}


def _case(name, op, B, L, d, depth, dtype="f32", grad=True, win=0, stride=0, proj="none", words=0):
    return dict(name=name, op=op, B=B, L=L, d=d, depth=depth, dtype=dtype, grad=grad, win=win, stride=stride,
                proj=proj, words=words)


def listed():
    return [
        # one short path of three channels, as a service gets them: nothing but latency
        _case("one_short_path", "sig", 1, 32, 3, 4, grad=False),
        # the batch of the quick start, as the layer of a small model in training: launches and host time
        _case("small_logsig_step", "logsig", 32, 128, 8, 4),
        # features of a small batch, no gradient (the repository's benchmark configuration c1)
        _case("batch_features", "sig", 32, 128, 8, 4, grad=False),
        # ordinary training batch, few channels and a deep truncation (benchmark configuration c2, the headline)
        _case("deep_step", "sig", 128, 1024, 4, 6),
        # overlapping sliding windows of every path (benchmark configuration c3)
        _case("windows_step", "sig", 64, 2048, 6, 5, win=64, stride=32),
        # a chosen set of words over a wide alphabet (benchmark configuration c4)
        _case("words_step", "sig", 256, 512, 16, 6, proj="words", words=2048),
        # log-signature in its minimal coordinates (benchmark configuration c5), in both precisions
        _case("lyndon_step", "logsig", 128, 1024, 8, 5, proj="lyndon"),
        _case("lyndon_step_f64", "logsig", 128, 1024, 8, 5, dtype="f64", proj="lyndon"),
        # log-signatures of sliding windows, as the input of a sequence model: thousands of short rows
        _case("lyndon_windows_step", "logsig", 32, 4096, 6, 4, win=64, stride=32, proj="lyndon"),
        # a handful of very long paths (tick data)
        _case("long_paths_step", "sig", 4, 20001, 3, 6),
        # sizes that fit nothing, in double precision (gradient checks, ill-conditioned fits)
        _case("odd_sizes_step_f64", "sig", 50, 333, 7, 5, dtype="f64"),
        # the largest: a training batch that fills the device
        _case("large_step", "sig", 256, 2048, 8, 5),
    ]


def _dense_size(d, depth):
    return sum(d ** k for k in range(1, depth + 1))


def _num_windows(case):
    return (case["L"] - case["win"]) // case["stride"] + 1 if case["win"] else 1


def _increments(case):
    return _num_windows(case) * (case["win"] - 1) if case["win"] else case["L"] - 1


def _nodes_dense(d, depth):
    return sum(d ** j for m in range(1, depth + 1) for j in range(1, m + 1))


def _log_size(rng, lo, hi):
    return max(lo, min(hi, round(math.exp(rng.uniform(math.log(lo), math.log(hi))))))


def draw(rng):
    """One more case of the ranges above: 1 to 512 paths of 16 to 4096 points (up to 16 paths of up to 20001), 2 to
    16 channels, depth 2 to 8 as long as a signature has at most 70 000 coefficients, both precisions, with and
    without gradient, windows and projections."""
    most_flops = 6.0 * _nodes_dense(8, 5) * 2047 * 256
    while True:
        op = "sig" if rng.random() < 0.6 else "logsig"
        B = _log_size(rng, 1, 512)
        L = _log_size(rng, 16, 20001 if B <= 16 else 4096)
        d = rng.randint(2, 16)
        depth = rng.randint(2, 8)
        dtype = "f64" if rng.random() < 0.25 else "f32"
        grad = rng.random() < 0.7
        win = stride = words = 0
        if rng.random() < 0.25 and 64 <= L <= 4096:
            win = _log_size(rng, 8, min(256, L // 2))
            stride = max(1, round(win * rng.choice((0.25, 0.5, 1.0))))
        if op == "logsig":
            proj = "lyndon" if rng.random() < 0.6 else "none"
        else:
            proj = rng.choices(("none", "words", "aniso"), (0.7, 0.2, 0.1))[0]
        if depth < 3 and proj != "none":
            proj = "none"
        if proj == "words":
            words = min(_log_size(rng, 16, 2048), d ** depth // 4)
            if words < 16:
                proj, words = "none", 0
        case = dict(op=op, B=B, L=L, d=d, depth=depth, dtype=dtype, grad=grad, win=win, stride=stride, proj=proj,
                    words=words)
        rows = B * _num_windows(case)
        if proj == "words":
            # (no limit on the dense size: the words are few)
            if rows * _increments(case) // _num_windows(case) * (words + d + d * d) > 256 * 511 * 2320 or L > 4096:
                continue
        else:
            if _dense_size(d, depth) > 70000 or rows * _dense_size(d, depth) > 40e6:
                continue
            if 6.0 * _nodes_dense(d, depth) * _increments(case) * B > most_flops:
                continue
        return case


def _word_list(case):
    """The chosen words: distinct, of lengths 3 to depth, every length and letter equally likely."""
    rng = random.Random(20240)
    seen, out = set(), []
    while len(out) < case["words"]:
        w = tuple(rng.randrange(case["d"]) for _ in range(rng.randint(3, case["depth"])))
        if w not in seen:
            seen.add(w)
            out.append(w)
    return sorted(out, key=len)


def _projection(case):
    d, depth = case["d"], case["depth"]
    if case["proj"] == "lyndon":
        return pathsig.projections.lyndon(depth=depth, path_dim=d)
    if case["proj"] == "words":
        return pathsig.projections.words(_word_list(case), depth=depth, path_dim=d, full_levels=(1, 2))
    if case["proj"] == "aniso":
        weights = [1.0 + i / (d - 1) for i in range(d)]
        return pathsig.projections.anisotropic(weights, 1.25 * depth, depth=depth, path_dim=d)
    return None


def prepare(case, seed):
    """Brownian paths of unit variance at the end, the module with its plan, and the gradient from above."""
    dtype = _DTYPE[case["dtype"]]
    B, L, d = case["B"], case["L"], case["d"]
    gen = torch.Generator(device="cuda").manual_seed(seed)
    steps = torch.randn(B, L, d, dtype=torch.float64, device="cuda", generator=gen) / math.sqrt(L)
    steps[:, 0] = 0
    path = steps.cumsum(dim=1).to(dtype)
    windows = None
    if case["win"]:
        starts = torch.arange(_num_windows(case), device="cuda") * case["stride"]
        windows = torch.stack([starts, starts + case["win"]], dim=1)
    proj = _projection(case)
    module = pathsig.Signature if case["op"] == "sig" else pathsig.LogSignature
    module = module(depth=case["depth"], projection=proj, windows=windows)
    if not case["grad"]:
        return {"module": module, "path": path}
    size = _dense_size(d, case["depth"]) if proj is None else proj.sig_size
    shape = (B, _num_windows(case), size) if case["win"] else (B, size)
    upstream = torch.randn(shape, dtype=dtype, device="cuda", generator=gen)
    return {"module": module, "path": path.requires_grad_(True), "upstream": upstream}


def run(state):
    if "upstream" not in state:
        with torch.no_grad():
            return state["module"](state["path"])
    out = state["module"](state["path"])
    (grad,) = torch.autograd.grad(out, state["path"], state["upstream"])
    return out, grad


def _wanted(case):
    """Per level: None where every word is wanted, else the set of codes of the wanted words."""
    d, depth = case["d"], case["depth"]
    proj = _projection(case)
    if proj is None:
        return [None] * depth
    codes, pos, wanted = proj.encoded_words.tolist(), 0, []
    for k in range(1, depth + 1):
        size = proj.level_sizes[k]
        if size == d ** k:
            wanted.append(None)
        else:
            wanted.append(set(codes[pos:pos + size]))
            pos += size
    if case["op"] == "logsig":  # the logarithm reads every word below the top level
        wanted[:-1] = [None] * (depth - 1)
    return wanted


def _nodes(case):
    """Multiply-adds of one increment: the words of length m and all their prefixes form a tree whose nodes each take
    one (Horner's rule for S (x) exp(dx)); prefixes of wanted words have to be carried too."""
    d, depth = case["d"], case["depth"]
    wanted = _wanted(case)
    total = 0
    for m in range(1, depth + 1):
        closure = set()
        for n in range(m, depth + 1):
            if wanted[n - 1] is None:
                closure = None
                break
            closure.update(c // d ** (n - m) for c in wanted[n - 1])
        if closure is None:
            total += sum(d ** j for j in range(1, m + 1))
        else:
            total += sum(len({c // d ** (m - j) for c in closure}) for j in range(1, m + 1))
    return total


def work(case):
    """Bytes: the paths and the results once (and in a step the two gradients).  Flops: the multiply-adds of the
    sweep over the increments, of the logarithm (n (n - 1) / 2 for a word of length n), and twice both for the
    gradient."""
    d, depth, B = case["d"], case["depth"], case["B"]
    item = 4 if case["dtype"] == "f32" else 8
    rows = B * _num_windows(case)
    proj = _projection(case)
    size = _dense_size(d, depth) if proj is None else proj.sig_size
    flops = 2.0 * _nodes(case) * _increments(case) * B
    if case["op"] == "logsig":
        top = d ** depth if proj is None else proj.level_sizes[depth]
        flops += rows * (sum(d ** n * n * (n - 1.0) for n in range(1, depth)) + top * depth * (depth - 1.0))
    values = B * case["L"] * d + rows * size
    return {"bytes": item * values * (2 if case["grad"] else 1), "flops": flops * (3 if case["grad"] else 1)}


def tolerance(case):
    """Sums over time in the order an implementation likes; the gradient of a logarithm is a difference of larger
    terms."""
    rel = 1e-5 if case["dtype"] == "f32" else 1e-12
    return {"rel": 2 * rel if case["op"] == "logsig" else rel}
