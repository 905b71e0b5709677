"""A forward hands its backward a buffer whose layout the tuning switches decide, and its size tells which: no two layouts
of a call have the same size (host side), and a backward that meets other switches recomputes (`-m gpu`)."""
import ctypes

import pytest
import torch

from .helpers import brownian_path, randn, rel_err


def _sizes(call):
    from pathsig_amd import _load
    lib, (dtype, B, L, d, depth, levels, kind) = _load.lib(), call
    host = None if levels is None else (ctypes.c_int64 * len(levels))(*levels)
    if kind == "sig":
        return lib.pathsig_sig_chunks_bytes(dtype, B, L, d, depth, host, 0)
    saved, forward, backward = ctypes.c_size_t(), ctypes.c_size_t(), ctypes.c_size_t()
    lib.pathsig_logsignature_sizes.argtypes = [ctypes.c_int] + [ctypes.c_int64] * 3 + [
        ctypes.c_int, ctypes.c_void_p, ctypes.c_int64] + [ctypes.POINTER(ctypes.c_size_t)] * 3
    lib.pathsig_logsignature_sizes(dtype, B, L, d, depth, host, 0, saved, forward, backward)
    return saved.value


# the smallest rows (sizes that any rounding would make equal), groups of four, a projection whose rows are swept with
# and without a second chunk, one that the switches move to the per-word kernels
@pytest.mark.parametrize("dtype", [0, 1])
@pytest.mark.parametrize("B,L,d,depth,levels", [
    (1, 60, 2, 2, None), (1, 60, 2, 3, None), (5, 60, 2, 3, None), (1, 5000, 2, 3, None), (3, 400, 4, 6, None),
    (2, 60, 3, 4, [0, 3, 9, 27, 20]), (2, 60, 2, 4, [0, 2, 4, 8, 3]), (2, 60, 3, 4, [0, 3, 4, 27, 81])])
def test_sizes_tell_the_layouts_apart(set_option, dtype, B, L, d, depth, levels):
    set_option("embed_share", 10 ** 6)
    for kind in ("sig", "logsig") if levels is None or levels[2] == d * d else ("sig",):
        seen = {}
        for tiled in (1, 0):
            set_option("tiled", tiled)
            for grouped in (1, 0):
                set_option("grouped", grouped)
                for chunks in (*range(1, 70), 255, 256, 1000, 1023, 1024):
                    set_option("chunks", chunks)
                    size = _sizes((dtype, B, L, d, depth, levels, kind))
                    if size == 0:
                        continue  # nothing is handed over
                    # (in fp64, and where four does not divide the chunks, the switch for groups changes nothing)
                    same = (tiled, chunks if tiled else 0)
                    assert seen.setdefault(size, (same, grouped))[0] == same
        assert seen


@pytest.mark.gpu
@pytest.mark.parametrize("dtype", [torch.float64, torch.float32])
@pytest.mark.parametrize("name", ["Signature", "LogSignature"])
@pytest.mark.parametrize("B,before,after", [(1, {"chunks": 2}, {"chunks": 5}), (5, {"chunks": 1}, {"chunks": 2}),
                                            (2, {"chunks": 8}, {"chunks": 8, "grouped": 0}),
                                            (2, {"chunks": 3}, {"chunks": 3, "tiled": 0}), (3, {"chunks": 4}, {"chunks": 1})])
def test_switches_that_change_between_forward_and_backward(set_option, dtype, name, B, before, after):
    import pathsig_amd as ps
    x = brownian_path(B, 60, 2, seed=910).to(dtype).cuda().requires_grad_(True)
    module = getattr(ps, name)(depth=3)
    for option, value in before.items():
        set_option(option, value)
    out = module(x)
    g = randn(tuple(out.shape), seed=91).to(dtype).cuda()
    (want,) = torch.autograd.grad(out, x, g, retain_graph=True)
    for option, value in after.items():
        set_option(option, value)
    (got,) = torch.autograd.grad(out, x, g)
    assert rel_err(got, want) < (1e-12 if dtype == torch.float64 else 1e-5)
