"""Scratch of the launches for long chains of time chunks: asked for where they are taken, and never at the price of a call
that the allocation-free backward can serve without them."""
import ctypes

import pytest
import torch

from .helpers import rel_err
from .test_zz_no_alloc import STATIC_BYTES, TOL, _both


@pytest.fixture(scope="module")
def lib():
    from pathsig_amd import _load
    return _load.lib()


# Sixteen chunks, whose products take one launch: the increment sums and three arrays of [rows, chunks, 1364] values.
@pytest.mark.parametrize("B", [128, 160])
def test_no_scratch_for_launches_that_are_not_made(lib, B):
    L, d, depth, low = 1024, 4, 6, 1364
    chunks = lib.pathsig_sig_forward_workspace(0, B, L, d, depth, None, 0) // (B * 4 * (low + 4 ** 6 + low))
    assert chunks == 16
    need = lib.pathsig_sig_backward_workspace(0, B, L, d, depth, None, 0)
    assert need <= B * (L - 1) * d * 4 + 3 * B * chunks * low * 4 + 4 * 256
    assert need < STATIC_BYTES


@pytest.mark.gpu
@pytest.mark.parametrize("dtype,B,L,beyond", [(torch.float32, 160, 1024, False), (torch.float64, 8, 6000, True),
                                              (torch.float64, 4, 12001, True)])
def test_allocation_free_backward_goes_without_the_chains(lib, dtype, B, L, beyond):
    rc, need, got, want = _both(lib, dtype, B, L, 4, 6)
    assert (need > STATIC_BYTES) == beyond  # what the call takes with a workspace of its own
    assert rc == 0, lib.pathsig_last_error()
    assert rel_err(got, want) < TOL[dtype]
    # (the choice ends with the call)
    assert lib.pathsig_sig_backward_workspace(0 if dtype == torch.float32 else 1, B, L, 4, 6, None, 0) == need


# Windows lie in device memory, so their lengths are not known where the chunks are chosen: a few short windows of a long
# path must not be cut into the hundreds of chunks that the whole path would be worth, nor take the launches for long
# chains where only the length of the path would pay for them.
@pytest.mark.parametrize("dtype,elem", [(0, 4), (1, 8)])
@pytest.mark.parametrize("B,W,L,d,depth,chains", [(1, 10, 20001, 4, 4, False), (1, 1, 20001, 4, 4, False), (1, 3, 4000, 6, 5, True),
                                                  (1, 5, 3500, 3, 6, True)])
def test_windows_are_not_taken_for_rows_as_long_as_the_path(lib, dtype, elem, B, W, L, d, depth, chains):
    whole = lib.pathsig_sig_forward_workspace(dtype, B * W, L, d, depth, None, 0)
    low, rows = sum(d ** k for k in range(1, depth)), B * W
    arrays = 3 if chains else 1  # of the levels below the top, beside the chunk signatures
    bound = rows * 64 * (low + d ** depth + arrays * low) * elem + (1 + arrays) * 256
    assert whole > bound or (elem == 4 and L - 1 > 4096)  # (paths of that length are cut further)
    assert 0 < lib.pathsig_sig_forward_workspace(dtype, B, L, d, depth, None, W) <= bound
    products = (2 + arrays) * (rows * 64 * low * elem + 256)
    assert lib.pathsig_sig_backward_workspace(dtype, B, L, d, depth, None, W) <= B * (L - 1) * d * elem + 256 + products
    assert lib.pathsig_sig_forward_workspace(dtype, B * W, L, d, depth, None, 0) == whole


@pytest.mark.parametrize("dtype", [0, 1])
@pytest.mark.parametrize("d", [2, 4, 8, 15, 32])
@pytest.mark.parametrize("rows", [512, 1024, 1536])
@pytest.mark.parametrize("L", [257, 1025, 4097])
def test_few_windows_of_depth_two_are_cut_into_chunks(lib, dtype, d, rows, L):
    """512 windows over two letters would be 16 waves of several windows each, every one of which walks its longest window alone:
    up to 2048 rows, calls keep to time chunks."""
    assert lib.pathsig_sig_forward_workspace(dtype, 8, L, d, 2, None, rows // 8) > 0
    assert lib.pathsig_sig_chunks_bytes(dtype, 8, L, d, 2, None, rows // 8) > 0
    assert lib.pathsig_sig_forward_workspace(dtype, 8, L, d, 2, None, 1024) == 0


# Words whose table takes longer to write and read than a short path to sweep, and words that keep the SIMDs busy as it is, are
# swept in one piece; few words of long paths in chunks.
@pytest.mark.parametrize("dtype,B,L,d,depth,top,chunks", [
    (1, 2, 105, 31, 4, 31000, False), (0, 3, 2436, 38, 4, 58000, False), (1, 68, 154, 37, 3, 1400, False), (0, 19, 75, 15, 1, 15, False),
    (0, 2, 2616, 35, 5, 300, True), (1, 40, 2976, 9, 5, 60, True), (0, 1, 928, 23, 8, 90, True)])
def test_words_are_cut_into_chunks_where_a_forward_gains(lib, dtype, B, L, d, depth, top, chunks):
    sizes = (ctypes.c_int64 * (depth + 1))(*[0] * depth, top)
    assert (lib.pathsig_sig_forward_scratch(dtype, B, L, d, depth, sizes, 0) > 0) == chunks
    assert lib.pathsig_sig_forward_workspace(dtype, B, L, d, depth, sizes, 0) == 0


# Far chunks, and short prefixes for their chunks' sake, only where a forward alone gains too.
@pytest.mark.parametrize("dtype,B,L,d,depth,chunks", [
    (1, 7, 109, 56, 3, False), (1, 5, 220, 4, 8, False), (0, 7, 196, 60, 3, False), (1, 21, 937, 16, 4, False), (1, 10, 697, 18, 4, False),
    (0, 2, 4000, 16, 4, True), (1, 13, 2799, 4, 7, True), (1, 8, 1091, 9, 5, True), (1, 35, 500, 32, 3, True), (0, 4, 1000, 9, 5, True)])
def test_far_chunks_are_taken_where_a_forward_gains(lib, dtype, B, L, d, depth, chunks):
    assert (lib.pathsig_sig_forward_workspace(dtype, B, L, d, depth, None, 0) > 0) == chunks
    assert (lib.pathsig_sig_chunks_bytes(dtype, B, L, d, depth, None, 0) > 0) == chunks
