"""Workgroups whose waves divide a (row tile, slice) among themselves along K and add their sums up in LDS: every
number of waves against the one-wave form, which rounds the same slice sums to fp16.  Only the order of the fp32 sums
differs (at most kt + 8 additions behind 64 products each), so the two differ by fp32 noise before the rounding and by
at most two units in the last place of fp16 (2 * 2^-10 of the value) after it, measured from the slab's own scale where
a sum cancels to almost nothing."""
import ctypes
import sys

import numpy as np
import pytest

import synth

pytestmark = pytest.mark.gpu


def launch(product, torch, w, b, n, split_k, pages, waves):
    fn = product.lib().flashllm_hip_launch_spmm
    fn.restype = ctypes.c_int
    fn.argtypes = [ctypes.c_void_p] * 4 + [ctypes.c_int, ctypes.c_void_p] + [ctypes.c_int] * 6
    out = torch.full((split_k * n * w.m,), float("nan"), dtype=torch.float16, device="cuda")
    stream = ctypes.c_void_p(torch.cuda.current_stream().cuda_stream)
    rc = fn(stream, w.comp.data_ptr(), w.offs.data_ptr(), b.data_ptr(), w.k, out.data_ptr(), w.m, n, w.k, split_k, pages, waves)
    assert rc == 0
    torch.cuda.synchronize()
    return out.cpu().numpy()


@pytest.mark.parametrize("n", [8, 16, 32, 64])
@pytest.mark.parametrize("split_k,pages", [(1, 0), (2, 1), (2, 0), (5, 1), (11, 1)])
def test_waves_sharing_a_slice_match_one_wave(product, n, split_k, pages):
    """Eleven k tiles: slices of 11, 6 and 5, 3, and 1 tile, so some waves get no tile at all; tile row 0 starts and
    ends with empty tiles, tile row 1 is empty, tile row 2 dense; three row tiles leave units beyond whole XCDs."""
    import torch

    assert torch.cuda.is_available()
    print(f"waves per slice n={n} split_k={split_k} pages={pages}", flush=True)
    sys.stdout.flush()
    m, k = 384, 704
    a = synth.sparse_matrix(m, k, 0.8, 90, dist="normal", sigma=0.05)
    a[:128, :64] = 0
    a[:128, 640:] = 0
    a[128:256, :] = 0
    a[256:, :] = synth.sparse_matrix(128, k, 0.0, 91, dist="normal", sigma=0.05)
    w = product.SparseWeight(a)
    b = torch.from_numpy(synth.dense_b(k, n, 92, dist="normal")).cuda()
    want = launch(product, torch, w, b, n, split_k, pages, 1).astype(np.float64)
    assert np.all(np.isfinite(want))
    for waves in (2, 4, 8):
        got = launch(product, torch, w, b, n, split_k, pages, waves).astype(np.float64)
        assert np.all(np.isfinite(got))
        # fp32 noise: 704 products of at most 0.25 * 4.5, 2^-24 each, far below half an fp16 unit of the scale
        bound = 2 * 2.0 ** -10 * np.abs(want) + 704 * 1.125 * 2.0 ** -23
        assert np.all(np.abs(got - want) <= bound), (waves, np.max(np.abs(got - want)))


def launch_group(product, torch, w, b, n, split_k, pages, runs):
    fn = product.lib().flashllm_hip_launch_spmm_group
    fn.restype = ctypes.c_int
    fn.argtypes = [ctypes.c_void_p] * 4 + [ctypes.c_int, ctypes.c_void_p] + [ctypes.c_int] * 6
    out = torch.full((split_k * n * w.m,), float("nan"), dtype=torch.float16, device="cuda")
    stream = ctypes.c_void_p(torch.cuda.current_stream().cuda_stream)
    rc = fn(stream, w.comp.data_ptr(), w.offs.data_ptr(), b.data_ptr(), w.k, out.data_ptr(), w.m, n, w.k, split_k, pages, runs)
    assert rc == 0
    torch.cuda.synchronize()
    return out.cpu().numpy()


@pytest.mark.parametrize("n", [128, 384])
@pytest.mark.parametrize("tiles,split_k,pages", [(11, 1, 0), (11, 2, 1), (11, 5, 0), (11, 11, 1), (100, 3, 0), (97, 2, 1)])
@pytest.mark.parametrize("dense", [False, True])
def test_groups_sharing_a_slice_match_one_group(product, n, tiles, split_k, pages, dense):
    """The same for wide B: three groups of four waves on runs of a slice, from runs without a tile (slices of 1 and 3)
    to runs of 11 and 12, 16 and 17; with a dense row tile both kernels hold three rounds of a tile instead of two."""
    import torch

    print(f"groups per slice n={n} tiles={tiles} split_k={split_k} pages={pages} dense={dense}", flush=True)
    m, k = 384, 64 * tiles
    a = synth.sparse_matrix(m, k, 0.8, 93, dist="normal", sigma=0.05)
    a[:128, :64] = 0
    a[128:256, :] = 0
    if dense:
        a[256:, :] = synth.sparse_matrix(128, k, 0.0, 94, dist="normal", sigma=0.05)
    w = product.SparseWeight(a)
    b = torch.from_numpy(synth.dense_b(k, n, 95, dist="normal")).cuda()
    want = launch_group(product, torch, w, b, n, split_k, pages, 1).astype(np.float64)
    got = launch_group(product, torch, w, b, n, split_k, pages, 3).astype(np.float64)
    assert np.all(np.isfinite(want)) and np.all(np.isfinite(got))
    # as above, with k products of at most 0.25 * 4.5
    bound = 2 * 2.0 ** -10 * np.abs(want) + k * 1.125 * 2.0 ** -23
    assert np.all(np.abs(got - want) <= bound), np.max(np.abs(got - want))
