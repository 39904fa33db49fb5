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


@pytest.mark.parametrize("k,split_k", [(1024, 2), (704, 1), (256, 1)])
def test_short_slices_at_64_columns_are_shared(product, k, split_k):
    """Slices of eight, eleven and four tiles on eight row tiles: the call takes several waves for each (17.3 against 11.4
    us with one and eight on 1024 x 1024, Split_K 2), i.e. its slabs are those of one of the several-wave launches."""
    import torch

    m = 1024
    w = product.SparseWeight(synth.sparse_matrix(m, k, 0.8, 99, dist="normal", sigma=0.05))
    b = torch.from_numpy(synth.dense_b(k, 64, 100, dist="normal")).cuda()
    c = torch.full((64 * m,), float("nan"), dtype=torch.float16, device="cuda")
    ws = torch.full((split_k * 64 * m,), float("nan"), dtype=torch.float16, device="cuda")
    product.spmm_partials(w.comp, w.offs, b, c, m, 64, k, ws, split_k)
    got = (c if split_k == 1 else ws).cpu().numpy()
    same = {waves: np.array_equal(got.view(np.uint16), launch(product, torch, w, b, 64, split_k, 0, waves).view(np.uint16))
            for waves in (1, 2, 4, 8) if waves <= k // 64 // split_k}
    assert any(same[waves] for waves in same if waves > 1) and not same[1], same


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
    """The same for wide B: four waves with a quarter of a slice each, from quarters without a tile (slices of 1 and 3)
    to odd ones; with a dense row tile the kernels hold more rounds of a tile in registers."""
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


@pytest.mark.parametrize("sparsity", [0.9, 0.8, 0.7, 0.2, 1.0])  # the three depths of the ring, tiles beyond it, no vectors at all
@pytest.mark.parametrize("tiles", [1, 2, 3, 7, 8, 17])           # runs of an odd number of tiles end with an empty one
def test_quarters_keep_inf_and_nan_where_they_are(product, tiles, sparsity):
    """An Inf or NaN in B shows in its own column only, as with the kernel whose waves share every tile: the empty tile
    behind an odd run multiplies zeros by zeros."""
    import torch

    print(f"quarters inf and nan tiles={tiles} sparsity={sparsity}", flush=True)
    m, k, n = 256, 64 * tiles, 128
    w = product.SparseWeight(synth.sparse_matrix(m, k, sparsity, 104, dist="normal", sigma=0.05))
    dense = synth.dense_b(k, n, 105, dist="normal").reshape(n, k)
    dense[3], dense[77, -1], dense[100, k // 2] = np.inf, np.nan, np.inf
    b = torch.from_numpy(dense).cuda()
    want = launch_group(product, torch, w, b, n, 1, 0, 1).astype(np.float64)
    got = launch_group(product, torch, w, b, n, 1, 0, 4).astype(np.float64)
    assert np.array_equal(np.isnan(got), np.isnan(want)) and np.array_equal(np.isinf(got), np.isinf(want))
    finite = np.isfinite(want)
    # two sums of the same k products, of at most 0.25 * 4.5, in another order
    bound = 2 * 2.0 ** -10 * np.abs(want[finite]) + k * 1.125 * 2.0 ** -23
    assert np.all(np.abs(got[finite] - want[finite]) <= bound)


@pytest.mark.parametrize("sparsity", [0.9, 0.8, 0.7, 0.2, 1.0])
@pytest.mark.parametrize("tiles,split_k,pages", [(1, 1, 0), (3, 1, 0), (7, 2, 1), (8, 3, 0), (17, 1, 0)])
def test_quarters_at_64_columns_match_one_wave(product, tiles, split_k, pages, sparsity):
    """N = 64: the one-wave form leaves tiles without vectors out, so an Inf or NaN opposite such a tile does not show."""
    import torch

    print(f"quarters at 64 columns tiles={tiles} split_k={split_k} pages={pages} sparsity={sparsity}", flush=True)
    m, k = 384, 64 * tiles
    a = synth.sparse_matrix(m, k, sparsity, 106, dist="normal", sigma=0.05)
    a[:128, -64:] = 0
    w = product.SparseWeight(a)
    dense = synth.dense_b(k, 64, 107, dist="normal").reshape(64, k)
    dense[3, -1], dense[40, -64], dense[50, k // 2] = np.inf, np.nan, np.inf
    b = torch.from_numpy(dense).cuda()
    product.lib().flashllm_hip_set_rows_per_workgroup(1)
    try:
        want = launch(product, torch, w, b, 64, split_k, pages, 1).astype(np.float64)
        got = launch(product, torch, w, b, 64, split_k, pages, 0).astype(np.float64)
    finally:
        product.lib().flashllm_hip_set_rows_per_workgroup(0)
    assert np.array_equal(np.isnan(got), np.isnan(want)) and np.array_equal(np.isinf(got), np.isinf(want))
    finite = np.isfinite(want)
    # two sums of the same k products, of at most 0.25 * 4.5, in another order
    bound = 2 * 2.0 ** -10 * np.abs(want[finite]) + k * 1.125 * 2.0 ** -23
    assert np.all(np.abs(got[finite] - want[finite]) <= bound)
