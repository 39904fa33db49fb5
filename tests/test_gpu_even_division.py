"""Wide B with the k tiles of all (row tile, 128 columns) divided evenly among the workgroups: shares that begin and end
anywhere in a unit, span several units or a part of one, and workgroups without any, against the product in 64 bits."""
import ctypes

import numpy as np
import pytest

import synth

pytestmark = pytest.mark.gpu


def launch(product, torch, w, b, n, share, relu=0):
    fn = product.lib().flashllm_hip_launch_spmm_even
    fn.restype = ctypes.c_int
    fn.argtypes = [ctypes.c_void_p] * 4 + [ctypes.c_int] + [ctypes.c_void_p] * 2 + [ctypes.c_int] * 5
    kt = w.k // 64
    assert share * 256 >= w.m // 128 * (n // 128) * kt
    c = torch.full((n * w.m,), float("nan"), dtype=torch.float16, device="cuda")
    ws = torch.full((((kt - 1) // share + 2) * n * w.m,), float("nan"), dtype=torch.float16, device="cuda")
    stream = ctypes.c_void_p(torch.cuda.current_stream().cuda_stream)
    rc = fn(stream, w.comp.data_ptr(), w.offs.data_ptr(), b.data_ptr(), w.k, c.data_ptr(), ws.data_ptr(), w.m, n, w.k, share, relu)
    assert rc == 0
    torch.cuda.synchronize()
    return c


@pytest.mark.parametrize("sparsity", [0.9, 0.8, 0.7, 0.2, 1.0])
@pytest.mark.parametrize("m,n,tiles,share", [(384, 128, 1, 1), (384, 256, 7, 5), (640, 128, 11, 3), (640, 384, 20, 2), (384, 128, 20, 64),
                                             (128, 128, 40, 13), (1152, 256, 9, 9)])
def test_even_shares(product, m, n, tiles, share, sparsity):
    import torch

    print(f"even shares m={m} n={n} tiles={tiles} share={share} sparsity={sparsity}", flush=True)
    k = 64 * tiles
    a = synth.sparse_matrix(m, k, sparsity, 111, dist="normal", sigma=0.05)
    a[:128, :64] = 0
    w = product.SparseWeight(a)
    dense = synth.dense_b(k, n, 112, dist="normal").reshape(n, k)
    b = torch.from_numpy(dense).cuda()
    got = launch(product, torch, w, b, n, share)
    want = dense.astype(np.float64) @ a.astype(np.float64).T
    size = np.abs(dense).astype(np.float64) @ np.abs(a).astype(np.float64).T
    # every part and the sum are rounded to fp16 (2^-11 of at most `size`, and half its smallest step), fp32 sums of k products
    parts = min((tiles - 1) // share + 2, tiles)
    bound = (parts + 1) * (2.0 ** -11 * size / 2 + 2.0 ** -25) + 2.0 ** -11 * np.abs(want) + k * 2.0 ** -24 * size
    assert np.all(np.abs(got.cpu().numpy().reshape(n, m).astype(np.float64) - want) <= bound)
    relu = launch(product, torch, w, b, n, share, relu=1)
    assert torch.equal(relu, torch.where(got > 0, got, torch.zeros_like(got)))


@pytest.mark.parametrize("sparsity", [0.99, 0.88, 0.75, 0.6])  # the four depths of the ring
@pytest.mark.parametrize("share", [9, 16])               # runs of parts of a unit, and of whole units
def test_even_shares_with_a_few_long_tiles(product, share, sparsity):
    import torch

    print(f"even shares with long tiles share={share} sparsity={sparsity}", flush=True)
    m, k, n = 512, 64 * 16, 128
    a = synth.sparse_matrix(m, k, sparsity, 113, dist="normal", sigma=0.05)
    for row_tile, tile in enumerate((0, 5, 10, 15)):
        a[128 * row_tile:128 * row_tile + 128, 64 * tile:64 * tile + 64] = 0.05
    w = product.SparseWeight(a)
    dense = synth.dense_b(k, n, 114, dist="normal").reshape(n, k)
    got = launch(product, torch, w, torch.from_numpy(dense).cuda(), n, share)
    want = dense.astype(np.float64) @ a.astype(np.float64).T
    size = np.abs(dense).astype(np.float64) @ np.abs(a).astype(np.float64).T
    bound = 4 * (2.0 ** -11 * size / 2 + 2.0 ** -25) + 2.0 ** -11 * np.abs(want) + k * 2.0 ** -24 * size  # as above, three parts
    assert np.all(np.abs(got.cpu().numpy().reshape(n, m).astype(np.float64) - want) <= bound)


def test_a_call_takes_it_and_keeps_inf_and_nan_where_they_are(product):
    """36864 x 9216, N = 128, Split_K 3 (864 workgroups of whole slices; 256 shares of 162 tiles): the call's C is this kernel's."""
    import torch

    print("even shares through the call", flush=True)
    m, k, n, split_k = 36864, 9216, 128, 3
    g = torch.Generator(device="cuda").manual_seed(7)
    a = torch.empty(m, k, dtype=torch.float16, device="cuda").normal_(0.0, 0.02, generator=g)
    a.masked_fill_(torch.rand(m, k, device="cuda", generator=g) >= 0.2, 0.0)
    comp, offs = product.device_compress(a)
    b = torch.empty(n, k, dtype=torch.float16, device="cuda").normal_(generator=g)
    b[5, 100], b[77, -1] = float("inf"), float("nan")
    c = torch.full((n * m,), float("nan"), dtype=torch.float16, device="cuda")
    ws = torch.full((split_k * n * m,), float("nan"), dtype=torch.float16, device="cuda")
    product.spmm_splitk(comp, offs, b, c, m, n, k, ws, split_k)

    class Weight:
        pass

    w = Weight()
    w.m, w.k, w.comp, w.offs = m, k, comp, offs
    assert torch.equal(c.view(torch.int16), launch(product, torch, w, b, n, 162).view(torch.int16))
    c = c.view(n, m)
    others = torch.tensor([i for i in range(n) if i not in (5, 77)], device="cuda")
    assert bool(torch.isfinite(c[others]).all()) and not bool(torch.isfinite(c[77]).any())
    rows = torch.arange(0, m, 97, device="cuda")
    want = b[others].double() @ a[rows].double().t()
    assert float((c[others][:, rows].double() - want).norm() / want.norm()) <= 5e-4


@pytest.mark.parametrize("m,k,n,split_k", [(43008, 5440, 128, 3), (19072, 4288, 256, 6), (27264, 3136, 384, 3)])
def test_calls_that_gain_little_keep_their_slices(product, m, k, n, split_k):
    """Products that an even division makes slower (107 us instead of 94, 71 and 61, 115 and 105 with rows of uneven density): the
    call's C is that of its two halves, which have Split_K slices."""
    import torch

    print(f"slices kept m={m} k={k} n={n} split_k={split_k}", flush=True)
    g = torch.Generator(device="cuda").manual_seed(m)
    a = torch.empty(m, k, dtype=torch.float16, device="cuda").normal_(0.0, 0.02, generator=g)
    a.masked_fill_(torch.rand(m, k, device="cuda", generator=g) >= 0.3, 0.0)
    comp, offs = product.device_compress(a)
    b = torch.empty(n * k, dtype=torch.float16, device="cuda").normal_(generator=g)
    c, want = torch.empty(n * m, dtype=torch.float16, device="cuda"), torch.empty(n * m, dtype=torch.float16, device="cuda")
    ws = torch.empty(split_k * n * m, dtype=torch.float16, device="cuda")
    product.spmm_splitk(comp, offs, b, c, m, n, k, ws, split_k)
    product.spmm_partials(comp, offs, b, want, m, n, k, ws, split_k)
    product.splitk_reduce(want, ws, m, n, split_k)
    assert torch.equal(c.view(torch.int16), want.view(torch.int16))


@pytest.mark.parametrize("sparsity", [0.99, 0.88, 0.75, 0.6])  # the four depths of the ring
def test_positions_beyond_the_tile_stay_inside_it(product, sparsity):
    import copy

    import torch

    print(f"even shares, positions beyond the tile, sparsity={sparsity}", flush=True)
    m, k, n = 512, 64 * 16, 128
    a = synth.sparse_matrix(m, k, sparsity, 115, dist="normal", sigma=0.05)
    a[128:256, 320:384] = 0.5  # and a tile longer than the ring
    w = product.SparseWeight(a)
    b = torch.from_numpy(synth.dense_b(k, n, 116, dist="normal")).cuda()
    damaged = copy.copy(w)
    damaged.comp = w.comp ^ (torch.randint(0, 8, w.comp.shape, dtype=torch.int32, device="cuda") << 29)
    assert torch.equal(launch(product, torch, damaged, b, n, 9), launch(product, torch, w, b, n, 9))
