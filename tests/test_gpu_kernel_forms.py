"""Every form a product can take, launched by itself: the kernel for N <= 64 with 1, 2, 4 or 8 waves per slice or eight row
tiles per workgroup, four waves with a quarter of a slice each at N = 64 and wide B, the four-wave and the 256-column kernel.  Each with the
activation stored with the sums, with B's columns farther apart than K (the attention-output linear reads B so), and on a
matrix without nonzeros, whose Compressed_A holds a single item; the results are compared bit for bit with the plain form's."""
import ctypes

import numpy as np
import pytest

import synth

pytestmark = pytest.mark.gpu

# kernel, N, waves or groups per slice; "rows8" stands for eight row tiles per workgroup
FORMS = ([("stream", n, waves) for n in (8, 16, 32, 64) for waves in (1, 2, 4, 8)] + [("rows8", 64, 1), ("stream", 64, 0)]
         + [("group", n, runs) for n in (128, 384) for runs in (1, 3)] + [("wide", 256, 1), ("wide", 512, 1)])
M, K, SPLIT_K = 3072, 704, 3           # eleven k tiles: slices of 4, 4 and 3
WIDE_M, WIDE_SPLIT_K = 128 * 132, 3    # enough workgroups for 256 columns each

RELU = 2


def launch(product, torch, form, w, b, ldb, out, split_k, store):
    kernel, n, waves = form
    L = product.lib()
    fn = L.flashllm_hip_launch_spmm if kernel in ("stream", "rows8") else L.flashllm_hip_launch_spmm_group
    fn.restype = ctypes.c_int
    fn.argtypes = [ctypes.c_void_p] * 4 + [ctypes.c_int, ctypes.c_void_p] + [ctypes.c_int] * 6
    columns = L.flashllm_hip_columns_per_workgroup
    columns.restype, columns.argtypes = ctypes.c_int, [ctypes.c_int] * 3
    if kernel in ("group", "wide"):
        assert columns(n, w.m, split_k) == (256 if kernel == "wide" else 128)
    L.flashllm_hip_set_rows_per_workgroup(8 if kernel == "rows8" else 1)
    try:
        stream = ctypes.c_void_p(torch.cuda.current_stream().cuda_stream)
        rc = fn(stream, w.comp.data_ptr(), w.offs.data_ptr(), b.data_ptr(), ldb, out.data_ptr(), w.m, n, w.k, split_k, store, waves)
    finally:
        L.flashllm_hip_set_rows_per_workgroup(0)
    assert rc == 0
    torch.cuda.synchronize()
    return out


def nan_halfs(torch, count):
    return torch.full((count,), float("nan"), dtype=torch.float16, device="cuda")


def same_bits(torch, x, y):
    return torch.equal(x.view(torch.int16), y.view(torch.int16))


@pytest.fixture(scope="module")
def weights(product):
    """By (kernel, split into slices or not): M x K with an empty row tile and a dense one, enough rows for the kernel."""
    cache = {}

    def weight(kernel, split_k):
        wide = kernel == "wide"
        m, k = (WIDE_M if split_k > 1 else 51200, K if split_k > 1 else 192) if wide else (M, K)
        if (m, k) not in cache:
            a = synth.sparse_matrix(m, k, 0.8, m + k, dist="normal", sigma=0.05)
            a[:128] = 0
            a[256:384] = synth.sparse_matrix(128, k, 0.0, 5, dist="normal", sigma=0.05)
            cache[m, k] = product.SparseWeight(a)
        return cache[m, k]

    return weight


@pytest.mark.parametrize("form", FORMS, ids=lambda f: "-".join(map(str, f)))
def test_activation_is_that_of_the_plain_store(product, weights, form):
    import torch

    print("activation", form, flush=True)
    kernel, n, _ = form
    w = weights(kernel, 1)
    b = torch.from_numpy(synth.dense_b(w.k, n, 101, dist="normal")).cuda().view(-1)
    b[:w.k] = float("nan")  # a column of NaN is 0 behind the activation
    plain = launch(product, torch, form, w, b, w.k, nan_halfs(torch, n * w.m), 1, 0)
    got = launch(product, torch, form, w, b, w.k, nan_halfs(torch, n * w.m), 1, RELU)
    assert bool(torch.isnan(plain[256:w.m]).any()) and bool((plain[w.m:] < 0).any()) and bool((plain[w.m:] > 0).any())
    assert same_bits(torch, got, torch.where(plain > 0, plain, torch.zeros_like(plain)))


@pytest.mark.parametrize("split_k,store", [(1, 0), (3, 0), (3, 1)])  # C, plain slabs, slabs by workgroup
@pytest.mark.parametrize("form", FORMS, ids=lambda f: "-".join(map(str, f)))
def test_columns_of_b_farther_apart_than_k(product, weights, form, split_k, store):
    import torch

    print("leading dimension", form, split_k, store, flush=True)
    kernel, n, _ = form
    w = weights(kernel, split_k)
    dense = torch.from_numpy(synth.dense_b(w.k, n, 102, dist="normal")).cuda().view(n, w.k)
    apart = nan_halfs(torch, n * (w.k + 72)).view(n, w.k + 72)  # what lies between the columns must not be multiplied
    apart[:, :w.k] = dense
    want = launch(product, torch, form, w, dense, w.k, nan_halfs(torch, split_k * n * w.m), split_k, store)
    got = launch(product, torch, form, w, apart, w.k + 72, nan_halfs(torch, split_k * n * w.m), split_k, store)
    assert bool(torch.isfinite(want).all())
    assert same_bits(torch, got, want)


@pytest.mark.parametrize("form", FORMS, ids=lambda f: "-".join(map(str, f)))
@pytest.mark.parametrize("split_k", [1, 3])
def test_matrix_without_nonzeros(product, form, split_k):
    import torch

    print("empty matrix", form, split_k, flush=True)
    kernel, n, _ = form
    m, k = (WIDE_M if split_k > 1 else 51200, K if split_k > 1 else 192) if kernel == "wide" else (M, K)
    w = product.SparseWeight(np.zeros((m, k), dtype=np.float16))
    assert w.comp.numel() == 1 and w.nnz == 0
    b = torch.from_numpy(synth.dense_b(k, n, 103, dist="normal")).cuda()
    got = launch(product, torch, form, w, b, k, nan_halfs(torch, split_k * n * m), split_k, 0)
    assert bool((got == 0).all())


@pytest.mark.parametrize("form", FORMS, ids=lambda f: "-".join(map(str, f)))
def test_positions_beyond_the_tile_stay_inside_it(product, weights, form):
    """An item's position has 13 bits; the three above them, which a damaged Compressed_A may have set, change nothing: no item leaves
    the tile of the wave that stores it."""
    import copy

    import torch

    print("positions beyond the tile", form, flush=True)
    _, n, _ = form
    w = weights(form[0], 3)
    b = torch.from_numpy(synth.dense_b(w.k, n, 104, dist="normal")).cuda()
    damaged = copy.copy(w)
    damaged.comp = w.comp ^ (torch.randint(0, 8, w.comp.shape, dtype=torch.int32, device="cuda") << 29)
    assert not torch.equal(damaged.comp, w.comp)
    want = launch(product, torch, form, w, b, w.k, nan_halfs(torch, 3 * n * w.m), 3, 0)
    got = launch(product, torch, form, damaged, b, w.k, nan_halfs(torch, 3 * n * w.m), 3, 0)
    assert bool(torch.isfinite(want).all()) and same_bits(torch, got, want)
