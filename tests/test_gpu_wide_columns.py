"""Workgroups of 256 columns (wide B, enough workgroups to fill the GPU): their slabs against those of the one-wave kernel
on groups of 64 columns, bit for bit (the same products in the same order), and the call's own order of slabs against
the plain one."""
import ctypes

import numpy as np
import pytest

import synth

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("sparsity", [0.8, 0.6, 0.1])  # two rounds of a tile in registers, three, and more than that
@pytest.mark.parametrize("m,k,n,split_k", [(3200, 2240, 256, 16),   # slices of 3 tiles, of 2, and empty ones
                                           (1792, 832, 512, 15),    # slices of one tile
                                           (51200, 192, 256, 1)])   # straight to C
def test_256_columns_match_the_one_wave_kernel(product, m, k, n, split_k, sparsity):
    import torch

    print(f"256 columns m={m} k={k} n={n} split_k={split_k} sparsity={sparsity}", flush=True)
    a = synth.sparse_matrix(m, k, sparsity, 96, dist="normal", sigma=0.05, threads=8)
    a[128:256, :] = 0
    a[:128, :64] = 0
    w = product.SparseWeight(a)
    b = torch.from_numpy(synth.dense_b(k, n, 97, dist="normal")).cuda()
    L = product.lib()
    L.flashllm_hip_columns_per_workgroup.restype = ctypes.c_int
    L.flashllm_hip_columns_per_workgroup.argtypes = [ctypes.c_int] * 3
    assert L.flashllm_hip_columns_per_workgroup(n, m, split_k) == 256
    c = torch.full((n * m,), float("nan"), dtype=torch.float16, device="cuda")
    plain, pages = (torch.full((split_k * n * m,), float("nan"), dtype=torch.float16, device="cuda") for _ in range(2))
    product.spmm_splitk(w.comp, w.offs, b, c, m, n, k, pages, split_k)
    c_plain = torch.full_like(c, float("nan"))
    if split_k > 1:
        product.spmm_partials(w.comp, w.offs, b, c_plain, m, n, k, plain, split_k)
        product.splitk_reduce(c_plain, plain, m, n, split_k)
        assert torch.equal(c.view(torch.int16), c_plain.view(torch.int16))
    else:
        plain = c
    fn = L.flashllm_hip_launch_spmm
    fn.restype = ctypes.c_int
    fn.argtypes = [ctypes.c_void_p] * 4 + [ctypes.c_int, ctypes.c_void_p] + [ctypes.c_int] * 6
    stream = ctypes.c_void_p(torch.cuda.current_stream().cuda_stream)
    for part in range(n // 64):
        columns = b.view(n, k)[part * 64:(part + 1) * 64]
        want = torch.full((split_k * 64 * m,), float("nan"), dtype=torch.float16, device="cuda")
        product.lib().flashllm_hip_set_rows_per_workgroup(1)
        rc = fn(stream, w.comp.data_ptr(), w.offs.data_ptr(), columns.data_ptr(), k, want.data_ptr(), m, 64, k, split_k, 0, 1)
        product.lib().flashllm_hip_set_rows_per_workgroup(0)
        assert rc == 0
        torch.cuda.synchronize()
        got = plain.view(split_k, n, m)[:, part * 64:(part + 1) * 64]
        assert bool(torch.isfinite(want).all())
        assert torch.equal(got.reshape(-1).view(torch.int16), want.view(torch.int16)), part


@pytest.mark.parametrize("tokens,ffn", [(8, 1024), (32, 1024), (64, 1024), (64, 25600), (128, 1024), (256, 4096), (512, 25600)])
@pytest.mark.parametrize("split_k", [1, 2])
def test_activation_is_stored_with_the_sums(product, tokens, ffn, split_k):
    """FFN1's ReLU in every kernel that can store its sums (several waves or one per slice, groups of four waves, three
    such groups, 256 columns) and in the reduction."""
    import torch

    print(f"activation tokens={tokens} ffn={ffn} split_k={split_k}", flush=True)
    hidden = 2048 if ffn <= 4096 else 256

    def weight(m, k, seed):
        return product.SparseWeight(synth.sparse_matrix(m, k, 0.8, seed, dist="normal", sigma=0.05, threads=8), split_k=split_k)

    layer = product.DecoderLayer(weight(3 * hidden, hidden, 1), weight(hidden, hidden, 2), weight(ffn, hidden, 3), weight(hidden, ffn, 4))
    x = torch.from_numpy(synth.dense_b(hidden, tokens, 98, dist="normal")).cuda().view(-1)
    x[:hidden] = float("nan")  # a column of NaN: 0 behind the activation
    ws = torch.empty(split_k * max(3 * hidden, ffn) * tokens, dtype=torch.float16, device="cuda")
    _, (_, _, attn_out, ffn_mid, _) = layer.forward(x, tokens, workspace=ws)
    used = 1 if tokens > 128 else split_k
    want = torch.empty_like(ffn_mid)
    w = layer.weights[2]
    product.spmm_splitk(w.comp, w.offs, attn_out, want, w.m, tokens, w.k, ws, used)
    torch.cuda.synchronize()
    assert bool(torch.isnan(want[:w.m]).all()) and bool((want[w.m:] < 0).any())
    want = torch.where(want > 0, want, torch.zeros_like(want))
    assert torch.equal(ffn_mid.view(torch.int16), want.view(torch.int16))
