"""A weight without its zeros, as it crosses the link to the GPU (host side): first values, bits and values of every group."""
import ctypes

import numpy as np
import pytest

import synth

GROUP, PIECE = 2048, 65536
BITS, VALUES, STRIDE = PIECE // GROUP * 4, PIECE // GROUP * 4 + PIECE // 8, PIECE // GROUP * 4 + PIECE // 8 + PIECE * 2 + 128


def _halfs(form, n):
    a = synth.sparse_matrix(n // 64, 64, 0.8, 7).view(np.uint16).reshape(-1).copy()
    if form == "empty":
        a[:] = 0
    elif form == "dense":
        a[:] = np.arange(n) % 65535 + 1
    elif form == "special":  # what is not all zero bits stays: -0, NaN, subnormals
        a[::3] = 0x8000
        a[1::7] = 0x7e01
        a[2::5] = 1
    return a


@pytest.mark.parametrize("way", ["flashllm_pack_piece", "flashllm_pack_piece_plain"])
@pytest.mark.parametrize("form", ["sparse", "empty", "dense", "special"])
@pytest.mark.parametrize("n", [GROUP, 3 * GROUP, PIECE - GROUP, PIECE])
def test_a_piece_holds_every_half_that_is_not_all_zero_bits(product, form, n, way):
    a = _halfs(form, n)
    out = np.full(STRIDE + 64, 0xa5, dtype=np.uint8)
    fn = getattr(product.lib(), way)
    fn.restype, fn.argtypes = None, [ctypes.c_void_p, ctypes.c_size_t, ctypes.c_void_p]
    fn(a.ctypes.data, n, out.ctypes.data)
    kept = a != 0
    assert np.array_equal(out[BITS:BITS + n // 8], np.packbits(kept, bitorder="little"))
    before = np.concatenate([[0], np.cumsum(kept.reshape(-1, GROUP).sum(1))])
    assert np.array_equal(out[:4 * (n // GROUP)].view(np.uint32), before[:-1])
    assert np.array_equal(out[VALUES:VALUES + 2 * before[-1]].view(np.uint16), a[kept])
    assert (out[STRIDE:] == 0xa5).all()
