"""Which way a host matrix takes to the GPU: without its zeros where that is quicker, as it is elsewhere (no GPU: the two ways are
recorded, not taken)."""
import ctypes

import numpy as np
import pytest
import torch

import synth


class Recorded:
    """The library with both uploads replaced by a note of the call."""

    def __init__(self, lib):
        self.lib, self.ways, self.nothing_to_pin = lib, [], False

    def __getattr__(self, name):
        if name not in ("flashllm_hip_upload", "flashllm_hip_upload_packed"):
            return getattr(self.lib, name)

        def call(*_):
            self.ways.append(name.removeprefix("flashllm_hip_upload") or "as it is")
            return 0

        return call


@pytest.fixture
def way_of(product, monkeypatch):
    """way_of(shape, threads): which upload the matrix takes.  Device and pinned memory are ordinary memory here."""
    real = torch.empty
    recorded = Recorded(product.lib())

    def empty(*args, pin_memory=False, device=None, **kw):
        assert not pin_memory or device == "cpu"  # torch pins no memory of another device, and the default one may be the GPU
        if pin_memory and recorded.nothing_to_pin:
            raise RuntimeError("out of pinned memory")
        return real(*args, device="cpu", **kw)

    monkeypatch.setattr(torch, "empty", empty)
    monkeypatch.setattr(product, "lib", lambda: recorded)
    monkeypatch.setattr(product, "_stream", lambda stream: ctypes.c_void_p(0))

    def way(a, threads, nothing_to_pin=False):
        recorded.ways.clear()
        recorded.nothing_to_pin = nothing_to_pin
        recorded.flashllm_set_compress_threads(threads)
        try:
            assert product._upload(a).shape == a.shape
        finally:
            recorded.flashllm_set_compress_threads(0)
        assert len(recorded.ways) == 1
        return recorded.ways[0]

    return way


@pytest.mark.parametrize("shape", [(1280, 1536), (2048, 2048), (7168, 2048)])
def test_one_thread_packs_no_faster_than_the_copy(way_of, shape):
    a = synth.sparse_matrix(*shape, 0.8, 3)
    assert way_of(a, 1) == "as it is"
    assert way_of(a, 2) == "_packed"
    assert way_of(a, 16) == "_packed"


def test_a_small_matrix_with_few_zeros_goes_as_it_is(way_of):
    assert way_of(synth.sparse_matrix(1280, 1536, 0.0, 3), 16) == "as it is"
    assert way_of(synth.sparse_matrix(1280, 1536, 0.5, 3), 16) == "as it is"
    assert way_of(synth.sparse_matrix(1280, 1536, 0.7, 3), 16) == "_packed"
    assert way_of(synth.sparse_matrix(1024, 4032, 0.0, 3), 16) == "as it is"
    assert way_of(synth.sparse_matrix(1024, 4096, 0.0, 3), 16) == "_packed"
    assert way_of(synth.sparse_matrix(1024, 1024, 0.8, 3), 16) == "as it is"
    assert way_of(synth.sparse_matrix(1024, 1280, 0.8, 3), 16) == "_packed"


def test_without_pinned_memory_it_goes_as_it_is(way_of):
    a = synth.sparse_matrix(2048, 2048, 0.8, 3)
    assert way_of(a, 16) == "_packed"
    assert way_of(a, 16, nothing_to_pin=True) == "as it is"


def test_pinned_memory_for_the_matrix_and_no_more_than_the_ring(product):
    fn = product.lib().flashllm_hip_upload_stage
    stride = 128 + 65536 // 8 + 2 * 65536 + 128
    for n, pieces in ((2048, 1), (65536, 1), (65536 + 2048, 2), (1024 * 1024, 16), (223 * 65536, 223), (224 * 65536, 224), (225 * 65536, 224), (1 << 33, 224)):
        assert fn(n) == pieces * stride
