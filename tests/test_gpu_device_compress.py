"""GPU parity of the device-side Tiled-CSL compressor (flashllm_device_tile_offsets +
flashllm_device_compress, through the C ABI): Compressed_A and TileOffsets are compared bit for bit
with the CPU oracle's restatement of InitSparseMatrixA_API, and at the full headline size with the
product's host compressor (itself bit-exact against the oracle at the sizes the oracle finishes)."""
import sys

import numpy as np
import pytest

import synth

pytestmark = pytest.mark.gpu


def say(*a):
    print(*a, flush=True)
    sys.stdout.flush()


@pytest.fixture(scope="module")
def torch_gpu():
    import torch

    assert torch.cuda.is_available(), "these tests need the GPU"
    return torch


def device_compress(product, torch, a):
    a_dev = torch.from_numpy(np.ascontiguousarray(a).view(np.float16)).cuda()
    comp, offs = product.device_compress(a_dev)
    torch.cuda.synchronize()
    return comp.cpu().numpy().view(np.uint32), offs.cpu().numpy()


def check_against_oracle(product, oracle, torch, a, what):
    say("device compress:", what, a.shape)
    items, offsets = device_compress(product, torch, a)
    _, want_items, want_offsets = oracle.compress_reorder(a)
    assert np.array_equal(offsets, want_offsets), f"{what}: TileOffsets differ"
    assert items.shape == want_items.shape, f"{what}: {items.shape} vs {want_items.shape}"
    bad = np.flatnonzero(items != want_items)
    assert bad.size == 0, f"{what}: {bad.size} items differ, first at {bad[:4]}"
    assert product.device_compress_status() == 0, f"{what}: the encoder recorded an error"


def test_config1(product, oracle, torch_gpu):
    check_against_oracle(product, oracle, torch_gpu, synth.sparse_matrix(1024, 1024, 0.8, 0), "config1")


def test_config2(product, oracle, torch_gpu):
    check_against_oracle(product, oracle, torch_gpu, synth.sparse_matrix(9216, 9216, 0.8, 0), "config2")


@pytest.mark.parametrize("sparsity", [0.0, 0.3, 0.5, 0.9, 0.99, 0.999, 1.0])
def test_any_density(product, oracle, torch_gpu, sparsity):
    a = synth.sparse_matrix(384, 320, sparsity, 11)
    check_against_oracle(product, oracle, torch_gpu, a, f"sparsity {sparsity}")


def test_every_padding_count_and_short_tiles(product, oracle, torch_gpu):
    # one tile per case: 0..40 nonzeros (fewer vectors than banks: tail part only), around 128 and 256
    # items (main part only, main + tail), all four values of nnz % 4
    rng = np.random.default_rng(5)
    counts = list(range(0, 41)) + [124, 125, 126, 127, 128, 129, 130, 131, 253, 254, 255, 256, 257, 508, 512, 516, 8189, 8190, 8191, 8192]
    a = np.zeros((128 * len(counts), 64), dtype=np.float16)
    for i, c in enumerate(counts):
        flat = np.zeros(128 * 64, dtype=np.float16)
        where = rng.choice(128 * 64, size=c, replace=False)
        flat[where] = rng.uniform(0.5, 1.0, size=c).astype(np.float16)
        a[i * 128:(i + 1) * 128] = flat.reshape(128, 64)
    check_against_oracle(product, oracle, torch_gpu, a, "padding counts / short tiles")


def test_uneven_banks(product, oracle, torch_gpu):
    # nonzeros concentrated in a few columns (= a few LDS banks): the drain levels very uneven banks,
    # and padding lands in banks that hold nothing
    rng = np.random.default_rng(6)
    a = np.zeros((512, 256), dtype=np.float16)
    for t in range(16):
        r0, c0 = (t // 4) * 128, (t % 4) * 64
        cols = rng.choice(64, size=1 + t % 5, replace=False)
        for c in cols:
            rows = rng.choice(128, size=int(rng.integers(1, 129)), replace=False)
            a[r0 + rows, c0 + c] = rng.uniform(-1, 1, size=rows.size).astype(np.float16)
    check_against_oracle(product, oracle, torch_gpu, a, "uneven banks")


@pytest.mark.parametrize("top", [127, 128, 129, 255, 256])
def test_tallest_bank(product, oracle, torch_gpu, top):
    # one bank holds `top` nonzeros beside sparse ones: 128 is the last tile the encoder sorts in LDS
    rng = np.random.default_rng(top)
    tiles = []
    for extra in range(4):  # every padding count
        rows = np.zeros((128, 32, 2), dtype=np.float16)  # [row][bank]: the two swizzled columns of a bank
        flat = rows.reshape(128, 64)
        flat[rng.random((128, 64)) < 0.2] = 0.5
        bank = np.zeros(256, dtype=np.float16)
        bank[rng.choice(256, size=top, replace=False)] = rng.uniform(0.5, 1.0, size=top).astype(np.float16)
        rows[:, 7 * extra + 3, :] = bank.reshape(128, 2)
        other = np.flatnonzero(rows[:, 0, 0] == 0)[:extra]
        rows[other, 0, 0] = 0.25
        column = np.arange(64)[None, :] ^ ((np.arange(128)[:, None] % 8) << 3)
        tile = np.zeros((128, 64), dtype=np.float16)
        np.put_along_axis(tile, column, flat, axis=1)
        tiles.append(tile)
    check_against_oracle(product, oracle, torch_gpu, np.concatenate(tiles, axis=1), f"tallest bank {top}")


@pytest.mark.parametrize("row_tiles,k_tiles", [(256, 16), (241, 17), (1025, 4)])
def test_counts_alone_and_by_rows(product, oracle, torch_gpu, row_tiles, k_tiles):
    # 4096 tiles, the most that are counted a tile to a wave; 4097 in rows of 17, whose last piece is one tile, and 4100 in rows of 4
    a = synth.sparse_matrix(128 * row_tiles, 64 * k_tiles, 0.9, row_tiles, threads=8)
    check_against_oracle(product, oracle, torch_gpu, a, f"{row_tiles} x {k_tiles} tiles")


@pytest.mark.parametrize("count", [3900, 4088, 4092, 4096, 4097, 4100, 4216, 4220, 4224, 4228, 6000, 8060, 8064, 8068, 8157, 8188])
def test_tiles_beyond_the_list(product, oracle, torch_gpu, count):
    # more than 128 levels: the pops leave in one part or two, around the counts where the second begins (4096 items and
    # the end of the first) and where it fills the list; one bank is full, the rest of the tile is random
    rng = np.random.default_rng(count)
    rows = np.zeros((128, 32, 2), dtype=np.float16)
    flat = rows.reshape(-1)
    bank = np.arange(128 * 64) // 2 % 32
    full = np.flatnonzero(bank == count % 32)
    rest = rng.choice(np.flatnonzero(bank != count % 32), size=count - full.size, replace=False)
    flat[np.concatenate([full, rest])] = rng.uniform(0.5, 1.0, size=count).astype(np.float16)
    column = np.arange(64)[None, :] ^ ((np.arange(128)[:, None] % 8) << 3)
    tile = np.zeros((128, 64), dtype=np.float16)
    np.put_along_axis(tile, column, rows.reshape(128, 64), axis=1)
    check_against_oracle(product, oracle, torch_gpu, np.concatenate([tile, tile[::-1].copy()], axis=1), f"{count} items")


def test_special_values(product, oracle, torch_gpu):
    # -0 and NaN are dropped, subnormals and infinities are kept (the reference's float compare)
    rng = np.random.default_rng(7)
    bits = rng.integers(0, 1 << 16, size=(256, 128), dtype=np.uint16)
    keep = rng.random((256, 128)) < 0.3
    bits = np.where(keep, bits, np.uint16(0))
    bits[0, :8] = [0x8000, 0x7E00, 0xFE00, 0x7C00, 0xFC00, 0x0001, 0x8001, 0x7C01]
    check_against_oracle(product, oracle, torch_gpu, bits.view(np.float16), "special values")


def test_headline_size_matches_host_compressor(product, torch_gpu):
    say("device compress: 36864x9216 against the host compressor")
    a = synth.sparse_matrix(36864, 9216, 0.8, 0, dist="normal", sigma=0.02, threads=16)
    items, offsets = device_compress(product, torch_gpu, a)
    want_items, want_offsets = product.init_sparse_matrix_a(a)
    assert np.array_equal(offsets, want_offsets)
    assert np.array_equal(items, want_items)


def test_spmm_on_device_compressed_weights(product, oracle, torch_gpu):
    # the device-compressed stream feeds the SpMM kernel directly
    from gpu_util import assert_close

    torch = torch_gpu
    m, k, n = 1024, 2048, 16
    a = synth.sparse_matrix(m, k, 0.8, 21)
    b = synth.dense_b(k, n, 22)
    comp, offs = product.device_compress(torch.from_numpy(a).cuda())
    b_dev = torch.from_numpy(b).cuda()
    c = torch.empty(n * m, dtype=torch.float16, device="cuda")
    ws = torch.empty(4 * n * m, dtype=torch.float16, device="cuda")
    product.spmm_splitk(comp, offs, b_dev, c, m, n, k, ws, 4)
    torch.cuda.synchronize()
    _, ref = oracle.spmm_model(a, b, n, 4)
    assert_close(c.cpu().numpy().reshape(n, m), ref, "spmm on device-compressed weights")


def test_status_reports_offsets_of_another_matrix(product, torch_gpu):
    """The encoder trusts TileOffsets for where a tile goes.  Given those of a different matrix it stays inside
    each tile's range, finishes normally, and says so through flashllm_device_compress_status; the word is
    cleared by reading it."""
    torch = torch_gpu
    say("device compress: status word")
    a = torch.from_numpy(synth.sparse_matrix(256, 128, 0.8, 31)).cuda()
    other = torch.from_numpy(synth.sparse_matrix(256, 128, 0.7, 32)).cuda()
    comp, offs = product.device_compress(a)
    assert product.device_compress_status() == 0
    _, offs_other = product.device_compress(other)
    assert product.device_compress_status() == 0
    out = torch.zeros(int(offs_other[-1].item()) * 4, dtype=torch.int32, device="cuda")
    rc = product.lib().flashllm_device_compress(None, a.data_ptr(), 256, 128, offs_other.data_ptr(), out.data_ptr())
    assert rc == 0
    assert product.device_compress_status() == product.ENCODE_OFFSETS
    assert product.device_compress_status() == 0
    # and the right offsets still give the right bytes afterwards
    again, _ = product.device_compress(a)
    assert torch.equal(again, comp) and product.device_compress_status() == 0


def test_rejects_bad_arguments(product, torch_gpu):
    torch = torch_gpu
    with pytest.raises(product.CompressError):
        product.device_compress(torch.zeros(100, 64, dtype=torch.float16, device="cuda"))
    with pytest.raises(product.CompressError):
        product.device_compress(torch.zeros(128, 96, dtype=torch.float16, device="cuda"))
    with pytest.raises(TypeError):
        product.device_compress(torch.zeros(128, 64, dtype=torch.float32, device="cuda"))


def test_sizes_are_copied_when_no_host_word_is_free(product, torch_gpu):
    """All words held: the size comes by a copy; some given back in between, and the same sizes through words."""
    torch = torch_gpu
    say("sizes without host words")
    hold = product.lib().flashllm_hip_hold_host_words
    mats = [synth.sparse_matrix(128 * (1 + i), 64 * (2 + i), 0.6 + 0.1 * i, 70 + i) for i in range(4)]
    devs = [torch.from_numpy(a).cuda() for a in mats]
    through_words = [product.device_compress(d) for d in devs]
    assert hold(1) == 64
    try:
        copied = [product.device_compress(d) for d in devs]
        assert hold(1) == 0  # none was free meanwhile
    finally:
        assert hold(0) == 64
    for a, word, copy in zip(mats, through_words, copied):
        items, offsets = product.init_sparse_matrix_a(a)
        for comp, offs in (word, copy):
            assert np.array_equal(comp.cpu().numpy().view(np.uint32), items) and np.array_equal(offs.cpu().numpy(), offsets)
    assert hold(1) == 64 and hold(0) == 64  # every call gave its word back


@pytest.mark.parametrize("words", [True, False])
def test_many_threads_compress_at_once(product, words):
    """Callers at the same time: each gets its own matrix's size and bytes, through a word of its own or a copy."""
    import concurrent.futures
    import threading

    import torch

    print("threads compressing at once", words, flush=True)
    count = 72
    mats = [synth.sparse_matrix(128 * (1 + i % 3), 64 * (1 + i % 5), 0.6 + 0.005 * i, i) for i in range(count)]
    devs = [torch.from_numpy(a).cuda() for a in mats]
    torch.cuda.synchronize()
    start = threading.Barrier(count, timeout=60)

    def work(i):
        stream = torch.cuda.Stream()
        with torch.cuda.stream(stream):
            start.wait()
            for _ in range(3):
                comp, offs = product.device_compress(devs[i])
            return comp.cpu().numpy().view(np.uint32), offs.cpu().numpy()

    hold = product.lib().flashllm_hip_hold_host_words
    if not words:
        assert hold(1) == 64
    try:
        with concurrent.futures.ThreadPoolExecutor(count) as pool:
            got = [f.result() for f in [pool.submit(work, i) for i in range(count)]]
    finally:
        hold(0)
    for i, a in enumerate(mats):
        items, offsets = product.init_sparse_matrix_a(a)
        assert np.array_equal(got[i][0], items) and np.array_equal(got[i][1], offsets), i


@pytest.mark.parametrize("case", ["pads", "dense", "empty", "late zeros", "special"])
def test_scan_order_matches_the_host(product, torch_gpu, case):
    """Every number of padding items (taken from the first zeros, in their place and as they are), none of them, and
    tiles whose first zeros lie at the end; the bytes are those of InitSparseMatrixA_API_NoReorder."""
    torch = torch_gpu
    say("device compress without reordering:", case)
    rng = np.random.default_rng(7)
    a = synth.sparse_matrix(384, 256, {"dense": 0.0, "empty": 1.0}.get(case, 0.8), 41)
    if case == "pads":
        for tile in range(12):  # tile by tile one more nonzero
            r, c = tile // 4 * 128, tile % 4 * 64
            a[r:r + 128, c:c + 64] = 0
            a[r:r + 128, c:c + 64].flat[rng.choice(8192, tile, replace=False)] = 1
    elif case == "late zeros":
        a[:] = 1
        for tile in range(12):
            a[tile // 4 * 128 + 127, tile % 4 * 64 + 63 - tile:tile % 4 * 64 + 64] = 0
    elif case == "special":
        bits = a.view(np.uint16)
        for value in (0x8000, 0x7e00, 0xfc01, 0x7c00, 0xfc00, 0x0001, 0x8001):  # -0, NaNs, infinities, subnormals
            bits.flat[rng.choice(bits.size, 2000, replace=False)] = value
    want, want_offs = product.init_sparse_matrix_a_noreorder(a)
    comp, offs = product.device_compress_noreorder(torch.from_numpy(a).cuda())
    assert np.array_equal(offs.cpu().numpy(), want_offs)
    assert np.array_equal(comp.cpu().numpy().view(np.uint32), want)
    assert product.device_compress_status() == 0


@pytest.mark.parametrize("reorder", [True, False])
@pytest.mark.parametrize("form", ["float16", "bits", "read-only", "strided", "empty"])
def test_loaded_weight_has_the_host_compressors_bytes(product, torch_gpu, form, reorder):
    torch = torch_gpu
    say("loaded weight:", form, reorder)
    a = synth.sparse_matrix(384, 576, 1.0 if form == "empty" else 0.8, 51)
    given = a
    if form == "bits":
        given = a.view(np.uint16)
    elif form == "read-only":
        given = np.frombuffer(a.tobytes(), dtype=np.float16).reshape(a.shape)
    elif form == "strided":
        given = np.asfortranarray(a)
    w = product.SparseWeight(given, reorder=reorder)
    items, offsets = (product.init_sparse_matrix_a if reorder else product.init_sparse_matrix_a_noreorder)(a)
    assert (w.m, w.k, w.nnz, w.num_offsets) == (384, 576, items.size, offsets.size)
    assert w.comp.dtype == torch.int32 and w.offs.dtype == torch.int32
    assert np.array_equal(w.comp.cpu().numpy().view(np.uint32), items if items.size else np.zeros(1, dtype=np.uint32))
    assert np.array_equal(w.offs.cpu().numpy(), offsets)


@pytest.mark.parametrize("threads", [1, 16])
@pytest.mark.parametrize("shape", [(128, 64), (1024, 1024), (1152, 1088), (4096, 4096), (7168, 2048), (8320, 4032)])
def test_a_matrix_arrives_whole_without_its_zeros_on_the_way(product, torch_gpu, shape, threads):
    """Pieces of 65536 halfs, parts of 32 of them, seven parts in the ring: less than a piece, a part, a piece and a bit more than whole
    parts, the ring gone round, every place taken again and two of them a third time by a part that is not full.  Every bit pattern that is
    not zero comes back, -0 and NaN too.  Other contents each time, and neither memory holds those of the time before: what is not written,
    or not there yet when it is read, shows."""
    torch, L = torch_gpu, product.lib()
    say("packed upload:", shape, threads)
    halfs = shape[0] * shape[1]
    dst = torch.empty(halfs, dtype=torch.int16, device="cuda")
    stage = torch.empty(L.flashllm_hip_upload_stage(halfs), dtype=torch.uint8, device="cpu", pin_memory=True)
    L.flashllm_set_compress_threads(threads)
    try:
        for turn in range(3):
            rng = np.random.default_rng([*shape, threads, turn])
            a = rng.integers(0, 65536, halfs, dtype=np.uint16)
            part = 32 * 65536
            for i, at in enumerate(range(0, halfs, part)):  # sparse, nearly empty, dense, half full, ... parts
                keep = (0.2, 0.01, 1.0, 0.5, 0.1)[(i + turn) % 5]
                some = a[at:at + part]
                some[rng.random(some.size, dtype=np.float32) >= keep] = 0
            a = a.reshape(shape)
            a[3::7] = 0
            a[1::9, ::2] = 0x8000
            dst.fill_(-1)
            stage.zero_()  # pieces without values, so that one fetched too early is an empty one and no index out of range
            torch.cuda.synchronize()
            assert L.flashllm_hip_upload_packed(product._stream(None), dst.data_ptr(), a.ctypes.data, a.size, stage.data_ptr()) == 0
            assert np.array_equal(dst.cpu().numpy().view(np.uint16).reshape(shape), a), (turn,)
    finally:
        L.flashllm_set_compress_threads(0)


def test_the_default_device_has_no_say_in_how_a_matrix_arrives(product, torch_gpu, monkeypatch):
    """torch refuses to pin memory on the GPU, where torch.empty allocates by default here: the way without zeros is taken all the same."""
    say("packed upload with the GPU as default device")
    L, calls = product.lib(), []

    class Watched:
        def __getattr__(self, name):
            calls.append(name)
            return getattr(L, name)

    a = synth.sparse_matrix(2048, 2048, 0.8, 53)
    monkeypatch.setattr(product, "lib", Watched)
    with torch_gpu.device("cuda"):
        got = product._upload(a)
    assert "flashllm_hip_upload_packed" in calls and "flashllm_hip_upload" not in calls
    assert np.array_equal(got.cpu().numpy().view(np.uint16), a.view(np.uint16))


def test_pinned_memory_of_loading_is_bounded_and_given_back(product, torch_gpu):
    """Twelve threads load at once, four of them pack at a time; the blocks stay in torch's cache until it is emptied."""
    import concurrent.futures

    torch = torch_gpu
    say("pinned memory of concurrent loads")
    mats = [synth.sparse_matrix(4096, 7168, 0.8, 80 + i) for i in range(12)]  # 14 parts each: the whole ring, 32 MB

    def pinned():
        return torch.cuda.host_memory_stats()["allocated_bytes.current"]

    torch._C._host_emptyCache()
    before = pinned()

    def load(i):
        with torch.cuda.stream(torch.cuda.Stream()):
            got = [product.SparseWeight(mats[i]) for _ in range(2)]
            return [(w.comp.cpu().numpy().view(np.uint32), w.offs.cpu().numpy()) for w in got]

    with concurrent.futures.ThreadPoolExecutor(12) as pool:
        got = list(pool.map(load, range(12)))
    for a, weights in zip(mats, got):
        items, offsets = product.init_sparse_matrix_a(a)
        for comp, offs in weights:
            assert np.array_equal(comp, items) and np.array_equal(offs, offsets)
    say("pinned by loading:", pinned() - before)
    assert 0 < pinned() - before <= 4 << 25
    torch._C._host_emptyCache()
    assert pinned() == before


def test_a_load_behind_other_work_leaves_the_cores_alone(product, torch_gpu):
    """The ring fills and the GPU is busy for a while: the packing threads sleep, only the caller's wait may take a core."""
    import time

    torch = torch_gpu
    say("packed upload behind other work")
    a = synth.sparse_matrix(4096, 7168, 0.8, 54)  # 14 parts, twice the ring
    x = torch.randn(8192, 8192, dtype=torch.float16, device="cuda")
    product.lib().flashllm_set_compress_threads(8)
    try:
        product._upload(a)
        y = x @ x
        torch.cuda.synchronize()
        for _ in range(150):
            y = x @ x
        cpu, wall = time.process_time(), time.perf_counter()
        got = product._upload(a)
        cpu, wall = time.process_time() - cpu, time.perf_counter() - wall
    finally:
        product.lib().flashllm_set_compress_threads(0)
    say(f"{wall * 1e3:.0f} ms, of the cores {cpu * 1e3:.0f}")
    assert wall > 0.05  # the work was in front of it
    assert cpu < 3 * wall
    assert np.array_equal(got.cpu().numpy().view(np.uint16), a.view(np.uint16))
    del y


@pytest.mark.parametrize("full_rows", [0, 15, 16, 17, 32, 48, 60, 64, 112, 127])
def test_padding_goes_to_the_first_zero_of_any_segment(product, oracle, torch_gpu, full_rows):
    """The first rows of the tile dense, so that a bank's first zero is in a later segment of 16 rows (64 rows fill 128 levels, the
    list's last); -0 and NaN behind them, which are zeros to the compressor; nnz % 4 of every kind."""
    a = np.zeros((4 * 128, 64), dtype=np.float16)
    for r in range(4):
        tile = a[128 * r:128 * r + 128]
        tile[:full_rows] = 0.5
        tile[full_rows:, ::3] = np.float16(-0.0)
        tile[full_rows:, 1::3] = np.float16("nan")
        tile[127, 2:2 + 3 * r:3] = np.float16(2.0 ** -24)
    check_against_oracle(product, oracle, torch_gpu, a, f"{full_rows} dense rows")


@pytest.mark.parametrize("k", [(1 << 26) - 64, 1 << 26])
def test_rows_of_the_most_columns_with_offsets_of_32_bits(product, torch_gpu, k):
    """17 GB with three tiles that are not empty, in the first, the middle and the last columns, whose items follow one another: a row of
    the other half of a wave lies 32 * k bytes on, up to 2^31 - 2048 by a 32-bit offset and from 2^31 on by a 64-bit address."""
    say("far columns:", k)
    torch = torch_gpu
    three = torch.from_numpy(synth.sparse_matrix(128, 192, 0.8, 61)).cuda()
    want, tiles = product.device_compress(three)
    at = [0, k // 128 * 64, k - 64]
    a = torch.zeros(128, k, dtype=torch.float16, device="cuda")
    for i, c in enumerate(at):
        a[:, c:c + 64] = three[:, 64 * i:64 * i + 64]
    comp, offs = product.device_compress(a)
    assert torch.equal(comp, want)
    assert product.device_compress_status() == 0
    for i, c in enumerate(at):
        assert offs[c // 64:c // 64 + 2].tolist() == tiles[i:i + 2].tolist()
    del a, comp, offs
    torch.cuda.empty_cache()


def test_loading_refuses_what_the_host_compressor_refuses(product, torch_gpu):
    for bad in (np.zeros((100, 64), np.float16), np.zeros((128, 96), np.float16), np.zeros((0, 64), np.float16)):
        with pytest.raises(product.CompressError):
            product.SparseWeight(bad)
    with pytest.raises(TypeError):
        product.SparseWeight(np.zeros((128, 64), np.float32))
    with pytest.raises(ValueError):
        product.SparseWeight(np.zeros((2, 128, 64), np.float16))


@pytest.mark.parametrize("where", ["tensor", "upload", "compress"])
def test_a_gpu_without_room_for_the_dense_matrix_takes_the_host_compressors_weight(product, torch_gpu, monkeypatch, where):
    """Whether torch or the runtime finds none; any other error is the caller's."""
    torch = torch_gpu
    say("loaded weight: no room", where)
    a = synth.sparse_matrix(256, 128, 0.8, 62)
    error = {"tensor": torch.cuda.OutOfMemoryError("full"), "upload": product.HipError(product.HIP_ERROR_OUT_OF_MEMORY),
             "compress": product.HipError(product.HIP_ERROR_OUT_OF_MEMORY)}[where]

    def full(*args):
        raise error

    monkeypatch.setattr(product, "device_compress" if where == "compress" else "_upload", full)
    w = product.SparseWeight(a)
    items, offsets = product.init_sparse_matrix_a(a)
    assert np.array_equal(w.comp.cpu().numpy().view(np.uint32), items) and np.array_equal(w.offs.cpu().numpy(), offsets)
    error = product.HipError(1)
    with pytest.raises(product.HipError):
        product.SparseWeight(a)
