"""The kernel that shares a tile's K range among the wavefronts of a block (some dozens of rows), pinned: every tile, with and without
K parts, under every epilogue, at ragged row tiles and where turns of its ring run out: one stage in all (one group has work), fewer
turns than the ring holds, a last turn with stages for some groups only.

Tolerance: products and sums are those of the oracle's several-row Linear in another order (assert_close)."""
import ctypes as C
import os

import numpy as np
import pytest

from denograd_amd import ffi
from denograd_amd.ffi import check
from denograd_amd.tensor import Tensor
from tests import test_gpu_gemm_tile as tile_tests
from tests import test_gpu_rows as rows_tests
from tests.test_gpu_gemm_tile import test_tiled_gemm_at_the_edges as check_gemm

pytestmark = pytest.mark.gpu


@pytest.fixture(autouse=True)
def own_numbers():
    """The stream of random numbers that the other files share goes on where it was."""
    before = rows_tests.RNG.bit_generator.state
    rows_tests.RNG.bit_generator.state = np.random.default_rng(5).bit_generator.state
    yield
    rows_tests.RNG.bit_generator.state = before


TILES = ["g16x64", "g16x64/3", "g16x128", "g16x128/2", "g32x64", "g32x64/5", "g32x128", "g32x128/3", "g64x64", "g64x64/3", "g64x128", "g64x128/2"]


@pytest.mark.parametrize("kind", ["float16", "int8", "nf4"])
@pytest.mark.parametrize("tile", TILES)
def test_every_group_tile(hip, monkeypatch, kind, tile):
    monkeypatch.setenv("JSG_GEMM_TILE", tile)
    k = 2 if kind == "nf4" else 1                             # stages are 64 elements, of int8 128, of nf4 256 (128 with 64 rows)
    for rows, out_f, in_f in ((2, 128, 128 * k), (16, 256, 1152 * k), (19, 128, 640 * k), (57, 768, 640 * k), (64, 128, 2048), (57, 4224, 512), (100, 256, 1408 * k)):
        check_gemm(hip, kind, rows, out_f, in_f)
    for rows in (5, 57):
        rows_tests.test_gemm_ffn_gate(hip, kind, rows, 640 * k, 384)
    rows_tests.test_gemm_qkv_rope_writes_queries_and_cache(hip, kind, 64, 3, 19, 640 * k)
    rows_tests.test_gemm_qkv_rope_writes_queries_and_cache(hip, kind, 128, 5, 9, 640 * k)
    if kind == "float16":
        check_gemm(hip, kind, 33, 128, 64)
        check_gemm(hip, kind, 9, 128, 8256)


@pytest.mark.parametrize("kind", ["float16", "int8", "nf4"])
def test_as_chosen(hip, monkeypatch, kind):
    """Calls that come to the group kernel by their sizes (more than one round of the streaming kernel's blocks, long rows, 33 to 64 rows of
    short ones), the same calls in a capture, and with scales at an odd multiple of two bytes."""
    sizes = ((20, 4224, 1024), (31, 256, 8192), (12, 256, 9216), (40, 384, 1024), (57, 128, 2048))
    for rows, out_f, in_f in sizes:
        check_gemm(hip, kind, rows, out_f, in_f)
        check_gemm(tile_tests.Captured(hip), kind, rows, out_f, in_f)
    for rows in (9, 24, 57):
        rows_tests.test_gemm_ffn_gate(hip, kind, rows, 1024, 4224)
        rows_tests.test_gemm_ffn_gate(tile_tests.Captured(hip), kind, rows, 1024, 4224)
    rows_tests.test_gemm_qkv_rope_writes_queries_and_cache(hip, kind, 64, 3, 9, 3072)
    if kind == "float16":
        return
    held = []

    def slice_of_scales(t):
        held.append(Tensor(np.concatenate([np.full(1, 7.0, np.float16), t.numpy().reshape(-1)])))
        return held[-1].ptr + 2

    monkeypatch.setattr(tile_tests, "sp", slice_of_scales)
    for rows, out_f, in_f in sizes:
        check_gemm(hip, kind, rows, out_f, in_f)


@pytest.mark.parametrize("rows,out_f,in_f", [(1, 4224, 1024), (9, 256, 8192), (16, 8320, 512), (24, 4224, 1024), (57, 128, 2048)])
@pytest.mark.parametrize("tile", ["", "g16x64", "g16x128", "g32x64/3", "g32x128", "g64x64", "g64x128/2"])
def test_int8_scales_between_two_words_take_the_same_kernel(hip, monkeypatch, rows, out_f, in_f, tile):
    """The bits of the call with scales at a multiple of four bytes, in every tile (8, 16 or 32 words of scales to a wavefront, one more here) and as
    chosen; the last scale is the last half of its allocation."""
    rng = np.random.default_rng(rows)
    w, s = rows_tests.make_weight("int8", out_f, in_f)
    x = Tensor(rng.standard_normal((rows, in_f)).astype(np.float16))
    tw, ts = Tensor(w), Tensor(s)
    odd = Tensor(np.concatenate([np.full(1, 7.0, np.float16), s.reshape(-1)]))
    if tile:
        monkeypatch.setenv("JSG_GEMM_TILE", tile)
    out = []
    for scales in (ts.ptr, odd.ptr + 2):
        y = Tensor.full((rows, out_f), 7.0, "float16")
        check(hip.jsgrad_hip_gemm(ffi.W_I8, tw.ptr, scales, out_f, in_f, x.ptr, rows, y.ptr, None))
        out.append(y.numpy().view(np.uint16))
    assert np.array_equal(*out)


@pytest.mark.parametrize("kind,rows,out_f,in_f,skinny", [
    ("float16", 24, 4096, 3072, True), ("float16", 24, 4096, 3584, False), ("float16", 24, 3072, 2048, True), ("float16", 24, 3072, 2560, False),
    ("int8", 16, 4096, 5632, True), ("int8", 12, 4096, 6144, False), ("int8", 16, 3072, 4032, True), ("int8", 16, 3072, 4096, False), ("int8", 16, 3072, 4608, False),
    ("int8", 24, 2048, 4096, True), ("int8", 24, 1024, 4096, False), ("int8", 24, 4096, 4608, False),
    ("nf4", 16, 4096, 8192, True), ("nf4", 16, 4096, 8704, False), ("nf4", 16, 3072, 4608, False), ("nf4", 8, 3072, 8192, True),
    ("nf4", 16, 3072, 8192, True), ("nf4", 12, 3072, 7168, False), ("nf4", 5, 4096, 11264, True), ("nf4", 8, 4096, 14336, False),
    ("nf4", 17, 4096, 5120, True), ("nf4", 17, 4096, 5632, False)])
def test_lines_to_the_kernel_for_short_rows(hip, monkeypatch, kind, rows, out_f, in_f, skinny):
    """Which kernel a call comes to, by its bits: the K groups and parts of this one add the sums in another order."""
    w = Tensor.randn((out_f * in_f // 2,), "float16", 1, 0.05)    # as fp16, half of the rows twice; as codes, any bits are some
    s = None if kind == "float16" else Tensor.full((out_f * (in_f // 64),), 0.01, "float16")
    x = Tensor.randn((rows * in_f,), "float16", 2, 1.0)
    if kind == "float16":
        w = Tensor(np.concatenate([w.numpy(), w.numpy()]))
    out = []
    for pin in ("", "1"):
        if pin:
            monkeypatch.setenv("JSG_GEMM_SKINNY_TILES", pin)
        y = Tensor.empty((rows, out_f), "float16")
        check(hip.jsgrad_hip_gemm(rows_tests.KINDS[kind], w.ptr, s.ptr if s is not None else None, out_f, in_f, x.ptr, rows, y.ptr, None))
        out.append(y.numpy().view(np.uint16))
    assert np.array_equal(*out) == skinny


@pytest.mark.parametrize("rows,hidden,dim,skinny", [(2, 4096, 4096, True), (24, 2560, 3584, True), (16, 4096, 3072, False), (16, 4096, 4608, False), (16, 4224, 4096, False)])
def test_lines_to_the_kernel_for_short_rows_of_nf4_gates(hip, monkeypatch, rows, hidden, dim, skinny):
    w, s, x = Tensor.randn((hidden * dim // 2,), "float16", 1, 0.05), Tensor.full((hidden * dim // 64,), 0.01, "float16"), Tensor.randn((rows * dim,), "float16", 2, 1.0)
    out = []
    for pin in ("", "1"):
        if pin:
            monkeypatch.setenv("JSG_GEMM_SKINNY_TILES", pin)
        y = Tensor.empty((rows, hidden), "float16")
        check(hip.jsgrad_hip_gemm_ffn_gate(ffi.W_NF4, w.ptr, s.ptr, w.ptr + hidden * dim // 2, s.ptr, x.ptr, rows, y.ptr, dim, hidden))
        out.append(y.numpy().view(np.uint16))
    assert np.array_equal(*out) == skinny


def test_a_process_without_an_environment(hip):
    """clearenv() leaves no list of variables at all: the calls that look for pins in it run as they do without any."""
    x, w = Tensor.randn((4 * 512,), "float16", 1, 1.0), Tensor.randn((128 * 512,), "float16", 2, 0.05)
    out = []
    for clear in (False, True):
        y = Tensor.empty((4, 128), "float16")
        if clear:
            C.CDLL(None).clearenv()
        try:
            status = hip.jsgrad_hip_gemm(ffi.W_F16, w.ptr, None, 128, 512, x.ptr, 4, y.ptr, None)
        finally:
            for name, value in os.environ.items():
                os.putenv(name, value)
        check(status)
        out.append(y.numpy().view(np.uint16))
    assert np.array_equal(*out)
