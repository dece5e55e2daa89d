"""The tiled several-row kernels where they can go wrong: every tile, with and without K parts, under every epilogue (pinned, since
most sizes that are quick to check choose the smallest tile); edges of the row tiles and one K tile as chosen; and what is left to
calls that may not allocate.

Tolerance: products and sums are those of the oracle's several-row Linear in another order (assert_close, an fp16 unit of the
result or of the operands of the residual sum)."""
import ctypes as C

import numpy as np
import pytest

import oracle as orc
from denograd_amd import ffi
from denograd_amd.ffi import check
from denograd_amd.tensor import Tensor
from tests.helpers import assert_close
from tests import test_gpu_rows as rows_tests
from tests.test_gpu_rows import KINDS, dev, make_weight, sp

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("kind", ["float16", "int8", "nf4"])
@pytest.mark.parametrize("rows,out_f,in_f", [(33, 128, 64), (64, 640, 128), (65, 384, 8192), (129, 256, 4096), (257, 768, 1088), (520, 128, 2048), (1100, 512, 512)])
def test_tiled_gemm_at_the_edges(hip, kind, rows, out_f, in_f):
    rng = np.random.default_rng(rows)
    w, s = make_weight(kind, out_f, in_f)
    x = rng.standard_normal((rows, in_f)).astype(np.float16)
    res = rng.standard_normal((rows, out_f)).astype(np.float16)
    tw, ts = dev(w, s)
    tx, tr = Tensor(x), Tensor(res)
    lin = orc.linear(w, s, x, out_f, in_f, True)
    ref = (res.astype(np.float32) + lin).astype(np.float16).astype(np.float32)
    runs = []
    for _ in range(3):
        y = Tensor.full((rows + 1, out_f), 7.0, "float16")
        check(hip.jsgrad_hip_gemm(KINDS[kind], tw.ptr, sp(ts), out_f, in_f, tx.ptr, rows, y.ptr, tr.ptr))
        runs.append(y.numpy())
    assert np.all(runs[0][rows] == 7.0)                                       # nothing behind the last row
    assert all(np.array_equal(runs[0].view(np.uint16), r.view(np.uint16)) for r in runs)   # parts are added in K order, whoever is last
    assert_close(runs[0][:rows].astype(np.float32), ref, True, f"{kind} {rows}x{out_f}x{in_f}", ulp_at=lin)


@pytest.mark.parametrize("kind,in_f", [("float16", 14336), ("int8", 14336), ("nf4", 14336), ("nf4", 14272)])
def test_tiled_gemm_captured_in_a_graph(hip, kind, in_f):
    """A call that is captured cannot allocate: no K parts, quantised weights dequantised as they are read, or (nf4, an odd
    number of 64-blocks per row) on their way into LDS.  Every replay equals the oracle, with eager work in between."""
    rows, out_f = 40, 512
    rng = np.random.default_rng(5)
    w, s = make_weight(kind, out_f, in_f)
    x = rng.standard_normal((rows, in_f)).astype(np.float16)
    tw, ts = dev(w, s)
    tx, y, other = Tensor(x), Tensor.empty((rows, out_f), "float16"), Tensor.empty((rows, out_f), "float16")
    ref = orc.linear(w, s, x, out_f, in_f, True)
    check(hip.jsgrad_hip_gemm(KINDS[kind], tw.ptr, sp(ts), out_f, in_f, tx.ptr, rows, other.ptr, None))
    graph = C.c_void_p()
    check(hip.jsgrad_hip_graph_begin())
    try:
        status = hip.jsgrad_hip_gemm(KINDS[kind], tw.ptr, sp(ts), out_f, in_f, tx.ptr, rows, y.ptr, None)
    finally:
        check(hip.jsgrad_hip_graph_end(C.byref(graph)))
    check(status)
    for _ in range(4):
        check(hip.jsgrad_hip_memset(y.ptr, 0, y.nbytes))
        check(hip.jsgrad_hip_graph_launch(graph))
        assert_close(y.numpy().astype(np.float32), ref, True, f"captured {kind}")
        check(hip.jsgrad_hip_gemm(KINDS[kind], tw.ptr, sp(ts), out_f, in_f, tx.ptr, rows, other.ptr, None))
        assert_close(other.numpy().astype(np.float32), ref, True, f"eager {kind}")
    check(hip.jsgrad_hip_graph_destroy(graph))


@pytest.mark.parametrize("kind", ["int8", "nf4"])
def test_scales_between_two_dwords(hip, monkeypatch, kind):
    """Scales are halves and may lie at any even address (a slice of a longer tensor), in every entry point, at the row counts
    that would otherwise read codes and scales in place; also in a capture."""
    held = {}

    def slice_of_scales(t):
        if id(t) not in held:                         # made by the first, eager, call: a capture copies nothing
            held[id(t)] = t, Tensor(np.concatenate([np.full(1, 7.0, np.float16), t.numpy().reshape(-1)]))
        return held[id(t)][1].ptr + 2

    monkeypatch.setattr(rows_tests, "sp", slice_of_scales)
    for rows in (33, 57, 130):
        rows_tests.test_gemm_matches_several_row_linear(hip, kind, rows, 384, 512)
        rows_tests.test_gemm_ffn_gate(hip, kind, rows, 256, 384)
    rows_tests.test_gemm_qkv_rope_writes_queries_and_cache(hip, kind, 64, 1, 57, 512)
    monkeypatch.setitem(globals(), "sp", slice_of_scales)
    test_tiled_gemm_captured_in_a_graph(hip, kind, 4096)


TILES = ["64x64", "64x64/3", "64x128", "64x128/3", "128x128", "128x128/2", "256x128", "256x128/5", "256x256"]
CODE_TILES = ["q64x64", "q64x64/3", "q64x128", "q64x128/2", "q128x128", "q128x128/3", "s32x128", "s128x128", "s256x128", "s256x256"]


@pytest.mark.parametrize("kind,tile", [(k, t) for k in ("float16", "int8") for t in TILES] + [(k, t) for k in ("int8", "nf4") for t in CODE_TILES])
def test_every_tile_under_every_epilogue(hip, monkeypatch, kind, tile):
    """Ragged row tiles (57 and 295 rows), K parts of unequal length (10 steps of 64, or 5 of 128, in 2, 3 or 5 parts); int8 under an
    fp16 tile is realised first.  The plain epilogue also repeats itself bit for bit."""
    monkeypatch.setenv("JSG_GEMM_TILE", tile)
    for rows in (57, 295):
        test_tiled_gemm_at_the_edges(hip, kind, rows, 768, 640)
        if "64x64" not in tile and tile != "s32x128":         # tiles of w1|w3 come in pairs
            rows_tests.test_gemm_ffn_gate(hip, kind, rows, 640, 384)
    rows_tests.test_gemm_qkv_rope_writes_queries_and_cache(hip, kind, 64, 3, 19, 640)
    rows_tests.test_gemm_qkv_rope_writes_queries_and_cache(hip, kind, 128, 5, 59, 640)


@pytest.mark.parametrize("kind,rows,dim,hidden", [("int8", 57, 3072, 1024), ("nf4", 57, 3072, 1024), ("float16", 371, 2048, 1024), ("int8", 371, 2048, 1024)])
def test_tiles_as_chosen_under_the_fused_epilogues(hip, kind, rows, dim, hidden):
    """K parts under SwiGLU (57 rows: codes 64x128 in 6 or 8 parts; 371 rows: fp16 and codes 64x128 in 2) and under the rotary epilogue
    (64x64 in 4 or 8)."""
    rows_tests.test_gemm_ffn_gate(hip, kind, rows, dim, hidden)
    rows_tests.test_gemm_qkv_rope_writes_queries_and_cache(hip, kind, 128, 1, 57, dim)


class Captured:
    """The library with its several-row products captured in a graph, which is then launched."""

    def __init__(self, hip):
        self.hip = hip

    def __getattr__(self, name):
        f = getattr(self.hip, name)
        if not name.startswith("jsgrad_hip_gemm"):
            return f

        def call(*args):
            graph = C.c_void_p()
            check(self.hip.jsgrad_hip_graph_begin())
            try:
                status = f(*args)
            finally:
                check(self.hip.jsgrad_hip_graph_end(C.byref(graph)))
            if status == 0:
                check(self.hip.jsgrad_hip_graph_launch(graph))
                check(self.hip.jsgrad_hip_sync())
            check(self.hip.jsgrad_hip_graph_destroy(graph))
            return status
        return call


@pytest.mark.parametrize("kind", ["int8", "nf4"])
def test_long_rows_without_memory(hip, monkeypatch, kind):
    """Captured, with codes that are not read in place (int8: scales between two dwords; nf4: an odd number of 64-blocks), rows longer
    than any piece of scratch memory would hold: served all the same, under every epilogue."""
    held = []

    def slice_of_scales(t):
        held.append(Tensor(np.concatenate([np.full(1, 7.0, np.float16), t.numpy().reshape(-1)])))
        return held[-1].ptr + 2

    if kind == "int8":
        monkeypatch.setattr(rows_tests, "sp", slice_of_scales)
    rows_tests.test_gemm_matches_several_row_linear(Captured(hip), kind, 3, 128, 65600)
    rows_tests.test_gemm_ffn_gate(Captured(hip), kind, 35, 32832, 128)
    rows_tests.test_gemm_qkv_rope_writes_queries_and_cache(Captured(hip), kind, 64, 1, 3, 65600)


@pytest.mark.parametrize("kind", ["float16", "int8"])
@pytest.mark.parametrize("tile", ["192x128", "192x128/3"])
def test_tiles_of_192_rows(hip, monkeypatch, kind, tile):
    """Three row tiles to a wavefront: whole and ragged tiles of 192 rows under every epilogue."""
    before = rows_tests.RNG.bit_generator.state               # the stream that the files share goes on where it was
    monkeypatch.setenv("JSG_GEMM_TILE", tile)
    for rows in (57, 192, 193, 371):
        test_tiled_gemm_at_the_edges(hip, kind, rows, 768, 640)
        rows_tests.test_gemm_ffn_gate(hip, kind, rows, 640, 384)
    rows_tests.test_gemm_qkv_rope_writes_queries_and_cache(hip, kind, 64, 4, 50, 640)
    rows_tests.test_gemm_qkv_rope_writes_queries_and_cache(hip, kind, 128, 5, 59, 640)
    rows_tests.RNG.bit_generator.state = before


@pytest.mark.parametrize("rows,captured", [(2, False), (16, True), (32, False), (33, False)])
def test_many_short_int8_rows(hip, rows, captured):
    """Up to 32 rows behind more than 192 weight rows of 512 codes per compute unit take the staged kernel's 32 x 128 tile; the last tile is a ragged one
    of x, and 33 rows stay where they were."""
    before = rows_tests.RNG.bit_generator.state               # the stream that the files share goes on where it was
    test_tiled_gemm_at_the_edges(Captured(hip) if captured else hip, "int8", rows, 49408, 512)
    rows_tests.RNG.bit_generator.state = before


@pytest.mark.parametrize("kind", ["float16", "int8"])
@pytest.mark.parametrize("tile", ["256x256/2", "256x256/3"])
def test_largest_tiles_in_parts(hip, monkeypatch, kind, tile):
    """K parts of the largest tile: where all tiles of a launch come in parts, under every epilogue, and where only two behind a whole round do."""
    before = rows_tests.RNG.bit_generator.state               # the stream that the files share goes on where it was
    monkeypatch.setenv("JSG_GEMM_TILE", tile)
    for rows in (57, 295):
        test_tiled_gemm_at_the_edges(hip, kind, rows, 768, 640)
        rows_tests.test_gemm_ffn_gate(hip, kind, rows, 640, 384)
    rows_tests.test_gemm_qkv_rope_writes_queries_and_cache(hip, kind, 64, 3, 19, 640)
    rows_tests.test_gemm_qkv_rope_writes_queries_and_cache(hip, kind, 128, 5, 59, 640)
    test_tiled_gemm_at_the_edges(hip, kind, 295, 129 * 256, 320)
    rows_tests.RNG.bit_generator.state = before


@pytest.mark.parametrize("rows,out_f,in_f,tile,other", [
    (4096, 6144, 4096, "256x128", "256x256/2"), (3000, 6144, 4096, "192x128", "256x256/5"), (4200, 5120, 3072, "256x128", "256x256/3"),
    (3300, 6144, 4096, "256x256/4", "256x128"), (1200, 4096, 14336, "256x256/3", "256x128")])
def test_lines_to_largest_tiles_in_parts(hip, monkeypatch, rows, out_f, in_f, tile, other):
    """Which tile a call comes to, by its bits: parts add the sums in another order."""
    x, w = Tensor.randn((rows * in_f,), "float16", 1, 1.0), Tensor.randn((out_f * in_f,), "float16", 2, 0.02)
    out = []
    for pin in ("", tile, other):
        if pin:
            monkeypatch.setenv("JSG_GEMM_TILE", pin)
        y = Tensor.empty((rows, out_f), "float16")
        check(hip.jsgrad_hip_gemm(ffi.W_F16, w.ptr, None, out_f, in_f, x.ptr, rows, y.ptr, None))
        out.append(y.numpy().view(np.uint16))
    assert np.array_equal(out[0], out[1]) and not np.array_equal(out[0], out[2])
