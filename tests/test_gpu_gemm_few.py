"""The kernel for at most 16 rows that streams fp16 or int8 weights past x in registers: every share of a weight row that it is built
for, and every way its tiles are dealt (only halves, whole tiles with idle blocks, whole rounds and halves behind them, whole
rounds and a ragged one).

Tolerance: products and sums are those of the oracle's several-row Linear in another order (assert_close)."""
import numpy as np
import pytest

import oracle as orc
from denograd_amd import ffi
from denograd_amd.ffi import check
from denograd_amd.tensor import Tensor
from tests.helpers import assert_close
from tests.test_gpu_rows import KINDS, dev, make_weight, sp, test_gemm_ffn_gate as ffn_gate, test_gemm_qkv_rope_writes_queries_and_cache as qkv_rope

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("kind,in_f", [("float16", k) for k in (1024, 1536, 2048, 3072, 4096, 6144, 8192)] + [("int8", k) for k in (2048, 3072, 4096, 6144, 8192)])
@pytest.mark.parametrize("rows,out_f", [(16, 128), (8, 128), (5, 2176), (2, 4224), (7, 4224), (16, 6400)])
def test_few_rows_against_oracle(hip, kind, in_f, rows, out_f):
    rng = np.random.default_rng(rows + in_f)
    w, s = make_weight(kind, out_f, in_f)
    x = rng.standard_normal((rows, in_f)).astype(np.float16)
    res = rng.standard_normal((rows, out_f)).astype(np.float16)
    tw, ts = dev(w, s)
    tx, tr = Tensor(x), Tensor(res)
    lin = orc.linear(w, s, x, out_f, in_f, True)
    for residual, ref in ((None, lin), (tr.ptr, (res.astype(np.float32) + lin).astype(np.float16).astype(np.float32))):
        y = Tensor.full((rows + 1, out_f), 7.0, "float16")
        check(hip.jsgrad_hip_gemm(KINDS[kind], tw.ptr, sp(ts), out_f, in_f, tx.ptr, rows, y.ptr, residual))
        got = y.numpy()
        assert np.all(got[rows] == 7.0)
        assert_close(got[:rows].astype(np.float32), ref, True, f"{kind} {rows}x{out_f}x{in_f}", ulp_at=lin if residual else None)


@pytest.mark.parametrize("kind,in_f,rows,out_f", [("float16", k, r, n) for k in (1024, 1536, 2048, 3072, 4096, 6144, 8192) for r, n in ((3, 8320), (2, 11392))] +
                         [("int8", 2048, 3, 8320), ("int8", 3072, 9, 8320), ("int8", 4096, 3, 8320), ("int8", 2048, 2, 11392), ("int8", 3072, 2, 11392)])
def test_few_rows_with_several_rounds_of_tiles(hip, kind, in_f, rows, out_f):
    """Outputs of 8192 and more give a block two tiles and more, whose steps follow each other through its ring (and x is waited for in
    front of them): two rounds and halves behind them, two rounds and a ragged third."""
    test_few_rows_against_oracle(hip, kind, in_f, rows, out_f)


@pytest.mark.parametrize("kind,dim,hidden", [("float16", 2048, 4224), ("float16", 1536, 128), ("int8", 3072, 4224), ("int8", 4096, 2176), ("int8", 4096, 640)])
def test_few_rows_ffn_gate(hip, kind, dim, hidden):
    ffn_gate(hip, kind, 9, dim, hidden)


@pytest.mark.parametrize("kind,hd,B,dim", [("float16", 64, 16, 3072), ("int8", 128, 3, 4096), ("int8", 128, 16, 4096), ("int8", 128, 16, 2048)])
def test_few_rows_qkv_rope(hip, kind, hd, B, dim):
    qkv_rope(hip, kind, hd, B, 1, dim)


@pytest.mark.parametrize("most,out_f,in_f", [(16, 1024, 8192), (12, 2048, 8192), (9, 3072, 8192), (16, 4096, 8192), (16, 2048, 6144), (13, 4096, 6144), (16, 14336, 6144)])
def test_long_fp16_rows_up_to_the_number_where_another_kernel_is_faster(hip, most, out_f, in_f):
    """A row's sums do not depend on the rows beside it, so the first rows of a call have the bits of the call of those rows alone exactly where both
    take this kernel; behind the line the sums are in another order."""
    w, x = Tensor.randn((out_f * in_f,), "float16", 1, 0.05), Tensor.randn((17 * in_f,), "float16", 2, 1.0)
    out = []
    for rows in (8, most, most + 1):
        y = Tensor.empty((rows, out_f), "float16")
        check(hip.jsgrad_hip_gemm(KINDS["float16"], w.ptr, None, out_f, in_f, x.ptr, rows, y.ptr, None))
        out.append(y.numpy().view(np.uint16)[:8])
    few, at, behind = out
    assert np.array_equal(at, few)
    assert not np.array_equal(behind, few)


@pytest.mark.parametrize("rows,out_f,in_f", [(9, 4096, 4096), (16, 4096, 4096), (16, 3200, 4096), (16, 3072, 4096), (12, 1024, 4096), (9, 128, 4096), (9, 4224, 4096)])
def test_int8_rows_of_4096_behind_up_to_16_rows(hip, rows, out_f, in_f):
    """Both sides of the line, x filling the whole ring in front of the weights: up to 4096 weight rows the bits of each row by itself, behind them another
    kernel's, and the oracle's values on all."""
    test_few_rows_against_oracle(hip, "int8", in_f, rows, out_f)
    w, s = dev(*make_weight("int8", out_f, in_f))
    x = Tensor.randn((rows * in_f,), "float16", 2, 1.0)
    out = []
    for n in (8, rows):
        y = Tensor.empty((n, out_f), "float16")
        check(hip.jsgrad_hip_gemm(KINDS["int8"], w.ptr, s.ptr, out_f, in_f, x.ptr, n, y.ptr, None))
        out.append(y.numpy().view(np.uint16)[:8])
    assert np.array_equal(*out) == (out_f <= 4096)


@pytest.mark.parametrize("kind,in_f", [("float16", 1024), ("int8", 2048)])
@pytest.mark.parametrize("rows", [9, 12, 13])
@pytest.mark.parametrize("out_f", [256, 6400])
def test_steps_of_256_bytes_ask_for_twelve_or_sixteen_rows(hip, kind, in_f, rows, out_f):
    """The fourth load of x is left out where nobody has its rows: the oracle's values, and the bits of the first rows of a call of 16."""
    test_few_rows_against_oracle(hip, kind, in_f, rows, out_f)
    w, s = dev(*make_weight(kind, out_f, in_f))
    x = Tensor.randn((16 * in_f,), "float16", 2, 1.0)
    out = []
    for n in (16, rows):
        y = Tensor.empty((n, out_f), "float16")
        check(hip.jsgrad_hip_gemm(KINDS[kind], w.ptr, sp(s), out_f, in_f, x.ptr, n, y.ptr, None))
        out.append(y.numpy().view(np.uint16)[:rows])
    assert np.array_equal(*out)


# A wavefront that stores a part of a unit's outputs leaves that store in flight behind the steps that it waits for; one to four of the eight do.  Several whole
# rounds of units, a last one of halves (8320 columns) or a ragged one (11392):

@pytest.mark.parametrize("rows,hidden", [(1, 11392), (4, 8320), (5, 11392), (13, 8320), (16, 8320)])
@pytest.mark.parametrize("dim", [1024, 2048, 3072])
def test_fp16_gates_with_several_rounds_of_tiles(hip, rows, hidden, dim):
    ffn_gate(hip, "float16", rows, dim, hidden)


@pytest.mark.parametrize("kind,dim", [("float16", 1024), ("float16", 2048), ("float16", 4096), ("int8", 2048)])
@pytest.mark.parametrize("rows,heads", [(1, 174), (4, 126), (5, 174), (13, 126), (16, 126)])
def test_qkv_rope_with_several_rounds_of_tiles(hip, kind, dim, rows, heads):
    """Against the plain product of the stacked matrices, which adds in the same order, and the oracle's rotary step."""
    hd, kv, ctx, start, rng = 64, 2, 16, 5, np.random.default_rng(rows + dim)
    n = (heads + 2 * kv) * hd
    w, s = dev(*make_weight(kind, n, dim))
    x = Tensor(rng.standard_normal((rows, dim)).astype(np.float16))
    y = Tensor.empty((rows, n), "float16")
    check(hip.jsgrad_hip_gemm(KINDS[kind], w.ptr, sp(s), n, dim, x.ptr, rows, y.ptr, None))
    raw = y.numpy().astype(np.float32)
    table = Tensor.empty((2 * ctx, hd // 2, 2), "float16")
    check(hip.jsgrad_hip_rope_table(table.ptr, hd, 2 * ctx, 500000.0, ffi.F16))
    fc = table.numpy().astype(np.float32)
    at = lambda row: (w.ptr + row * dim * (2 if kind == "float16" else 1), s.ptr + row * 2 if s is not None else None)
    q, ck, cv = Tensor.full((rows + 1, heads * hd), 7.0, "float16"), Tensor.zeros((rows, ctx, kv * hd), "float16"), Tensor.zeros((rows, ctx, kv * hd), "float16")
    check(hip.jsgrad_hip_gemm_qkv_rope(KINDS[kind], *at(0), *at(heads * hd), *at((heads + kv) * hd), x.ptr, rows, 1, start, table.ptr, q.ptr, ck.ptr, cv.ptr,
                                       dim, heads, kv, hd, ctx))
    assert np.all(q.numpy()[rows] == 7.0)
    q_raw, k_raw, v_raw = np.split(raw, [heads * hd, (heads + kv) * hd], axis=1)
    assert_close(q.numpy()[:rows].astype(np.float32), np.stack([orc.rope(r, heads, hd, fc[start], True) for r in q_raw]), True, "q", composed=True)
    assert_close(ck.numpy()[:, start].astype(np.float32), np.stack([orc.rope(r, kv, hd, fc[start], True) for r in k_raw]), True, "k", composed=True)
    assert np.array_equal(cv.numpy()[:, start].astype(np.float32), v_raw)
    rest = np.arange(ctx) != start
    assert not ck.numpy()[:, rest].any() and not cv.numpy()[:, rest].any()
