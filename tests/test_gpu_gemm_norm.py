"""Products whose input is normed on the way: rows in the registers of the kernel for few of them, others through a pass over memory.  Every such call against the norm and the product as two calls.

Tolerance: the two add a row's squares in another order, which moves its factor by a float rounding or two and with it an element of the
normed row by one fp16 rounding where it lay that close to a tie: assert_close's bound for a norm in front (composed)."""
import types

import numpy as np
import pytest

import oracle as orc
from denograd_amd import ffi, synthetic
from denograd_amd.ffi import check
from denograd_amd.llama3 import Llama3
from denograd_amd.tensor import Tensor
from tests import test_gpu_rows as rows_tests
from tests.helpers import assert_close
from tests.test_gpu_gemm_tile import Captured
from tests.test_gpu_rows import KINDS, dev, make_weight, sp

pytestmark = pytest.mark.gpu


@pytest.fixture(autouse=True)
def own_numbers():
    """The stream of random numbers that the other files share goes on where it was."""
    before = rows_tests.RNG.bit_generator.state
    rows_tests.RNG.bit_generator.state = np.random.default_rng(5).bit_generator.state
    yield
    rows_tests.RNG.bit_generator.state = before


EPS = 1e-5


def rows_and_norm(hip, rows, dim, seed=0):
    rng = np.random.default_rng(seed + rows + dim)
    x = (rng.standard_normal((rows, dim)) * 3).astype(np.float16)
    x[rows // 2] = 0.0                                        # eps alone under the root
    x[-1] *= np.float16(40.0)
    nw = (1.0 + 0.3 * rng.standard_normal(dim)).astype(np.float16)
    tx, tn, xn = Tensor(x), Tensor(nw), Tensor.full((rows, dim), 9.0, "float16")
    check(hip.jsgrad_hip_rmsnorm_rows(tx.ptr, tn.ptr, xn.ptr, rows, dim, EPS))
    return tx, tn, xn


def check_plain(hip, kind, rows, out_f, in_f, captured=False):
    tx, tn, xn = rows_and_norm(hip, rows, in_f)
    w, s = make_weight(kind, out_f, in_f)
    tw, ts = dev(w, s)
    scratch, y = Tensor.full((rows, in_f), 9.0, "float16"), Tensor.full((rows + 1, out_f), 7.0, "float16")
    call = Captured(hip).jsgrad_hip_gemm_norm if captured else hip.jsgrad_hip_gemm_norm
    check(call(KINDS[kind], tw.ptr, sp(ts), out_f, in_f, tx.ptr, tn.ptr, EPS, scratch.ptr, rows, y.ptr))
    got = y.numpy()
    assert np.all(got[rows] == 7.0)
    normed = xn.numpy()
    assert np.all(np.isfinite(got[:rows]))
    many = np.concatenate([normed, normed]) if rows == 1 else normed   # one row of the several-row arithmetic
    assert_close(got[:rows].astype(np.float32), orc.linear(w, s, many, out_f, in_f, True)[:rows], True, f"{kind} {rows}x{out_f}x{in_f}", composed=True)


@pytest.mark.parametrize("kind", ["float16", "int8", "nf4"])
@pytest.mark.parametrize("rows,out_f,in_f", [(1, 2176, 2048), (5, 384, 1024), (16, 128, 1536), (7, 4224, 2048), (2, 8320, 3072), (16, 4224, 4096), (9, 256, 4096), (3, 128, 64),
                                             (16, 4224, 512), (5, 128, 4608), (12, 256, 9216), (17, 256, 2048), (70, 384, 1024)])
def test_normed_gemm(hip, kind, rows, out_f, in_f):
    check_plain(hip, kind, rows, out_f, in_f)
    check_plain(hip, kind, rows, out_f, in_f, captured=True)


@pytest.mark.parametrize("kind", ["float16", "int8"])
@pytest.mark.parametrize("rows,out_f,in_f", [(1, 256, 8192), (5, 384, 6144), (8, 1024, 8192), (5, 384, 8192)])
def test_rows_too_long_to_norm_in_registers_take_the_kernel_of_normed_rows(hip, kind, rows, out_f, in_f):
    """Normed in memory, the call is that of two calls, bit for bit."""
    tx, tn, xn = rows_and_norm(hip, rows, in_f)
    w, s = make_weight(kind, out_f, in_f)
    tw, ts = dev(w, s)
    scratch, got, ref = Tensor.full((rows, in_f), 9.0, "float16"), Tensor.full((rows, out_f), 7.0, "float16"), Tensor.full((rows, out_f), 7.0, "float16")
    check(hip.jsgrad_hip_gemm(KINDS[kind], tw.ptr, sp(ts), out_f, in_f, xn.ptr, rows, ref.ptr, None))
    check(hip.jsgrad_hip_gemm_norm(KINDS[kind], tw.ptr, sp(ts), out_f, in_f, tx.ptr, tn.ptr, EPS, scratch.ptr, rows, got.ptr))
    assert np.array_equal(got.numpy().view(np.uint16), ref.numpy().view(np.uint16))


def factor_of_the_few_row_kernel(x, eps, kind):
    """A lane (a quarter of the 32 or 64 elements of a fragment read) adds its squares one by one, in float with one rounding each, the four quarters of a
    wavefront's eighth of the row meet in pairs and the eighths in order."""
    rows, dim = x.shape
    piece = 8 if kind == "float16" else 16
    lanes = x.astype(np.float64).reshape(rows, 8, -1, 4, piece).transpose(0, 1, 3, 2, 4).reshape(rows, 8, 4, -1)
    s = np.zeros(lanes.shape[:3], np.float32)
    for e in range(lanes.shape[3]):
        s = (s + lanes[..., e] ** 2).astype(np.float32)
    s = (s[..., 0] + s[..., 1]) + (s[..., 2] + s[..., 3])
    tot = s[:, 0]
    for w in range(1, 8):
        tot = tot + s[:, w]
    return np.sqrt(np.float32(1) / (tot * np.float32(1 / dim) + np.float32(eps)))


@pytest.mark.parametrize("kind,dim", [("float16", k) for k in (1024, 1536, 2048, 3072, 4096)] + [("int8", k) for k in (2048, 3072, 4096)])
@pytest.mark.parametrize("rows", [16, 5])
def test_squares_are_added_one_by_one(hip, kind, dim, rows):
    """Seen through an identity matrix: ordinary rows of three sizes, subnormal ones, rows where a lane begins with 2^24 and adds squares between one and two
    (each is rounded to two; the other half of the row makes the factor visible), the largest halves, and infinities and NaN, which spread over their own row
    and no further.  The device's square root may be one unit off, and it may round x times the factor to a half at once or to float first: every
    element of a row has to be that of one of three factors."""
    rng = np.random.default_rng(dim + rows)
    nw = (1.0 + 0.3 * rng.standard_normal(dim)).astype(np.float16)
    eye, one = np.eye(dim, dtype=np.float16 if kind == "float16" else np.int8), np.ones(dim, np.float16)
    w, s, tn = Tensor(eye), Tensor(one), Tensor(nw)
    scratch, y = Tensor.full((rows, dim), 9.0, "float16"), Tensor.full((rows, dim), 7.0, "float16")
    for turn in range(4):
        x = (rng.standard_normal((rows, dim)) * np.array([1.0, 3e-3, 30.0, 2e-6, 1.0])[np.arange(rows) % 5, None]).astype(np.float16)
        eighths = x[4::5].reshape(-1, 8, dim // 8)            # a view
        eighths[:, :4] = 1.0 + 0.2 * rng.random(eighths[:, :4].shape)
        eighths[:, :4, :64 if kind == "int8" else 32:16 if kind == "int8" else 8] = 4096.0
        if turn % 2:
            x[0] = 60000.0
            x[1, dim // 3], x[2, 7], x[3, dim - 1] = np.inf, np.nan, -np.inf
        tx, eps = Tensor(x), (EPS, 1e-16)[turn // 2]
        check(hip.jsgrad_hip_gemm_norm(KINDS[kind], w.ptr, s.ptr, dim, dim, tx.ptr, tn.ptr, eps, scratch.ptr, rows, y.ptr))
        got, whole = y.numpy(), np.isfinite(x).all(axis=1)
        assert np.isnan(got[~whole]).all()                    # 0 * NaN in every product of such a row
        r = factor_of_the_few_row_kernel(x[whole], eps, kind)
        fits = np.zeros(r.shape, bool)
        for f in (np.nextafter(r, np.float32(0)), r, np.nextafter(r, np.float32(np.inf))):
            a, b = (p.astype(np.float16) * nw for p in (x[whole].astype(np.float32) * f[:, None], x[whole].astype(np.float64) * f[:, None].astype(np.float64)))
            fits |= ((got[whole] == a) | (got[whole] == b)).all(axis=1)
        assert fits.all(), (kind, dim, rows, turn, np.nonzero(whole)[0][~fits])


@pytest.mark.parametrize("out_f,hidden", [(7040, 2944), (7168, 3072), (8192, 4096), (9216, 4608)])
def test_int8_rows_of_4096_have_the_same_bits_by_either_way_of_x(hip, out_f, hidden):
    """Up to seven rows in front of wide matrices x comes to registers straight, otherwise through the ring: the rows of calls of 1, 5 and 7 are those of
    a call of 8, under every epilogue, an infinite and a NaN row among them."""
    dim, hd, rng = 4096, 128, np.random.default_rng(out_f)
    x = (rng.standard_normal((8, dim)) * 3).astype(np.float16)
    x[2, 5], x[3, dim - 1], x[4] = np.inf, np.nan, 0.0
    tx, tn = Tensor(x), Tensor((1.0 + 0.3 * rng.standard_normal(dim)).astype(np.float16))
    w, s = dev(*make_weight("int8", out_f, dim))
    kv = 128
    q_rows = out_f - 2 * kv
    table, scratch = Tensor.zeros((64, hd // 2, 2), "float16"), Tensor.empty((8, dim), "float16")
    check(hip.jsgrad_hip_rope_table(table.ptr, hd, 64, 500000.0, ffi.F16))
    at = lambda row: (w.ptr + row * dim, s.ptr + row * 2)
    calls = []
    for rows in (8, 1, 5, 7):
        y, g, q = (Tensor.full((rows + 1, n), 7.0, "float16") for n in (out_f, hidden, q_rows))
        caches = [Tensor.full((rows, 32, kv), 7.0, "float16") for _ in range(2)]
        check(hip.jsgrad_hip_gemm_norm(ffi.W_I8, *at(0), out_f, dim, tx.ptr, tn.ptr, EPS, scratch.ptr, rows, y.ptr))
        check(hip.jsgrad_hip_gemm_ffn_gate_norm(ffi.W_I8, *at(0), *at(hidden), tx.ptr, tn.ptr, EPS, scratch.ptr, rows, g.ptr, dim, hidden))
        check(hip.jsgrad_hip_gemm_qkv_rope_norm(ffi.W_I8, *at(0), *at(q_rows), *at(q_rows + kv), tx.ptr, tn.ptr, EPS, scratch.ptr, rows, 1, 3, table.ptr, q.ptr,
                                                caches[0].ptr, caches[1].ptr, dim, q_rows // hd, kv // hd, hd, 32))
        for t in (y, g, q):
            assert np.all(t.numpy()[rows] == 7.0)
        calls.append([t.numpy()[:rows].view(np.uint16) for t in (y, g, q, *caches)])
    for got in calls[1:]:
        for a, b in zip(got, calls[0]):
            nan = np.isnan(a.view(np.float16)) & np.isnan(b[:len(a)].view(np.float16))
            assert np.array_equal(np.where(nan, 0, a), np.where(nan, 0, b[:len(a)]))


@pytest.mark.parametrize("rows,out_f,hidden", [(1, 7040, 2944), (1, 7168, 3072), (7, 7168, 3072), (8, 7168, 3072), (5, 9216, 4608)])
def test_normed_int8_rows_of_4096(hip, rows, out_f, hidden):
    check_plain(hip, "int8", rows, out_f, 4096)
    test_normed_ffn_gate(hip, "int8", rows, 4096, hidden)


@pytest.mark.parametrize("kind", ["float16", "int8", "nf4"])
@pytest.mark.parametrize("tile", ["g16x64", "g32x64/3"])
def test_normed_in_front_of_the_group_kernel(hip, monkeypatch, kind, tile):
    """A kernel that does not norm: through memory."""
    monkeypatch.setenv("JSG_GEMM_TILE", tile)
    for rows, out_f, in_f in ((2, 128, 256), (16, 256, 2304), (5, 128, 1280), (13, 256, 4096)):
        check_plain(hip, kind, rows, out_f, in_f)


@pytest.mark.parametrize("kind", ["float16", "int8", "nf4"])
@pytest.mark.parametrize("rows,dim,hidden", [(5, 2048, 4224), (16, 4096, 2176), (16, 2048, 384), (4, 4608, 128), (24, 1024, 384)])
def test_normed_ffn_gate(hip, kind, rows, dim, hidden):
    tx, tn, xn = rows_and_norm(hip, rows, dim, 1)
    (w1, s1), (w3, s3) = make_weight(kind, hidden, dim), make_weight(kind, hidden, dim)
    t1, ts1 = dev(w1, s1)
    t3, ts3 = dev(w3, s3)
    scratch, got, ref = (Tensor.full((rows, n), 9.0, "float16") for n in (dim, hidden, hidden))
    check(hip.jsgrad_hip_gemm_ffn_gate(KINDS[kind], t1.ptr, sp(ts1), t3.ptr, sp(ts3), xn.ptr, rows, ref.ptr, dim, hidden))
    check(hip.jsgrad_hip_gemm_ffn_gate_norm(KINDS[kind], t1.ptr, sp(ts1), t3.ptr, sp(ts3), tx.ptr, tn.ptr, EPS, scratch.ptr, rows, got.ptr, dim, hidden))
    assert_close(got.numpy().astype(np.float32), ref.numpy().astype(np.float32), True, f"{kind} {rows}", composed=True)


@pytest.mark.parametrize("rows,dim,hidden", [(1, 2048, 11392), (4, 2048, 8320), (5, 3072, 11392), (13, 2048, 8320), (16, 3072, 8320)])
def test_normed_fp16_gates_with_several_rounds_of_tiles(hip, rows, dim, hidden):
    test_normed_ffn_gate(hip, "float16", rows, dim, hidden)


@pytest.mark.parametrize("rows,dim,hidden", [(1, 3072, 8192), (16, 3072, 14976), (3, 3072, 15104), (9, 2048, 9216)])
def test_normed_ffn_gate_of_wide_int8_matrices(hip, rows, dim, hidden):
    """From 36 M codes on the norm decides between two kernels."""
    test_normed_ffn_gate(hip, "int8", rows, dim, hidden)


@pytest.mark.parametrize("kind", ["float16", "int8", "nf4"])
@pytest.mark.parametrize("batch,seq,dim", [(5, 1, 2048), (16, 1, 4096), (2, 7, 3072), (3, 9, 1024)])
def test_normed_qkv_rope(hip, kind, batch, seq, dim):
    hd, heads, kv, context, start, rows = 64, 8, 2, 32, 3, batch * seq
    tx, tn, xn = rows_and_norm(hip, rows, dim, 2)
    weights, held = [], []
    for n in (heads * hd, kv * hd, kv * hd):
        w, ts = dev(*make_weight(kind, n, dim))
        held += [w, ts]
        weights += [w.ptr, sp(ts)]
    table = Tensor.zeros((2 * context, hd // 2, 2), "float16")
    check(hip.jsgrad_hip_rope_table(table.ptr, hd, 2 * context, 500000.0, ffi.F16))
    scratch, outs = Tensor.full((rows, dim), 9.0, "float16"), []
    for norm in (False, True):
        q = Tensor.full((rows, heads * hd), 7.0, "float16")
        caches = [Tensor.full((batch, context, kv * hd), 7.0, "float16") for _ in range(2)]
        rest = (rows, seq, start, table.ptr, q.ptr, caches[0].ptr, caches[1].ptr, dim, heads, kv, hd, context)
        if norm:
            check(hip.jsgrad_hip_gemm_qkv_rope_norm(KINDS[kind], *weights, tx.ptr, tn.ptr, EPS, scratch.ptr, *rest))
        else:
            check(hip.jsgrad_hip_gemm_qkv_rope(KINDS[kind], *weights, xn.ptr, *rest))
        outs.append([t.numpy().astype(np.float32) for t in (q, *caches)])
    for name, a, b in zip("qkv", *outs):
        assert_close(b, a, True, name, composed=True)


def test_misaligned_and_missing_norm_arguments_are_refused(hip):
    t = Tensor.zeros((4096,), "float16")
    args = lambda nw, xn: (KINDS["float16"], t.ptr, None, 128, 64, t.ptr, nw, EPS, xn, 2, t.ptr)
    for nw, xn in ((None, t.ptr), (t.ptr, None), (t.ptr, t.ptr + 8)):
        assert hip.jsgrad_hip_gemm_norm(*args(nw, xn)) != 0


@pytest.mark.parametrize("kind", ["float16", "int8", "nf4"])
@pytest.mark.parametrize("rows,dim", [(5, 2048), (20, 1024), (70, 512)])
def test_norm_weights_at_any_even_address(hip, monkeypatch, kind, rows, dim):
    """A slice of a longer tensor as the norm's weights, in all three calls: what jsgrad_hip_rmsnorm_rows takes."""
    held = []

    def sliced(hip, rows, dim, seed=0):
        tx, tn, xn = whole(hip, rows, dim, seed)
        held.append(Tensor(np.concatenate([np.full(1, 7.0, np.float16), tn.numpy()])))
        return tx, types.SimpleNamespace(ptr=held[-1].ptr + 2), xn

    whole = rows_and_norm
    monkeypatch.setitem(globals(), "rows_and_norm", sliced)
    check_plain(hip, kind, rows, 384, dim)
    check_plain(hip, kind, rows, 384, dim, captured=True)
    test_normed_ffn_gate(hip, kind, rows, dim, 256)
    test_normed_qkv_rope(hip, kind, rows, 1, dim)


def test_a_model_whose_norm_weights_are_slices(hip):
    """A prompt and several sequences at once, against the same model with norm weights of their own."""
    cfg = synthetic.config("tiny16")
    prompt = np.arange(1, 25, dtype=np.int32).reshape(2, 12)
    out = []
    for sliced in (False, True):
        model = Llama3.from_config(cfg).load_weights(synthetic.random_state_dict(cfg, seed=0), quantized=True).model
        if sliced:
            for norm in [n for layer in model.layers for n in (layer.attention_norm, layer.ffn_norm)] + [model.norm]:
                longer = Tensor(np.concatenate([np.full(1, 7.0, np.float16), norm.weight.numpy().reshape(-1)]))
                norm.weight = Tensor(buffer=longer.lazydata.view(cfg["dim"], "float16", 2), shape=(cfg["dim"],), dtype="float16", device=longer.device)
        model.forward_rows(prompt[:1], 0)
        out.append([model.logits.numpy().astype(np.float32)])
        model.forward_rows(prompt, 0)
        model.forward_rows(prompt[:, :1].copy(), 12)
        out[-1].append(model.rows_logits().numpy().astype(np.float32))
    for a, b in zip(*out):
        assert_close(b, a, True, "logits", composed=True)


@pytest.mark.parametrize("rows,dim", [(3, 8), (19, 2040), (3, 2048), (3, 2056), (19, 4096), (3, 4104), (5, 8192), (3, 8200), (3, 4098), (1025, 2056), (1025, 8192)])
def test_rmsnorm_rows_of_every_length(hip, rows, dim):
    """Both sides of every line between block sizes and chunks; the sums' order is the only difference (assert_close)."""
    tx, tn, xn = rows_and_norm(hip, rows, dim, 3)
    got, x, w = xn.numpy(), tx.numpy(), tn.numpy()
    some = sorted({0, rows // 2, rows - 1})
    ref = np.stack([orc.rmsnorm(x[r], w, EPS, True) for r in some])
    assert_close(got[some].astype(np.float32), ref, True, f"{rows}x{dim}")
