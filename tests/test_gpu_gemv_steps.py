"""One-row products of rows of at most four k-steps (64 lanes x 16 bytes of weights): items have as many steps as the row.

A row and the same row with zeros behind it, up to four whole steps, meet lane by lane in the same order, so the two results are the
same bits; against float64 the sum of K products of two fp16 values in float is off by at most K * 2^-24 * sum |x w|, and the result by
half a unit in the last place of fp16."""
import numpy as np
import pytest

from denograd_amd import ffi
from denograd_amd.ffi import check
from denograd_amd.tensor import Tensor
from tests.ref_f64 import dequant

pytestmark = pytest.mark.gpu
KINDS = {"f16": (ffi.W_F16, 512, 8), "i8": (ffi.W_I8, 1024, 16), "nf4": (ffi.W_NF4, 2048, 64)}


def weights(kind, rows, k, rng):
    if kind == "f16":
        return (rng.standard_normal((rows, k)) * 0.05).astype(np.float16), None
    scale = rng.uniform(0.001, 0.01, (rows,) if kind == "i8" else (rows, k // 64)).astype(np.float16)
    return (rng.integers(-128, 128, (rows, k), dtype=np.int8) if kind == "i8" else rng.integers(0, 256, (rows, k // 2), dtype=np.uint8)), scale


def padded(kind, w, scale, k, to):
    n = (to - k) // 2 if kind == "nf4" else to - k
    return np.pad(w, ((0, 0), (0, n))), np.pad(scale, ((0, 0), (0, to // 64 - k // 64))) if kind == "nf4" else scale


def as_f64(kind, w, scale, k):
    sd = {"w.weight": w if kind != "nf4" else w.reshape(-1)}
    if scale is not None:
        sd["w.scale"] = scale
    return dequant(sd, "w", (w.shape[0], k))


def linear(hip, kind, w, scale, x):
    tw, ts, tx, y = Tensor(w), Tensor(scale if scale is not None else np.zeros(1, np.float16)), Tensor(x), Tensor.empty((w.shape[0],), "float16")
    check(hip.jsgrad_hip_linear(KINDS[kind][0], tw.ptr, ts.ptr, w.shape[0], x.size, tx.ptr, y.ptr, None, 1e-5, None, ffi.F16))
    return y.numpy()


@pytest.mark.parametrize("kind", KINDS)
@pytest.mark.parametrize("steps", [1, 2, 3])
@pytest.mark.parametrize("rows", [1, 3, 258, 8196])
def test_rows_of_few_steps(hip, kind, steps, rows):
    _, step, unit = KINDS[kind]
    rng = np.random.default_rng(1000 * steps + rows)
    for k in ({unit, step - unit, step} if steps == 1 else {(steps - 1) * step + unit, steps * step - unit, steps * step}):
        w, scale = weights(kind, rows, k, rng)
        x = rng.standard_normal(k).astype(np.float16)
        got = linear(hip, kind, w, scale, x)
        wide = linear(hip, kind, *padded(kind, w, scale, k, 4 * step), np.pad(x, (0, 4 * step - k)))
        assert np.array_equal(got.view(np.uint16), wide.view(np.uint16)), (kind, rows, k)
        w64, x64 = as_f64(kind, w, scale, k), x.astype(np.float64)
        bound = k * 2.0 ** -24 * (np.abs(w64) @ np.abs(x64))
        want = w64 @ x64
        assert np.all(np.abs(got.astype(np.float64) - want) <= bound + 2.0 ** -11 * (np.abs(want) + bound) + 2.0 ** -25), (kind, rows, k)


@pytest.mark.parametrize("kind", KINDS)
@pytest.mark.parametrize("hidden", [1, 130])
def test_gate_of_rows_of_one_step(hip, kind, hidden):
    code, step, unit = KINDS[kind]
    rng = np.random.default_rng(hidden)
    for k in (unit, step - unit, step, step + unit):
        (w1, s1), (w3, s3) = weights(kind, hidden, k, rng), weights(kind, hidden, k, rng)
        x, g = rng.standard_normal(k).astype(np.float16), Tensor.empty((hidden,), "float16")
        t = [Tensor(v if v is not None else np.zeros(1, np.float16)) for v in (w1, s1, w3, s3, x, np.ones(k, np.float16))]
        check(hip.jsgrad_hip_ffn_gate(code, *(v.ptr for v in t), 1e-5, g.ptr, k, hidden, ffi.F16))
        xn = (x.astype(np.float64) / np.sqrt(np.mean(x.astype(np.float64) ** 2) + 1e-5)).astype(np.float16).astype(np.float64)
        a, u = as_f64(kind, w1, s1, k) @ xn, as_f64(kind, w3, s3, k) @ xn
        want = a / (1 + np.exp(-a)) * u
        # the normed input, both products, the gate and the result are rounded to fp16: five roundings of 2^-11, the input's carried by the sums
        size = (1 + np.abs(u)) * (np.abs(as_f64(kind, w1, s1, k)) @ np.abs(xn)) + (1 + np.abs(a)) * (np.abs(as_f64(kind, w3, s3, k)) @ np.abs(xn))
        assert np.all(np.abs(g.numpy().astype(np.float64) - want) <= 2.0 ** -11 * (size + 3 * np.abs(want)) + 2.0 ** -20), (kind, hidden, k)
