"""The quantisers at the edges of their chunked kernels, bit for bit against the oracle: rows of one chunk, of the most a thread
keeps in registers, of one chunk more and of odd lengths (element by element), unaligned pointers, rows of zeros, subnormals,
infinities and NaN, values at the middle between two codes."""
import numpy as np
import pytest

import oracle as orc
from denograd_amd import ffi
from denograd_amd.ffi import check
from denograd_amd.tensor import Tensor

pytestmark = pytest.mark.gpu


def awkward(rng, shape):
    w = (rng.standard_normal(shape) * 0.02).astype(np.float16)
    w[0] = 0
    w[1] *= np.float16(2.0 ** -13)                  # subnormal values, subnormal or zero scale
    if len(w) > 2:
        w[2, -1], w[2, 0] = np.inf, -1.0
    if len(w) > 3:
        w[3, 0] = np.nan
    return w


@pytest.mark.parametrize("act,name", [(ffi.F16, "float16"), (ffi.F32, "float32")])
@pytest.mark.parametrize("in_f", [8, 64, 264, 2056, 16384, 16392, 1003])
def test_int8_quantise_row_lengths(hip, act, name, in_f):
    w = awkward(np.random.default_rng(in_f), (6, in_f)).astype(name)
    t, codes, scale = Tensor(w), Tensor.empty((6, in_f), "int8"), Tensor.empty((6,), "float16")
    check(hip.jsgrad_hip_int8_quantize(t.ptr, 6, in_f, codes.ptr, scale.ptr, act))
    c, s = orc.int8_quantize(w.astype(np.float32))
    sane = [0, 1, 4, 5]                              # the codes of rows with inf or NaN are not defined in C; they must not disturb others
    assert np.array_equal(scale.numpy()[sane].view(np.uint16), np.asarray(s).reshape(-1)[sane].view(np.uint16))
    assert np.array_equal(codes.numpy()[sane], np.asarray(c).reshape(6, in_f)[sane])


@pytest.mark.parametrize("act,name", [(ffi.F16, "float16"), (ffi.F32, "float32")])
@pytest.mark.parametrize("offset", [0, 1])
def test_nf4_quantise(hip, act, name, offset):
    rng = np.random.default_rng(3)
    code = orc.nf4_dequant(np.arange(16, dtype=np.uint8) * 17, np.ones(1, np.float16))[::2].astype(np.float32)
    mids = ((code[:-1] + code[1:]) / 2).astype(np.float32)
    w = awkward(rng, (5, 64 * 37)).astype(name)
    w[4, :64] = np.resize(np.concatenate([mids, np.nextafter(mids, np.float32(2)), np.nextafter(mids, np.float32(-2)), code]), 64)
    w[4, 63] = 1.0
    w = w[[0, 1, 4]]
    flat = np.concatenate([np.zeros(offset, name), w.reshape(-1)])
    t, packed, scale = Tensor(flat), Tensor.zeros((w.size // 2 + offset,), "uint8"), Tensor.empty((w.size // 64,), "float16")
    check(hip.jsgrad_hip_nf4_quantize(t.ptr + offset * flat.itemsize, w.size, packed.ptr + offset, scale.ptr, act))
    p, s = orc.nf4_quantize(w.astype(np.float32))
    assert np.array_equal(scale.numpy().view(np.uint16), np.asarray(s).reshape(-1).view(np.uint16))
    assert np.array_equal(packed.numpy()[offset:], np.asarray(p).reshape(-1))


@pytest.mark.parametrize("act,name", [(ffi.F16, "float16"), (ffi.F32, "float32")])
@pytest.mark.parametrize("offset", [0, 1])
def test_nf4_blocks_with_inf_or_nan(hip, act, name, offset):
    """The maximum of a block passes over NaN; a block of nothing but NaN has NaN for its scale, so that it is not read back as zeros.
    NaN, and what an infinite scale makes of infinities, get code 0; finite values beside an infinity get the code of zero."""
    w = np.full((5, 64), 0.25, np.float32)
    w[0] = np.nan
    w[1, 1:] = np.nan
    w[2, 60] = np.nan
    w[3, 17] = np.inf
    w[3, 18] = np.nan
    flat = np.concatenate([np.zeros(offset, name), w.reshape(-1).astype(name)])
    t, packed, scale = Tensor(flat), Tensor.zeros((w.size // 2 + offset,), "uint8"), Tensor.empty((5,), "float16")
    check(hip.jsgrad_hip_nf4_quantize(t.ptr + offset * flat.itemsize, w.size, packed.ptr + offset, scale.ptr, act))
    np.testing.assert_array_equal(scale.numpy(), np.array([np.nan, 0.25, 0.25, np.inf, 0.25], np.float16))
    codes = np.where(np.isfinite(w), 15, 0)
    codes[3] = np.where(np.isfinite(w[3]), 7, 0)
    np.testing.assert_array_equal(packed.numpy()[offset:], (codes.reshape(-1, 2) @ np.array([16, 1])).astype(np.uint8))


@pytest.mark.parametrize("act,name", [(ffi.F16, "float16"), (ffi.F32, "float32")])
@pytest.mark.parametrize("in_f", [64, 264, 1003])
def test_int8_rows_with_inf_or_nan(hip, act, name, in_f):
    """The maximum of a row passes over NaN, whose code is 0; beside an infinity every code is 0."""
    w = np.full((4, in_f), 0.25, np.float32)
    w[0] = np.nan
    w[1, in_f // 2] = np.nan
    w[2, in_f - 1] = -np.inf
    t, codes, scale = Tensor(w.astype(name)), Tensor.empty((4, in_f), "int8"), Tensor.empty((4,), "float16")
    check(hip.jsgrad_hip_int8_quantize(t.ptr, 4, in_f, codes.ptr, scale.ptr, act))
    s = np.float16(np.float32(0.25) * np.float32(np.float16(1 / 127)))
    np.testing.assert_array_equal(scale.numpy(), np.array([0, s, np.inf, s], np.float16))
    want = np.where(np.isnan(w), 0, 127)
    want[2] = 0
    np.testing.assert_array_equal(codes.numpy(), want)
