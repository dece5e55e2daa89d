"""Gathered rows are exact, in whole pieces and element by element: widths around a block's pieces, tables and outputs between two pieces."""
import numpy as np
import pytest

import oracle as orc
from denograd_amd import ffi
from denograd_amd.ffi import check
from denograd_amd.tensor import Tensor

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dim", [8, 317, 2040, 2048, 2056])
@pytest.mark.parametrize("table_off,out_off", [(0, 0), (1, 0), (0, 1), (8, 8)])
def test_rows_of_any_width_and_address(hip, dim, table_off, out_off):
    """Offsets in elements; token ids outside the table take its first or last row."""
    rng = np.random.default_rng(dim)
    vocab, toks = 37, np.int32([0, 36, 5, 5, -3, 40, 17])
    rows = np.clip(toks, 0, vocab - 1)
    table = rng.standard_normal((vocab, dim)).astype(np.float16)
    codes, scale = orc.int8_quantize(table.astype(np.float32))
    tk, ts = Tensor(toks), Tensor(scale)
    for kind, t, want in ((ffi.W_F16, table, table[rows]), (ffi.W_I8, codes, orc.int8_dequant(codes, scale)[rows])):
        tt = Tensor(np.concatenate([np.zeros(table_off, t.dtype), t.reshape(-1)]))
        out = Tensor.full((toks.size * dim + out_off + 8,), 7.0, "float16")
        check(hip.jsgrad_hip_embed_rows(kind, tt.ptr + table_off * t.dtype.itemsize, ts.ptr, tk.ptr, toks.size, out.ptr + 2 * out_off, dim, vocab))
        got = out.numpy()
        assert np.array_equal(got[out_off:out_off + want.size].view(np.uint16), want.reshape(-1).view(np.uint16))
        assert np.all(got[:out_off] == 7.0) and np.all(got[out_off + want.size:] == 7.0)
