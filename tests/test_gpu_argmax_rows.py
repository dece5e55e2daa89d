"""Greedy argmax of several rows of logits, in whole 16-byte pieces and not."""
import numpy as np
import pytest

from denograd_amd.ffi import check
from denograd_amd.tensor import Tensor

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n", [128256, 8, 65536 + 8, 1027])
def test_argmax_rows_ties_and_special_values(hip, n):
    """Lowest index among the maxima, wherever the thread that meets it first; not-a-number never wins; a row of -inf gives its first
    element."""
    rng = np.random.default_rng(n)
    x = rng.standard_normal((5, n)).astype(np.float16)
    x[1, [n // 2, n - 1, 5]] = 9.0
    x[2, :] = -np.inf
    x[3, [1, n - 2]] = np.nan
    x[3, [4, n // 3]] = 60000.0
    tx, out = Tensor(x), Tensor.empty((5,), "int32")
    check(hip.jsgrad_hip_argmax_rows(tx.ptr, 5, n, out.ptr))
    assert list(out.numpy()) == [int(np.nanargmax(r.astype(np.float32))) if not np.all(np.isneginf(r)) else 0 for r in x]


@pytest.mark.parametrize("n,at", [(8192, 0), (8200, 0), (8200, 1), (16384 + 8, 0), (70000, 0)])
def test_argmax_rows_where_pieces_end(hip, n, at):
    """Rows around the length from which whole pieces are read, of a number of pieces that leaves threads with none or the last one again,
    and rows that do not begin at a piece; the maximum, twice, in a thread's first, second or last piece, alone among -inf or NaN."""
    rng = np.random.default_rng(n + at)
    x = np.full((8, n), -np.inf, np.float16)
    x[:4] = rng.standard_normal((4, n))
    x[1, [n - 1, n - 8]] = 9.0
    x[2, [8 * 1023 + 7, 8 * 1024 if n > 8192 else 8 * 1023 + 6]] = 9.0
    x[3, 3:] = np.nan
    x[5, n - 1] = -3.0
    x[6, :] = np.nan
    x[6, n - 5] = -np.inf
    x[7, :8] = np.nan
    tx, out = Tensor(np.concatenate([np.full(at, 70.0, np.float16), x.reshape(-1)])), Tensor.empty((8,), "int32")
    check(hip.jsgrad_hip_argmax_rows(tx.ptr + 2 * at, 8, n, out.ptr))
    assert list(out.numpy()) == [int(np.flatnonzero(r == np.nanmax(r))[0]) for r in x]
