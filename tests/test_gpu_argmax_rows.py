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
