"""The arg-max of a vocabulary that one block has in its registers, at the edges of its rounds (512 elements) and of its range (4096)."""
import numpy as np
import pytest

from denograd_amd import ffi
from denograd_amd.ffi import check
from denograd_amd.tensor import Tensor

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dt,act", [("float16", ffi.F16), ("float32", ffi.F32)])
@pytest.mark.parametrize("n", [1, 63, 511, 512, 513, 3584, 4095, 4096, 4097])
def test_lowest_index_among_the_maxima(hip, dt, act, n):
    rng = np.random.default_rng(n)
    plain = rng.standard_normal(n).astype(dt)
    tie = plain.copy()
    tie[sorted({n - 1, n // 2, n // 3})] = 9                  # the lowest of them wins
    with_nan = tie.copy()
    with_nan[0] = np.nan                                      # never a maximum
    want_nan = n if n == 1 else n // 3 if n // 3 else n // 2 if n // 2 else n - 1
    for x, want in ((plain, int(np.argmax(plain))), (tie, n // 3), (np.full(n, -np.inf, dt), 0), (np.full(n, np.nan, dt), n), (with_nan, want_nan)):
        st, toks, tx = Tensor(np.int32([7, 5])), Tensor.zeros((8,), "int32"), Tensor(x)
        for step in range(2):
            check(hip.jsgrad_hip_argmax(tx.ptr, n, st.ptr, toks.ptr, 8, 1, act))
            assert list(st.numpy()) == [want, 6 + step] and toks.numpy()[5 + step] == want
