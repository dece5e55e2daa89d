"""The step state {token, position}: written in stream order, while earlier work that reads it is still queued."""
import numpy as np
import pytest

from denograd_amd import ffi, synthetic
from denograd_amd.ffi import check
from denograd_amd.llama3 import Llama3
from denograd_amd.tensor import Tensor

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n", [1, 2, 300])
def test_state_words_in_stream_order(hip, n):
    state, hist = Tensor(np.zeros(2, np.int32)), Tensor.zeros((n, 2), "int32")
    want = np.array([[i * 7 - 1, 0x7fffffff - i] for i in range(n)], np.int32)
    for i in range(n):
        check(hip.jsgrad_hip_set_state(state.ptr, int(want[i, 0]), int(want[i, 1])))
        check(hip.jsgrad_hip_copy(hist.ptr + i * 8, state.ptr, 8))
    np.testing.assert_array_equal(hist.numpy(), want)


def test_null_state_is_refused(hip):
    with pytest.raises(ffi.HipError, match="null pointer"):
        check(hip.jsgrad_hip_set_state(None, 0, 0))


@pytest.mark.parametrize("number", [int, float, np.int64, np.float32, np.array])
def test_any_number_sets_the_state_of_a_model(hip, number):
    cfg = synthetic.config("tiny16")
    model = Llama3.from_config(cfg).load_weights(synthetic.random_state_dict(cfg, seed=0), quantized=True).model
    model.set_state(number(7), number(3))
    np.testing.assert_array_equal(model.state.numpy().reshape(-1), [7, 3])
