"""The step state {token, position}: written in stream order, while earlier work that reads it is still queued."""
import ctypes as C
import threading

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


def test_read_step_returns_the_token_and_the_error_word_in_stream_order(hip):
    """Every read sees what was queued before it and nothing older; the error word is the one of the workspace named, and stays."""
    state, wo, attn = Tensor(np.zeros(2, np.int32)), Tensor.zeros((512,), "uint8"), Tensor.zeros((256,), "uint8")
    words = (C.c_int32 * 2)()
    for i in range(300):
        token = (i * 40503 - 7) & 0x7fffffff
        check(hip.jsgrad_hip_set_state(state.ptr, token, i))
        check(hip.jsgrad_hip_memset(wo.ptr + 256, i % 3, 4))
        check(hip.jsgrad_hip_memset(attn.ptr, i % 5, 4))
        check(hip.jsgrad_hip_read_step(state.ptr, wo.ptr, attn.ptr, words))
        assert list(words) == [token, i % 3 * 0x01010101]
        check(hip.jsgrad_hip_read_step(state.ptr, None, attn.ptr, words))
        assert list(words) == [token, i % 5 * 0x01010101]
    check(hip.jsgrad_hip_read_step(state.ptr, None, None, words))
    assert list(words) == [token, 0]
    with pytest.raises(ffi.HipError, match="null pointer"):
        check(hip.jsgrad_hip_read_step(None, None, None, words))


def test_read_step_from_two_threads(hip):
    states = [Tensor(np.array([t * 1000 + 5, 0], np.int32)) for t in range(2)]
    bad, done = [], [0, 0]

    def loop(t):
        words = (C.c_int32 * 2)()
        for _ in range(200):
            check(hip.jsgrad_hip_read_step(states[t].ptr, None, None, words))
            done[t] += 1                                      # a thread that an error has ended stays below 200
            if list(words) != [t * 1000 + 5, 0]:
                bad.append((t, list(words)))

    threads = [threading.Thread(target=loop, args=(t,)) for t in range(2)]
    for t in threads:
        t.start()
    for t in threads:
        t.join()
    assert not bad and done == [200, 200]


def test_an_error_of_the_attention_launches_is_raised_with_the_token(hip):
    cfg = synthetic.config("tiny16")
    llm = Llama3.from_config(cfg).load_weights(synthetic.random_state_dict(cfg, seed=0), quantized=True)
    llm.chat_tokens([1, 2, 3], 2)
    assert llm.model._ctx.fuse_attn_wo
    check(hip.jsgrad_hip_memset(llm.model._ctx.attn_wo_ws.ptr + 256, 1, 4))     # as a bounded wait that ran out would leave it
    with pytest.raises(ffi.HipError, match="gave up waiting"):
        llm._call(4)


def test_the_token_is_the_one_that_the_models_call_returns(hip):
    """A call of the user's own on top of the model's, which picks another token from the logits."""
    cfg = synthetic.config("tiny16")
    llm = Llama3.from_config(cfg).load_weights(synthetic.random_state_dict(cfg, seed=0), quantized=True)
    plain = llm.model.call

    def second_best(*args):
        plain(*args)
        return Tensor(np.argsort(llm.model.logits.numpy().astype(np.float32))[-2:-1].astype(np.int32))

    llm.chat_tokens([1, 2, 3], 2)
    llm.model.call = second_best
    got = llm._call(4)
    llm.model.call = plain
    order = np.argsort(llm.model.logits.numpy().astype(np.float32))
    assert got == order[-2] != order[-1]
    assert llm._call(4) == llm.model.state.numpy()[0]
