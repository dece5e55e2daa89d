"""What the host side of a model call hands to whom: the library, or the model, is replaced by one that writes its calls down."""
import types

import pytest

from denograd_amd import ffi
from denograd_amd.llama import Attention, FeedForward, TransformerBlock
from denograd_amd.llama3 import Llama3

buffer = lambda p: types.SimpleNamespace(ptr=p)
X, XN, H2 = buffer(100), buffer(200), buffer(300)


class Library:
    def __init__(self):
        self.calls = []

    def __getattr__(self, name):
        return lambda *args: self.calls.append((name, args)) or 0


@pytest.fixture
def lib(monkeypatch):
    lib = Library()
    monkeypatch.setattr(ffi, "load", lambda: lib)
    return lib


def block(feed_forward=FeedForward):
    b = TransformerBlock(64, 128, 1, 1, 1e-5, 32, feed_forward=feed_forward)
    for i, layer in enumerate((b.attention.wq, b.attention.wk, b.attention.wv, b.attention.wo, b.feed_forward.w1, b.feed_forward.w2, b.feed_forward.w3)):
        layer.weight = types.SimpleNamespace(ptr=1000 + i, dtype="float16")
    b.attention_norm.weight, b.ffn_norm.weight = buffer(1), buffer(2)
    b.attention.cache_kv = types.SimpleNamespace(ptr=5000, nbytes=64)
    return b


def run(b):
    rows = types.SimpleNamespace(xn=XN, h2=H2, q=buffer(400), attn=buffer(500), g=buffer(600), workspace=buffer(700))
    return b.call_rows(X, 2, 3, 4, buffer(800), buffer(900), rows)


def test_a_block_norms_on_the_way(lib):
    assert run(block()) is X
    assert [name for name, _ in lib.calls] == ["jsgrad_hip_gemm_qkv_rope_norm", "jsgrad_hip_attn_prefill", "jsgrad_hip_gemm", "jsgrad_hip_gemm_ffn_gate_norm", "jsgrad_hip_gemm"]


class OwnAttention(Attention):
    def call_rows(self, xn, bsz, seqlen, start_pos, state, freqs_cis, rows, residual, out):
        self.seen = (xn, residual, out)
        return out


class OwnFeedForward(FeedForward):
    def call_rows(self, xn, n, rows, residual, out):
        self.seen = (xn, residual, out)
        return out


def own_of_the_class(b):
    b.attention.__class__, b.feed_forward.__class__ = OwnAttention, OwnFeedForward


def own_on_the_object(b):
    def attention(xn, bsz, seqlen, start_pos, state, freqs_cis, rows, residual, out):
        b.attention.seen = (xn, residual, out)
        return out

    def feed_forward(xn, n, rows, residual, out):
        b.feed_forward.seen = (xn, residual, out)
        return out

    b.attention.call_rows, b.feed_forward.call_rows = attention, feed_forward


def own_in_the_class(b, monkeypatch):
    monkeypatch.setattr(Attention, "call_rows", OwnAttention.call_rows)
    monkeypatch.setattr(FeedForward, "call_rows", OwnFeedForward.call_rows)


def own_objects(b):
    b.attention, b.feed_forward = types.SimpleNamespace(dim=64), types.SimpleNamespace()
    own_on_the_object(b)


@pytest.mark.parametrize("own", [own_of_the_class, own_in_the_class, own_on_the_object, own_objects])
def test_parts_of_the_callers_own_take_their_rows_normed(lib, own, monkeypatch):
    b = block()
    own(b, *[monkeypatch] * (own is own_in_the_class))
    assert run(b) is X
    assert b.attention.seen == (XN, X, H2) and b.feed_forward.seen == (XN, H2, X)
    assert lib.calls == [("jsgrad_hip_rmsnorm_rows", (X.ptr, 1, XN.ptr, 6, 64, 1e-5)), ("jsgrad_hip_rmsnorm_rows", (H2.ptr, 2, XN.ptr, 6, 64, 1e-5))]


def test_a_model_of_the_callers_own_is_asked_for_its_token_and_its_errors():
    llm, seen = Llama3.__new__(Llama3), []

    class Model:
        def call(self, tokens, start_pos, *sampling):
            seen.append((tokens.tolist(), start_pos, sampling))
            return types.SimpleNamespace(item=lambda: 42.0)

        def check_errors(self):
            seen.append("errors")

    llm.model, llm.start_pos = Model(), 5
    llm.temperature, llm.top_k, llm.top_p, llm.alpha_f, llm.alpha_p = 0.5, 1, 0.2, 0.3, 0.4
    assert llm._call(7) == 42
    assert seen == [([[7]], 5, (0.5, 1, 0.2, 0.3, 0.4)), "errors"]
