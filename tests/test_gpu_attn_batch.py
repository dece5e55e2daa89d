"""Attention of many sequences at one new position each, where the chunks' length changes with the position and the number of
sequences: one chunk in all (nothing to merge), the first with two, and both sides of every line between lengths.  One workspace
serves all positions in turn, so each launch leaves its counters as it found them.

Tolerance: the float64 result rounded to fp16 and the float sums in another order, as in test_gpu_rows."""
import numpy as np
import pytest

from denograd_amd.ffi import check
from denograd_amd.tensor import Tensor
from tests.test_gpu_rows import attention_ref

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("hd,B,H,KV,positions", [
    (64, 2, 8, 2, (1, 64, 65, 256, 257, 300, 799, 800, 1399, 1400, 1)),
    (128, 2, 6, 2, (1, 32, 33, 160, 161, 399, 400, 799, 800, 160, 1500)),
    (64, 20, 8, 8, (256, 257, 599, 600, 3)), (128, 20, 16, 8, (160, 161, 600, 97)),
    (64, 3, 8, 1, (70, 300)), (128, 3, 8, 1, (70, 300)),
])
def test_attn_decode_batch_at_the_chunk_lines(hip, hd, B, H, KV, positions):
    rng = np.random.default_rng(hd + B)
    ctx = max(positions) + 5
    q = rng.standard_normal((B, H * hd)).astype(np.float16)
    ck, cv = (rng.standard_normal((B, ctx, KV, hd)).astype(np.float16) for _ in range(2))
    tq, tk, tv = Tensor(q), Tensor(ck), Tensor(cv)
    ws = Tensor.zeros((hip.jsgrad_hip_attn_batch_workspace_bytes(B, H, KV, hd),), "uint8")
    for T in positions:
        st = Tensor(np.array([0, T - 1], np.int32))
        out = Tensor.full((B + 1, H * hd), 7.0, "float16")
        check(hip.jsgrad_hip_attn_decode_batch(tq.ptr, tk.ptr, tv.ptr, st.ptr, out.ptr, ws.ptr, B, H, KV, hd, ctx))
        got = out.numpy().astype(np.float64)
        assert np.all(got[B] == 7.0)
        ref = attention_ref(q, ck, cv, B, 1, T - 1, H, KV, hd)
        assert np.max(np.abs(got[:B] - ref)) < 4e-3, T


@pytest.mark.parametrize("hd,B,H,KV,positions", [
    (64, 1, 8, 2, (1, 31, 32, 33, 127, 128, 129, 385, 2100, 4096, 9000)), (128, 1, 12, 4, (15, 16, 17, 64, 65, 257, 1025, 8200)),   # many blocks to a pair
    (64, 16, 16, 16, (128, 129, 400, 513, 5)), (128, 16, 16, 16, (64, 193, 256, 257, 500)),   # one
    (64, 41, 32, 8, (50, 900)), (128, 41, 24, 8, (50, 450)),   # more pairs than compute units
    (64, 33, 32, 8, (50, 896, 897, 1500)), (128, 36, 24, 8, (448, 449, 1400)),   # a few more
    (64, 18, 32, 8, (1152, 1153, 2200)), (128, 20, 24, 8, (1472, 1473, 1700)),   # one unit a pair leaves many idle
    (64, 4, 16, 2, (40, 700)), (128, 4, 16, 2, (40, 700)), (64, 4, 6, 2, (40, 700)), (128, 3, 2, 1, (40, 700)),
])
def test_attn_decode_batch_at_the_edges_of_tiles(hip, hd, B, H, KV, positions):
    """Part tiles, wavefronts and blocks with no or one tile, merges of one and of several batches of blocks, every number of query heads per kv
    head.  The cache behind the position holds no numbers, which must not be met by a weight of zero."""
    rng = np.random.default_rng(hd + B + H)
    ctx = max(positions) + 5
    q = rng.standard_normal((B, H * hd)).astype(np.float16)
    ck, cv = (rng.standard_normal((B, ctx, KV, hd)).astype(np.float16) for _ in range(2))
    tq = Tensor(q)
    ws = Tensor.zeros((hip.jsgrad_hip_attn_batch_workspace_bytes(B, H, KV, hd),), "uint8")
    for T in positions:
        k, v = ck.copy(), cv.copy()
        k[:, T:], v[:, T:] = np.nan, np.inf
        tk, tv = Tensor(k), Tensor(v)
        st = Tensor(np.array([0, T - 1], np.int32))
        for _ in range(2):                                    # the counters come back to zero
            out = Tensor.full((B + 1, H * hd), 7.0, "float16")
            check(hip.jsgrad_hip_attn_decode_batch(tq.ptr, tk.ptr, tv.ptr, st.ptr, out.ptr, ws.ptr, B, H, KV, hd, ctx))
            got = out.numpy().astype(np.float64)
            assert np.all(got[B] == 7.0)
            ref = attention_ref(q, ck, cv, B, 1, T - 1, H, KV, hd)
            assert np.max(np.abs(got[:B] - ref)) < 4e-3, T


@pytest.mark.parametrize("hd,B,H,KV,T", [(64, 1, 8, 1, 20000), (128, 2, 4, 2, 12000), (128, 33, 8, 8, 1400)])
def test_the_workspace_has_room_for_the_most_blocks(hip, hd, B, H, KV, T):
    """Nothing behind the bytes that the library asks for is written; counters are zero again.  The last sequence's partial results end where they do."""
    rng = np.random.default_rng(T)
    q = rng.standard_normal((B, H * hd)).astype(np.float16)
    ck, cv = (rng.standard_normal((B, T, KV, hd)).astype(np.float16) for _ in range(2))
    nbytes = hip.jsgrad_hip_attn_batch_workspace_bytes(B, H, KV, hd)
    assert nbytes == B * (256 + H * 64 * (hd + 2) * 4)
    ws = Tensor(np.concatenate([np.zeros(nbytes, np.uint8), np.full(4096, 7, np.uint8)]))
    tq, tk, tv, st, out = Tensor(q), Tensor(ck), Tensor(cv), Tensor(np.array([0, T - 1], np.int32)), Tensor.full((B, H * hd), 7.0, "float16")
    check(hip.jsgrad_hip_attn_decode_batch(tq.ptr, tk.ptr, tv.ptr, st.ptr, out.ptr, ws.ptr, B, H, KV, hd, T))
    words = ws.numpy()
    assert np.all(words[nbytes:] == 7) and not words[:B * KV * 4].any()
    assert np.max(np.abs(out.numpy().astype(np.float64) - attention_ref(q, ck, cv, B, 1, T - 1, H, KV, hd))) < 4e-3
