"""Causal attention over several new positions where its grid does not fill the chip: query heads of a kv head share a block, and
the keys are cut into parts whose running sums the last part folds.  Long contexts behind few new positions, parts that hold no
key a row sees, ragged tiles of rows and keys, three heads per kv head.

Tolerance: the float64 restatement rounds probabilities to fp16 after the division, the kernel before it; both roundings are
2^-11 relative per probability, so an output differs by at most 2^-10 of the largest |v| (about 4), as in the cases of
test_gpu_rows.py."""
import numpy as np
import pytest

from denograd_amd.ffi import check
from denograd_amd.tensor import Tensor
from tests.test_gpu_rows import attention_ref

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("hd,H,KV", [(64, 4, 1), (128, 6, 2), (128, 8, 8)])
@pytest.mark.parametrize("B,S,start", [(1, 1, 1500), (1, 57, 1000), (2, 33, 630), (1, 130, 490), (3, 2, 0), (1, 300, 5), (1, 9, 4000)])
def test_attn_prefill_in_key_parts(hip, hd, H, KV, B, S, start):
    rng = np.random.default_rng(S)
    ctx = start + S + 1
    q = rng.standard_normal((B * S, H * hd)).astype(np.float16)
    ck = rng.standard_normal((B, ctx, KV, hd)).astype(np.float16)
    cv = rng.standard_normal((B, ctx, KV, hd)).astype(np.float16)
    tq, tk, tv = Tensor(q), Tensor(ck), Tensor(cv)
    runs = []
    for _ in range(3):
        to = Tensor.full((B * S + 1, H * hd), 5.0, "float16")
        check(hip.jsgrad_hip_attn_prefill(tq.ptr, tk.ptr, tv.ptr, to.ptr, B, S, start, H, KV, hd, ctx))
        runs.append(to.numpy())
    assert np.all(runs[0][B * S] == 5.0)
    assert all(np.array_equal(runs[0].view(np.uint16), r.view(np.uint16)) for r in runs)   # parts are folded in order, whoever is last
    assert np.max(np.abs(runs[0][:B * S].astype(np.float64) - attention_ref(q, ck, cv, B, S, start, H, KV, hd))) < 4e-3


@pytest.mark.parametrize("hd", [64, 128])
def test_the_largest_probability_of_a_row_is_not_rounded(hip, hd):
    """Two keys that a row can see, a tile apart, the later one larger by a factor of 2^5 to 2^8: its probability, the largest, is
    exact in fp16 whatever the maximum was before, so what is off is the rounding of the other (2^-5 times 2^-11 of the
    difference of two values), float sums, and half an fp16 unit of the result."""
    S, start, ctx, small, large = 40, 100, 160, 3, 70
    rng = np.random.default_rng(hd)
    delta = np.linspace(5.0, 7.9, S) * np.log(2.0)
    q = np.zeros((S, hd), np.float16)
    q[:, 0] = delta / 4 * np.sqrt(hd)
    ck = np.zeros((1, ctx, 1, hd), np.float16)
    ck[0, :, 0, 0] = -4000
    ck[0, small, 0, 0], ck[0, large, 0, 0] = 0, 4
    cv = rng.standard_normal((1, ctx, 1, hd)).astype(np.float16)
    tq, tk, tv, to = Tensor(q), Tensor(ck), Tensor(cv), Tensor.empty((S, hd), "float16")
    check(hip.jsgrad_hip_attn_prefill(tq.ptr, tk.ptr, tv.ptr, to.ptr, 1, S, start, 1, 1, hd, ctx))
    w = np.exp(-4.0 * q[:, :1].astype(np.float64) / np.sqrt(hd))
    v = cv[0, :, 0].astype(np.float64)
    ref = (v[large] + w * v[small]) / (1 + w)
    half_unit = np.spacing(np.abs(ref).astype(np.float16)).astype(np.float64) / 2
    assert np.all(np.abs(to.numpy().astype(np.float64) - ref) <= 1.01 * half_unit + 2.0 ** -16 * np.abs(v[large] - v[small]) + 2.0 ** -20)


@pytest.mark.parametrize("hd", [64, 128])
@pytest.mark.parametrize("KV,n_rep,B,S,start", [(3, 1, 3, 130, 5), (3, 3, 5, 37, 70), (1, 5, 2, 131, 0), (2, 6, 3, 9, 200), (7, 7, 1, 61, 3), (1, 16, 3, 17, 64), (5, 33, 1, 6, 1)])
def test_attn_prefill_any_head_geometry(hip, hd, KV, n_rep, B, S, start):
    """Row, block and head numbers are divided by reciprocals: numbers of heads, kv heads and tiles that are not powers of two.  Nothing
    behind the last row is written."""
    H, ctx = KV * n_rep, start + S + 3
    rng = np.random.default_rng(H + S)
    q = rng.standard_normal((B * S, H * hd)).astype(np.float16)
    ck, cv = (rng.standard_normal((B, ctx, KV, hd)).astype(np.float16) for _ in range(2))
    tq, tk, tv, to = Tensor(q), Tensor(ck), Tensor(cv), Tensor.full((B * S + 1, H * hd), 5.0, "float16")
    check(hip.jsgrad_hip_attn_prefill(tq.ptr, tk.ptr, tv.ptr, to.ptr, B, S, start, H, KV, hd, ctx))
    got = to.numpy()
    assert np.all(got[B * S] == 5.0)
    assert np.max(np.abs(got[:B * S].astype(np.float64) - attention_ref(q, ck, cv, B, S, start, H, KV, hd))) < 4e-3
