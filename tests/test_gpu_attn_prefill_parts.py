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
