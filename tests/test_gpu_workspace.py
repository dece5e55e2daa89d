"""The workspace of the several-row calls: one block that the library keeps, whatever LRU says, that nobody else is handed, and
without which the calls give the same results to a rounding."""
import ctypes as C
import os
import subprocess
import sys

import numpy as np
import pytest

from denograd_amd import ffi
from denograd_amd.ffi import check
from denograd_amd.tensor import Tensor

pytestmark = pytest.mark.gpu
ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))


def mem(hip):
    live, idle = C.c_size_t(), C.c_size_t()
    check(hip.jsgrad_hip_mem_info(C.byref(live), C.byref(idle)))
    return live.value, idle.value


def calls(hip):
    """K parts and their sums, a realised matrix with sums behind it, key parts."""
    from tests import test_gpu_attn_prefill_parts as attn
    from tests import test_gpu_gemm_tile as tile
    for kind in ("float16", "int8", "nf4"):
        tile.test_tiled_gemm_at_the_edges(hip, kind, 65, 384, 8192)
        tile.test_tiled_gemm_at_the_edges(hip, kind, 2100, 128, 8192)
    attn.test_attn_prefill_in_key_parts(hip, 128, 8, 8, 1, 57, 1000)


def test_workspace_is_kept_and_is_nobodys_buffer(hip):
    out_f, in_f, rows = 384, 8192, 65
    w, x, y = Tensor.zeros((out_f, in_f), "float16"), Tensor.zeros((rows, in_f), "float16"), Tensor.empty((rows, out_f), "float16")
    check(hip.jsgrad_hip_free_cache())
    live, idle = mem(hip)
    assert idle == 0
    check(hip.jsgrad_hip_gemm(ffi.W_F16, w.ptr, None, out_f, in_f, x.ptr, rows, y.ptr, None))
    size = mem(hip)[1]
    assert size > 0 and mem(hip)[0] == live
    p = C.c_void_p()
    check(hip.jsgrad_hip_malloc(size, C.byref(p)))      # a buffer of the workspace's own size
    assert mem(hip)[1] == size
    check(hip.jsgrad_hip_gemm(ffi.W_F16, w.ptr, None, out_f, in_f, x.ptr, rows, y.ptr, None))
    assert mem(hip) == (live + size, size)
    check(hip.jsgrad_hip_free(p))
    check(hip.jsgrad_hip_free_cache())
    assert mem(hip) == (live, 0)


CHILD = """
import sys
sys.path.insert(0, sys.argv[1])
from denograd_amd import ffi
from tests.test_gpu_workspace import calls, mem
hip = ffi.load()
ffi.check(hip.jsgrad_hip_init(0))
calls(hip)
first = mem(hip)[1]
calls(hip)
print(first, mem(hip)[1])
"""


@pytest.mark.parametrize("mb,kept", [(None, True), (0, False), (1, None)])
def test_several_row_calls_without_reuse_of_blocks(hip, mb, kept):
    """LRU=0 in a process of its own: the workspace alone stays between calls.  Without one (0), and with one that holds the sums of
    some calls and no realised matrix (1), the results are the same to a rounding."""
    env = {**os.environ, "LRU": "0", **({"JSGRAD_HIP_WORKSPACE_MB": str(mb)} if mb is not None else {})}
    r = subprocess.run([sys.executable, "-c", CHILD, ROOT], env=env, capture_output=True, text=True, timeout=110)
    assert r.returncode == 0, r.stdout + r.stderr
    first, second = map(int, r.stdout.split())
    assert kept is None or (first > 0) == kept
    assert kept is not True or first == second
