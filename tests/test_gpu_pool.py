"""GPU: device memory that a context keeps between runs is given back when the
caller asks for it, and a context can be told to keep none."""
import ctypes as C

import numpy as np
import pytest

import bellhopcuda_amd as bh
from bellhopcuda_amd.env import munk_env
from parity import env_context

pytestmark = pytest.mark.gpu

GB = 1 << 30


def _free_bytes():
    hip = C.CDLL("libamdhip64.so")
    f, t = C.c_size_t(), C.c_size_t()
    assert hip.hipMemGetInfo(C.byref(f), C.byref(t)) == 0
    return f.value


# 2121 receivers with 65536 candidate slots of 64 bytes: 8.9e9 bytes
def _arrivals():
    return bh.Problem(munk_env(nbeams=101, nrz=21, nrr=101, run_type="AG"))


def test_trim_gives_the_memory_back():
    print("\n[gpu-case] pool_trim", flush=True)
    p = _arrivals()
    ctx = bh.Context(0)
    try:
        a = bh.field_run(p, ctx=ctx, max_narr=10)
        held = _free_bytes()
        ctx.trim()
        assert _free_bytes() - held > 8 * GB
        b = bh.field_run(p, ctx=ctx, max_narr=10)
        assert a.narr.sum() > 0 and np.array_equal(a.narr, b.narr) and bytes(a.arr) == bytes(b.arr)
    finally:
        ctx.close()


def test_nothing_kept_without_a_limit():
    print("\n[gpu-case] pool_limit_0", flush=True)
    p = _arrivals()
    ctx = env_context(BHC_POOL_MB=0)
    try:
        bh.field_run(munk_env(nbeams=11, nrz=5, nrr=11), ctx=ctx)     # the segment buffer is the context's for good
        before = _free_bytes()
        r = bh.field_run(p, ctx=ctx, max_narr=10)
        assert r.narr.sum() > 0 and before - _free_bytes() < GB
    finally:
        ctx.close()
