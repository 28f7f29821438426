"""SpMV on numpy arrays does not wait for another thread's kernel to compile
(marked gpu)."""
import threading
import time

import numpy as np
import pytest

from sable_amd import _lib, synth
from sable_amd.convert import ROUTE_DENSE_MFMA

pytestmark = pytest.mark.gpu


def test_calls_go_on_while_a_plan_compiles(tmp_path):
    from sable_amd import runtime as rt
    rt.init()
    vbr, x, _ = synth.mixed_vbr(900, 20, 5, 100, 0.1, 0.5, (0.8, 1.0), (0.02, 0.2), 4)
    plan = rt.Plan.from_vbr(vbr, None)
    x = np.ascontiguousarray(x, np.float32)
    ref = plan.spmv(x)
    took, errors = [], []

    def compile_one():
        t = time.perf_counter()
        try:
            # N = 112 on MFMA: a kernel of some seconds' compilation, not in the empty cache
            rt.Plan.from_vbr(vbr, np.full(len(vbr.bindx), ROUTE_DENSE_MFMA, np.uint8), op="spmm", n_rhs=112)
        except Exception as e:
            errors.append(e)
        took.append(time.perf_counter() - t)

    print("case: host spmv beside a compilation", flush=True)
    _lib.lib.sable_set_cache_dir(str(tmp_path).encode())
    try:
        th = threading.Thread(target=compile_one)
        th.start()
        calls = []
        while th.is_alive():
            t = time.perf_counter()
            y = plan.spmv(x)
            calls.append(time.perf_counter() - t)
            assert np.array_equal(y, ref)
        th.join()
    finally:
        _lib.lib.sable_set_cache_dir(_lib.RTC_CACHE.encode())
    assert not errors
    print(f"compiled in {took[0]:.2f} s, {len(calls)} calls, the longest {max(calls) * 1e3:.2f} ms", flush=True)
    assert max(calls) < took[0] / 4
