"""SpMV on numpy arrays (marked gpu): the pinned path gives the bits of the
device path for every call, from several threads at once, and so does the
path for longer vectors."""
import threading

import numpy as np
import pytest

from sable_amd import synth

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def rt():
    from sable_amd import runtime
    runtime.init()
    return runtime


def _device(rt, plan, x):
    y = rt.DeviceArray(plan.nrows)
    plan.spmv(rt.DeviceArray.from_numpy(x), y)
    return y.numpy()


def test_calls_and_threads_match_the_device_path(rt):
    jobs = []
    for seed, n in ((1, 700), (2, 2600), (3, 5000)):
        vbr, _, _ = synth.mixed_vbr(n, n // 50, 5, 100, 0.1, 0.5, (0.8, 1.0), (0.02, 0.2), seed)
        plan = rt.Plan.from_vbr(vbr, None)
        xs = [np.random.default_rng(10 * seed + k).uniform(-1, 1, n).astype(np.float32) for k in range(8)]
        jobs.append((plan, xs, [_device(rt, plan, x) for x in xs]))
    bad = []

    def work(plan, xs, ref):
        for _ in range(5):
            for x, r in zip(xs, ref):
                if not np.array_equal(plan.spmv(x), r):
                    bad.append(len(x))

    print("case: host spmv from three threads", flush=True)
    threads = [threading.Thread(target=work, args=j) for j in jobs]
    for t in threads:
        t.start()
    for t in threads:
        t.join()
    assert not bad


@pytest.mark.parametrize("n", [1, (1 << 20), (1 << 20) + 1])
def test_vector_lengths(rt, n):
    """One block of 3 x min(n, 40) at the end of an n-column matrix: the
    longest vectors of the pinned path, and beyond it."""
    w = min(n, 40)
    val = np.random.default_rng(n).standard_normal(3 * w).astype(np.float32)
    cp = [0, n] if n == w else [0, n - w, n]
    plan = rt.Plan(val, [0, 3 * w], [len(cp) - 2], [0, 3], cp, [0], [1])
    x = np.random.default_rng(4).uniform(-1, 1, n).astype(np.float32)
    print(f"case: host spmv n={n}", flush=True)
    y = plan.spmv(x)
    assert np.array_equal(y, _device(rt, plan, x))
    ref = val.reshape(w, 3).T.astype(np.float64) @ x[n - w:]
    assert np.max(np.abs(y - ref)) <= 1e-5 * np.sum(np.abs(val))
