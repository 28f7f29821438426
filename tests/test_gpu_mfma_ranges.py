"""MFMA pieces whose X rows come from 1 to 9 separate column ranges, and tiles
of several pieces (xcap), against 64-bit sums (marked gpu).  The dropped
products of the three-term split are 2^-24 relative, the accumulation is FP32:
(terms + 8) * 2^-23 * sum |a x| bounds both."""
import numpy as np
import pytest

from sable_amd.convert import ROUTE_DENSE_MFMA, vbr_to_dense

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module", autouse=True)
def rt():
    from sable_amd import runtime
    runtime.init()
    return runtime


@pytest.mark.parametrize("nranges", [1, 3, 4, 5, 9])
@pytest.mark.parametrize("n_rhs,wg", [(16, 128), (64, 256), (128, 256), (128, 512)])
@pytest.mark.parametrize("xcap", [40, 4095])
def test_ranges(rt, nranges, n_rhs, wg, xcap):
    g = np.random.default_rng(nranges)
    rows, w = [33, 17], [7 + 3 * (j % 4) for j in range(2 * nranges + 1)]
    rp, cp = np.concatenate([[0], np.cumsum(rows)]), np.concatenate([[0], np.cumsum(w)])
    bindx = np.concatenate([np.arange(nranges) * 2, np.arange(nranges) * 2 + 1])   # every other block column
    size = np.array([h * w[b] for h, b in zip(np.repeat(rows, nranges), bindx)])
    indx = np.concatenate([[0], np.cumsum(size)])
    bb = np.array([0, nranges])
    a = dict(val=g.standard_normal(indx[-1]).astype(np.float32), indx=indx, bindx=bindx, rpntr=rp, cpntr=cp,
             bpntrb=bb, bpntre=bb + nranges)
    X = g.standard_normal((int(cp[-1]), n_rhs)).astype(np.float32)
    print(f"case: ranges {nranges} N {n_rhs} wg {wg} xcap {xcap}", flush=True)
    plan = rt.Plan(**a, routes=np.full(len(bindx), ROUTE_DENSE_MFMA, np.uint8), op="spmm", n_rhs=n_rhs, wg=wg,
                   xcap=xcap)
    Y = plan.spmm(X)
    D = vbr_to_dense(a["val"], indx, bindx, rp, cp, bb, bb + nranges).astype(np.float64)
    X64 = X.astype(np.float64)
    bound = (np.count_nonzero(D, axis=1)[:, None] + 8) * 2.0 ** -23 * (np.abs(D) @ np.abs(X64))
    assert np.all(np.abs(Y - D @ X64) <= bound)
