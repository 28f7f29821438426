"""SpMV tiles whose first dense batch is loaded while x is staged: staging
groups that begin with a dense piece, hold one behind a sparse piece, behind
several, or none, against 64-bit sums (marked gpu).  The bound is that of any
order of summation in FP32: terms * 2^-24 * sum |a x| per row."""
import numpy as np
import pytest

from sable_amd import synth
from sable_amd.convert import ROUTE_DENSE, ROUTE_SPARSE, vbr_to_dense

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module", autouse=True)
def rt():
    from sable_amd import runtime
    runtime.init()
    return runtime


# xcap: one group per tile, or several of a few blocks; routes: all dense, all
# sparse, alternating (sparse before dense in a group), dense only at the end
@pytest.mark.parametrize("xcap", [60, 300, 4095])
@pytest.mark.parametrize("routes", ["dense", "sparse", "mixed", "last"])
@pytest.mark.parametrize("wg,unroll", [(64, 1), (256, 4), (512, 2)])
def test_groups(rt, xcap, routes, wg, unroll):
    vbr, x, _ = synth.mixed_vbr(700, 14, 1, 90, 0.5, 0.5, (0.8, 1.0), (0.05, 0.3), seed=11, ncols=900, col_parts=40)
    nb = len(vbr.bindx)
    r = {"dense": np.zeros(nb), "sparse": np.ones(nb), "mixed": np.arange(nb) % 2,
         "last": np.arange(nb) < nb - nb // 8}[routes].astype(np.uint8)
    r = np.where(r == 1, ROUTE_SPARSE, ROUTE_DENSE).astype(np.uint8)
    print(f"case: xcap {xcap} {routes} wg {wg} unroll {unroll}", flush=True)
    plan = rt.Plan.from_vbr(vbr, r, wg=wg, unroll=unroll, xcap=xcap, min_tiles=1)
    y = plan.spmv(np.asarray(x, dtype=np.float32))
    D = vbr_to_dense(vbr.val, vbr.indx, vbr.bindx, vbr.rpntr, vbr.cpntr, vbr.bpntrb, vbr.bpntre).astype(np.float64)
    x64 = np.asarray(x, dtype=np.float32).astype(np.float64)
    bound = (np.count_nonzero(D, axis=1) + 8) * 2.0 ** -24 * (np.abs(D) @ np.abs(x64))
    assert np.all(np.abs(y - D @ x64) <= bound + 1e-30)
