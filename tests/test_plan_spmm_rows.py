"""SpMM plans keep max_seg_rows as the upper bound of their tiles' heights
(MFMA tiles, whole 16-row units, from 16 on) and still hold the matrix."""
import numpy as np
import pytest

from oracle.vbr_oracle import vbr_to_dense
from sable_amd import synth
from sable_amd.convert import ROUTE_DENSE, ROUTE_DENSE_MFMA, ROUTE_SPARSE
from sable_amd.runtime import Plan
from test_plan_host import reconstruct


@pytest.mark.parametrize("n_rhs", [16, 128])
@pytest.mark.parametrize("rows", [1, 5, 15, 16, 17, 20, 31, 40, 100, 128])
@pytest.mark.parametrize("kinds", [[ROUTE_DENSE, ROUTE_SPARSE], [ROUTE_DENSE, ROUTE_SPARSE, ROUTE_DENSE_MFMA]])
def test_max_seg_rows(kinds, rows, n_rhs):
    vbr, _, _ = synth.mixed_vbr(700, 9, 1, 190, 0.4, 0.5, (0.8, 1.0), (0.05, 0.3), seed=rows)
    routes = np.random.default_rng(rows).choice(kinds, len(vbr.bindx)).astype(np.uint8)
    plan = Plan.from_vbr(vbr, routes, op="spmm", n_rhs=n_rhs, wg=256, max_seg_rows=rows, host_only=True)
    tiles, nm = plan.export("tiles"), plan.stats["ntiles_mfma"]
    assert tiles["nrows"][nm:].max() <= rows and (nm == 0 or tiles["nrows"][:nm].max() <= max(rows // 16 * 16, 16))
    if nm == 0:
        D = vbr_to_dense(vbr.val, vbr.indx, vbr.bindx, vbr.rpntr, vbr.cpntr, vbr.bpntrb, vbr.bpntre)
        M, _, cover = reconstruct(plan)
        assert np.array_equal(M, D) and np.all(cover == 1)


def test_default_tiles_are_whole_fragments():
    vbr, _, _ = synth.mixed_vbr(700, 9, 1, 190, 0.4, 0.5, (0.8, 1.0), (0.05, 0.3), seed=3)
    plan = Plan.from_vbr(vbr, None, op="spmm", n_rhs=64, wg=256, host_only=True)
    start = vbr.rpntr[np.searchsorted(vbr.rpntr, plan.export("tiles")["row0"], side="right") - 1]
    assert np.all((plan.export("tiles")["row0"] - start) % 16 == 0)
