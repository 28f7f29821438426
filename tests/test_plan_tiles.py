"""SpMV plans on their own: the tile target follows the matrix and the
workgroups the device holds at once (768 of 512 threads, 1536 of 256), and
every such plan still holds the matrix exactly."""
import numpy as np
import pytest

from oracle.vbr_oracle import vbr_to_dense
from sable_amd import synth
from sable_amd.convert import threshold_routes
from sable_amd.runtime import Plan
from test_plan_host import reconstruct


def _plan(vbr, thr, whole=False, **kw):
    plan = Plan.from_vbr(vbr, thr, host_only=True, **kw)
    if not whole:
        return plan
    D = vbr_to_dense(vbr.val, vbr.indx, vbr.bindx, vbr.rpntr, vbr.cpntr, vbr.bpntrb, vbr.bpntre)
    M, _, cover = reconstruct(plan)
    assert np.array_equal(M, D) and np.all(cover == 1)
    return plan


# one round of slots is kept where the block rows allow it; few tiles are cut
# down to 16 KiB; a given tile size is an upper bound; a given min_tiles halves
# the target as before
@pytest.mark.parametrize("rows,frac,wg", [(900, 0.02, 512), (3000, 0.3, 512), (3000, 0.3, 256), (4000, 0.4, 512)])
def test_target_follows_slots(rows, frac, wg):
    vbr, _, _ = synth.mixed_vbr(rows, rows // 60, 20, 120, frac, 0.5, (0.8, 1.0), (0.05, 0.3), seed=rows)
    thr = threshold_routes(vbr.val, vbr.indx, 15).astype(np.uint8)
    plan = _plan(vbr, thr, whole=True, wg=wg, unroll=2)
    assert 0 < plan.stats["ntiles"] <= 768 * 512 // wg
    small = _plan(vbr, thr, wg=wg, unroll=2, tile_bytes=16 << 10)
    assert small.stats["ntiles"] >= plan.stats["ntiles"]
    many = _plan(vbr, thr, wg=wg, unroll=2, min_tiles=1024)
    assert many.stats["ntiles"] == _plan(vbr, thr, wg=wg, unroll=2, tile_bytes=16 << 10, min_tiles=1).stats["ntiles"] \
        or many.stats["ntiles"] >= 1024
