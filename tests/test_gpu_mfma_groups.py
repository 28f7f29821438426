"""MFMA SpMM at the widths whose column groups are 48 and 32 wide (marked
gpu): tile numbers around the XCD order's eights, k chunks whose partial-sum
blocks lie N apart, both splits, against 64-bit sums.

The bound: FP32 sums of K products err by (K + 8) 2^-23 sum|a x|; the
three-term split drops products below 2^-24, the two-term split three of
2^-18 each."""
import numpy as np
import pytest

from sable_amd.convert import ROUTE_DENSE_MFMA, vbr_to_dense

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module", autouse=True)
def rt():
    from sable_amd import runtime
    runtime.init()
    return runtime


@pytest.mark.parametrize("n_rhs,wg,split", [(96, 128, 3), (96, 256, 3), (96, 256, 2), (144, 256, 3), (160, 128, 3),
                                            (160, 256, 3), (224, 256, 3), (240, 256, 3)])
@pytest.mark.parametrize("heights", [[5], [33, 17, 130, 16, 40, 1, 64], [20] * 17])
def test_groups(rt, n_rhs, wg, split, heights):
    g = np.random.default_rng(n_rhs + len(heights))
    w = [70, 9, 101]
    nr = len(heights)
    rp, cp = np.concatenate([[0], np.cumsum(heights)]), np.concatenate([[0], np.cumsum(w)])
    bindx = np.tile([0, 2], nr)                         # two ranges with a gap
    indx = np.concatenate([[0], np.cumsum(np.repeat(heights, 2) * np.asarray(w)[bindx])])
    bb = 2 * np.arange(nr)
    a = dict(val=g.standard_normal(indx[-1]).astype(np.float32), indx=indx, bindx=bindx, rpntr=rp, cpntr=cp, bpntrb=bb,
             bpntre=bb + 2)
    X = g.standard_normal((int(cp[-1]), n_rhs)).astype(np.float32)
    D = vbr_to_dense(a["val"], indx, bindx, rp, cp, bb, bb + 2).astype(np.float64)
    X64 = X.astype(np.float64)
    bound = ((171 + 8) * 2.0 ** -23 + (2.0 ** -16 if split == 2 else 0)) * (np.abs(D) @ np.abs(X64))
    for kchunk in (-1, 2):
        print(f"case: groups N {n_rhs} wg {wg} split {split} block rows {nr} kchunk {kchunk}", flush=True)
        plan = rt.Plan(**a, routes=np.full(2 * nr, ROUTE_DENSE_MFMA, np.uint8), op="spmm", n_rhs=n_rhs, wg=wg,
                       mfma_split=split, mfma_kchunk=kchunk)
        assert np.all(np.abs(plan.spmm(X) - D @ X64) <= bound)
