"""MFMA SpMM at N = 16 and 32 with 256 threads and more, where the wavefronts
share the k-steps: tiles of 1 to 16 row units and pieces of fewer k-steps than
wavefronts, as many, and more, against 64-bit sums (marked gpu).  The dropped
products are 2^-24 (three terms) or 3 * 2^-16 (two) relative, the accumulation
is FP32: (terms + 8) * 2^-23, or 2^-14 more, times sum |a x| bounds both."""
import numpy as np
import pytest

from sable_amd.convert import ROUTE_DENSE_MFMA, vbr_to_dense

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module", autouse=True)
def rt():
    from sable_amd import runtime
    runtime.init()
    return runtime


@pytest.mark.parametrize("n_rhs,wg,split", [(16, 256, 3), (16, 512, 3), (32, 256, 3), (32, 512, 2), (16, 256, 2)])
@pytest.mark.parametrize("rows", [1, 16, 33, 64, 81, 113, 128, 250])
@pytest.mark.parametrize("cols,kchunk", [(1, 0), (33, 0), (127, 0), (129, 0), (300, 0), (700, 4)])
def test_units_and_steps(rt, n_rhs, wg, split, rows, cols, kchunk):
    g = np.random.default_rng(rows * 1000 + cols)
    rp, cp = np.array([0, rows, rows + 5]), np.array([0, 3, 3 + cols, 10 + cols])
    bindx, bb, be = np.array([1, 0, 2]), np.array([0, 1]), np.array([1, 3])
    indx = np.concatenate([[0], np.cumsum([rows * cols, 5 * 3, 5 * 7])])
    a = dict(val=g.standard_normal(indx[-1]).astype(np.float32), indx=indx, bindx=bindx, rpntr=rp, cpntr=cp,
             bpntrb=bb, bpntre=be)
    X = g.standard_normal((10 + cols, n_rhs)).astype(np.float32)
    plan = rt.Plan(**a, routes=np.full(3, ROUTE_DENSE_MFMA, np.uint8), op="spmm", n_rhs=n_rhs, wg=wg,
                   mfma_split=split, mfma_kchunk=kchunk)
    Y = plan.spmm(X)
    D = vbr_to_dense(a["val"], indx, bindx, rp, cp, bb, be).astype(np.float64)
    terms = np.count_nonzero(D, axis=1)[:, None]
    bound = ((terms + 8) * 2.0 ** -23 + (2.0 ** -14 if split == 2 else 0)) * (np.abs(D) @ np.abs(X.astype(np.float64)))
    assert np.all(np.abs(Y - D @ X.astype(np.float64)) <= bound)
