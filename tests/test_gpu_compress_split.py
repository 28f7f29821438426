"""Compression on the GPU where blocks are gathered by several wavefronts and
rows walked by several threads (sb_gather_dense, sb_csr_rows): the sizes at
which the shares change, against the host's arrays, bit for bit."""
import numpy as np
import pytest

from sable_amd import convert as C

pytestmark = pytest.mark.gpu


# block rows, block columns: one value; 64 rows and one more; blocks of
# 512 * 2 values and one less (one wavefront or two); 32 sparse columns per
# segment, 16 segments and beyond, shares that cut a block; widths of 1
@pytest.mark.parametrize("hs,ws", [
    ([1], [1]),
    ([64], [64]),
    ([65, 63], [63, 1, 64]),
    ([32], [31, 32]),
    ([31, 33], [33, 32]),
    ([257, 1, 300], [300, 1, 211]),
    ([7, 200], [1] * 40 + [513]),
    ([130], [9, 700, 2, 1000]),
])
@pytest.mark.parametrize("keep", [1, 2])
def test_shares_match_host(hs, ws, keep):
    rng = np.random.default_rng(len(ws) * 100 + hs[0] + keep)
    rp, cp = np.concatenate([[0], np.cumsum(hs)]), np.concatenate([[0], np.cumsum(ws)])
    size = np.outer(hs, ws).ravel()
    nb = len(size)
    indx = np.concatenate([[0], np.cumsum(size)])
    v = rng.standard_normal(indx[-1])
    v[rng.random(len(v)) < 0.4] = 0.0
    v[0] = np.nan                                 # kept: it is not zero
    bb = np.arange(len(hs)) * len(ws)
    bindx = np.tile(np.arange(len(ws)), len(hs))
    for routes in (np.zeros(nb), np.ones(nb), np.arange(nb) % (keep + 1) > 0):
        a = (v, rp.tolist(), cp.tolist(), indx.tolist(), bindx.tolist(), bb.tolist(), (bb + len(ws)).tolist(),
             np.asarray(routes).astype(np.uint8))
        print(f"case: {hs} x {ws[:4]}.. sparse blocks {int(a[-1].sum())}", flush=True)
        for h, d in zip(C.compress_with_routes(*a), C.compress_with_routes_device(*a)):
            assert h.dtype == d.dtype and np.array_equal(h, d, equal_nan=h.dtype.kind == "f")
