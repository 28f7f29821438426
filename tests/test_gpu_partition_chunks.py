"""The device transpose where the rows leave few chunks of columns (marked
gpu): 64 MiB of counts are eight chunks at 2 M rows and one above 8 M."""
import numpy as np
import pytest
import scipy.sparse

from sable_amd import autopartition as AP

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("nrows,ncols", [((1 << 21) + 3, 21), ((1 << 23) + 5, 3)])
def test_few_chunks(nrows, ncols):
    rng = np.random.default_rng(ncols)
    cols = []
    for _ in range(ncols):                              # runs of rows, so that neighbours overlap
        start = rng.integers(0, nrows - 50, 40)
        cols.append(np.unique((start[:, None] + np.arange(50)).ravel()))
    ip = np.concatenate([[0], np.cumsum([len(c) for c in cols])])
    ix = np.concatenate(cols).astype(np.int32)
    A = scipy.sparse.csc_matrix((rng.integers(1, 5, len(ix)).astype(np.float64), ix, ip), shape=(nrows, ncols))
    print(f"case: {nrows}x{ncols}", flush=True)
    both = AP._both_cuts_gpu(A, 0.2, AP.similarity2)
    assert both == (AP._axis_cuts_gpu(A, 0.2, AP.similarity2), AP._axis_cuts_gpu(A.T.tocsc(), 0.2, AP.similarity2))
