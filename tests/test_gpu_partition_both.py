"""Both axes of the partitioner from one upload (marked gpu): the device
transpose's chunk edges, and the matrices that keep the per-axis path, all
against the host partitioner."""
import numpy as np
import pytest
import scipy.sparse

from sable_amd import autopartition as AP

pytestmark = pytest.mark.gpu


def _random(n, m, density, seed):
    rng = np.random.default_rng(seed)
    A = scipy.sparse.random(n, m, density=density, format="csc", random_state=rng, data_rvs=rng.standard_normal)
    A.sort_indices()
    if A.nnz:
        A.data[rng.choice(A.nnz, A.nnz // 40, replace=False)] = 0.0       # stored zeros
    return A


# columns around one, two and three per chunk of 512; one line; every row full
@pytest.mark.parametrize("n,m,d", [(50, 1, 0.5), (1, 50, 0.5), (300, 511, 0.05), (300, 512, 0.05), (300, 513, 0.05),
                                   (70, 1500, 0.2), (2000, 1023, 0.02), (257, 64, 1.0), (40, 30, 0.0)])
@pytest.mark.parametrize("kind", ["similarity2", "similarity2_numba", "similarity1"])
def test_both_axes_match_host(n, m, d, kind):
    A = _random(n, m, d, n * 7 + m)
    sim = getattr(AP, kind)
    print(f"case: {n}x{m} density {d} {kind}", flush=True)
    assert AP._both_cuts_gpu(A, 0.2, sim) is not None
    for thr in (0.05, 0.2):
        assert AP.cut_indices2(A, thr, sim, device=True) == AP.cut_indices2(A, thr, sim)


def test_what_keeps_the_per_axis_path():
    A = _random(200, 150, 0.1, 3)
    unsorted = scipy.sparse.csc_matrix((A.data.copy(), A.indices.copy(), A.indptr.copy()), shape=A.shape)
    j = int(np.argmax(np.diff(A.indptr)))
    a, b = A.indptr[j], A.indptr[j] + 1
    unsorted.indices[[a, b]] = unsorted.indices[[b, a]]
    unsorted.data[[a, b]] = unsorted.data[[b, a]]
    dup = A.copy()
    dup.indices = dup.indices.copy()
    dup.indices[a + 1] = dup.indices[a]                                   # a repeated row in one column
    dup.has_canonical_format = False
    for name, M in (("unsorted", unsorted), ("duplicate", dup)):
        print(f"case: {name}", flush=True)
        assert AP._both_cuts_gpu(M, 0.2, AP.similarity2) is None
        assert AP.cut_indices2(M, 0.2, AP.similarity2, device=True) == AP.cut_indices2(M, 0.2, AP.similarity2)
    for dt in (np.float32, np.int32, bool):
        M = (A * 3).astype(dt)
        assert AP.cut_indices2(M, 0.2, AP.similarity2, device=True) == AP.cut_indices2(M, 0.2, AP.similarity2)
    with pytest.raises(ValueError):
        AP.cut_indices2(A, 0.2, lambda x, y: 0.0, device=True)
