"""Which matrices the partitioner transposes on the GPU: none whose chunk of
columns, walked one after another, would take longer than the host's
transpose."""
import scipy.sparse

from sable_amd import autopartition as AP


def test_many_lines_of_few_entries_keep_the_host_transpose():
    # one chunk of all columns: declined before any GPU call
    A = scipy.sparse.identity(9_000_000, format="csc")
    assert AP._both_cuts_gpu(A, 0.2, AP.similarity2) is None


def test_rule():
    pays = AP._device_transpose_pays
    assert pays(1, 1, 0) and pays(6007, 6007, 1_900_000) and pays(1 << 25, 40, 0)
    assert pays(500_000, 500_000, 2_500_000) and pays(1000, 1 << 20, 1 << 20)
    assert not pays(2_000_000, 2_000_000, 10_000_000)           # 250,000 columns a chunk: 88 ms against 60
    assert pays(2_000_000, 2_000_000, 100_000_000)              # the same against 600
    assert not pays(1 << 25, 1 << 25, 1 << 27)
