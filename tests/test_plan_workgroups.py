"""SpMV plans on their own in workgroups other than the tuned 512 threads:
below 256 the tile target is halved until there are 1,024 tiles, above it may
reach the tuned 512 KiB, and one workgroup per CU counts as two."""
import numpy as np
import pytest

from sable_amd.runtime import Plan


def _plan(block_rows, height, width, per_row, **kw):
    n = block_rows * per_row
    val = np.ones(n * height * width, np.float32)
    bindx = np.tile(np.arange(per_row), block_rows)
    begin = np.arange(block_rows) * per_row
    return Plan(val, np.arange(n + 1) * height * width, bindx, np.arange(block_rows + 1) * height,
                np.arange(per_row + 1) * width, begin, begin + per_row, host_only=True, **kw)


@pytest.mark.parametrize("wg", [64, 128])
@pytest.mark.parametrize("shape", [(5000, 8, 50, 10), (40, 100, 100, 40), (3, 20, 10, 2)])
def test_small_workgroups_halve(wg, shape):
    plan, asked = _plan(*shape, wg=wg), _plan(*shape, wg=wg, min_tiles=1024, tile_bytes=512 << 10)
    assert np.array_equal(plan.export("tiles"), asked.export("tiles"))


def test_large_workgroups_take_the_tuned_bound():
    # 40 block rows of 4 MB for 512 workgroups: 437,500-byte tiles, ten a block row
    assert _plan(40, 100, 100, 100, wg=1024).stats["ntiles"] == 40 * 10


def test_one_workgroup_per_cu_counts_as_two():
    # 157 spans of 40,000 rows of 240 entries, 38.4 MB: three tiles each for
    # 512 workgroups, two for 256
    assert _plan(40000, 1, 40, 6, wg=512, unroll=8).stats["ntiles"] == 469
