"""The tile target of SpMV plans on their own, where the first target gives
more tiles than the device holds at once (768 workgroups of 512 threads), and
what building a plan costs."""
import subprocess
import sys
import time

import numpy as np
import pytest

from conftest import ROOT
from sable_amd import synth
from sable_amd.runtime import Plan

HEIGHT, WIDTH = 40, 400


def _uniform(n, height=HEIGHT, val=None, **kw):
    """n block rows of one height x WIDTH block each."""
    if val is None:
        val = np.random.default_rng(n).standard_normal(n * height * WIDTH).astype(np.float32)
    return Plan(val, np.arange(n + 1) * height * WIDTH, np.zeros(n, np.int64), np.arange(n + 1) * height, [0, WIDTH],
                np.arange(n), np.arange(n) + 1, host_only=True, **kw), val


# n equal block rows of W bytes: the targets are f * n * W / 768 for f = 1.4,
# 1.6, 1.9, 2.2, and a block row is one tile from a target of W on, two from
# W / 2 on.  530 fit at 1.6, 450 at 1.9, 360 at 2.2; 700 fit at 1.4, 770 never
@pytest.mark.parametrize("n,ntiles", [(360, 720), (385, 385), (450, 450), (530, 530), (700, 700), (770, 770)])
def test_larger_targets(n, ntiles):
    plan, val = _uniform(n, wg=512, unroll=2, tile_bytes=512 << 10)
    assert plan.stats["ntiles"] == ntiles
    tiles, pieces, dval = plan.export("tiles"), plan.export("pieces"), plan.export("dval")
    A = val.reshape(n, WIDTH, HEIGHT)
    rows = np.zeros(n * HEIGHT, np.int64)
    for t in tiles:                                     # the plan holds the matrix
        a, r = divmod(int(t["row0"]), HEIGHT)
        p = pieces[t["piece_begin"]]
        assert t["piece_end"] == t["piece_begin"] + 1 and p["ncols"] == WIDTH
        panel = dval[p["data_off"]:p["data_off"] + WIDTH * t["nrows"]].reshape(WIDTH, t["nrows"])
        assert np.array_equal(panel, A[a, :, r:r + t["nrows"]])
        rows[t["row0"]:t["row0"] + t["nrows"]] += 1
    assert np.all(rows == 1)


def test_a_plan_is_held_once():
    """Host memory of a plan that takes a larger target: one plan's arrays and
    their growth, not two plans'."""
    code = (f"import sys\nsys.path[:0] = [{ROOT!r}, {ROOT + '/tests'!r}]\n"
            "import numpy as np\nfrom test_plan_ladder import _uniform\n"
            "def rss():\n"
            "    return 1024 * int(next(s for s in open('/proc/self/status') if s.startswith('VmHWM')).split()[1])\n"
            "val = np.ones(450 * 160 * 400, np.float32)\nbefore = rss()\n"
            "plan, _ = _uniform(450, 160, val, wg=512, unroll=2, tile_bytes=512 << 10)\n"
            "print(plan.stats['ntiles'], (rss() - before) / val.nbytes)\n")
    out = subprocess.run([sys.executable, "-c", code], capture_output=True, text=True, timeout=120, check=True).stdout
    ntiles, times = out.split()
    assert int(ntiles) <= 768 and float(times) < 2.4


def test_spmm_without_mfma_is_built_once():
    """The tiles of such a plan do not follow tile_bytes: no number of tiles
    asked for builds it again."""
    vbr, _, _ = synth.mixed_vbr(4000, 60, 30, 120, 0.3, 0.5, (0.8, 1.0), (0.05, 0.3), seed=2)

    def build(min_tiles):
        best = []
        for _ in range(3):
            t = time.process_time()
            plan = Plan.from_vbr(vbr, None, op="spmm", n_rhs=64, min_tiles=min_tiles, host_only=True)
            best.append(time.process_time() - t)
        return min(best), plan.export("tiles")

    once, tiles = build(1)
    asked, same = build(1 << 20)
    assert np.array_equal(tiles, same) and asked < 2.5 * once
