"""FP32 SpMM: a sparse-routed row multiplies its own values and no others
(marked gpu).  Infinities and NaN among the values of one row, next to empty
rows, shorter rows and rows that end a batch of entries; trailing empty rows,
behind whose piece the value array ends.

Every value is a power of two or not finite and X is 1, 2 or 4, so the finite
sums are exact and the results are compared for equality."""
import numpy as np
import pytest

from sable_amd.convert import ROUTE_DENSE, ROUTE_DENSE_MFMA, ROUTE_SPARSE
from sable_amd.vbr import VBR

pytestmark = pytest.mark.gpu

# entries per row of the sparse block: around the batches of 4 and 16 entries
# and the four and eight in flight
COUNTS = [1, 0, 1, 2, 3, 0, 4, 5, 0, 15, 16, 17, 0, 33, 8, 7, 0, 40, 1, 0, 0]
WIDTHS = [48, 9]


@pytest.fixture(scope="module")
def rt():
    from sable_amd import runtime
    runtime.init()
    return runtime


def _matrix(special):
    """Two block rows of two blocks: columns 0..47 hold COUNTS entries per row
    (the last one of every row in ``special`` not finite), the rest is full."""
    rng = np.random.default_rng(6)
    h = len(COUNTS)
    blocks = []
    for a in range(2):
        S = np.zeros((h, WIDTHS[0]), np.float32)
        for r, c in enumerate(COUNTS):
            cols = np.sort(rng.choice(WIDTHS[0], c, replace=False))
            S[r, cols] = 2.0 ** rng.integers(-3, 4, c)
            if c and (a, r) in special:
                S[r, cols[-1 if special[a, r][0] else 0]] = special[a, r][1]
        blocks += [S, (2.0 ** rng.integers(-3, 4, (h, WIDTHS[1]))).astype(np.float32)]
    size = [b.size for b in blocks]
    vbr = VBR(np.concatenate([b.T.ravel() for b in blocks]), np.concatenate([[0], np.cumsum(size)]).astype(np.int64),
              np.asarray([0, 1, 0, 1], np.int64), np.asarray([0, h, 2 * h], np.int64),
              np.asarray([0, WIDTHS[0], sum(WIDTHS)], np.int64), np.asarray([0, 2], np.int64),
              np.asarray([2, 4], np.int64))
    return vbr, np.block([blocks[:2], blocks[2:]])


def _expect(A, X):
    """Sums over the entries alone (a zero of A is no entry; the full block
    has none)."""
    out = np.zeros((A.shape[0], X.shape[1]), np.float32)
    for r in range(A.shape[0]):
        c = np.flatnonzero(A[r])
        out[r] = (A[r, c, None].astype(np.float64) * X[c]).sum(axis=0)
    return out


# where: the last entry of its row (repeated by lanes past the row's end) or
# the first (read by the empty row before it)
SPECIAL = {(0, 0): (True, np.inf), (0, 2): (False, np.inf), (0, 4): (True, np.nan), (0, 6): (False, -np.inf),
           (0, 9): (True, np.inf), (0, 13): (False, np.nan), (0, 17): (True, -np.inf), (1, 0): (False, np.nan),
           (1, 10): (True, np.inf), (1, 18): (True, np.nan)}


@pytest.mark.parametrize("use_rtc", [True, False])
@pytest.mark.parametrize("n_rhs", [4, 16, 32, 64, 128, 512])
@pytest.mark.parametrize("full", [ROUTE_SPARSE, ROUTE_DENSE, ROUTE_DENSE_MFMA])
def test_values_stay_in_their_rows(rt, full, n_rhs, use_rtc):
    if full == ROUTE_DENSE_MFMA and (n_rhs % 16 or n_rhs > 256):
        full = ROUTE_DENSE
    rng = np.random.default_rng(n_rhs)
    X = (2.0 ** rng.integers(0, 3, (sum(WIDTHS), n_rhs))).astype(np.float32)
    routes = np.asarray([ROUTE_SPARSE, full] * 2, np.uint8)
    for special in ({}, SPECIAL):
        vbr, A = _matrix(special)
        print(f"case: full={full} n={n_rhs} rtc={use_rtc} special={len(special)}", flush=True)
        # memory that the plan's arrays may take over holds NaN words
        poison = [rt.DeviceArray.from_numpy(np.full(k, -1, np.int32)) for k in (64, 256, 512, 1024, 4096) for _ in range(8)]
        for p in poison:
            p.free()
        Y = rt.Plan.from_vbr(vbr, routes, op="spmm", n_rhs=n_rhs, wg=256, use_rtc=use_rtc).spmm(X)
        assert np.array_equal(Y, _expect(A, X), equal_nan=True)


@pytest.mark.parametrize("n_rhs", [16, 64])
def test_values_stay_in_their_member(rt, n_rhs):
    """The same in a group, whose members' arrays are their own."""
    X = np.full((sum(WIDTHS), n_rhs), 2.0, np.float32)
    plans, xs, ys, ref = [], [], [], []
    for special in ({}, SPECIAL):
        vbr, A = _matrix(special)
        plans.append(rt.Plan.from_vbr(vbr, np.full(4, ROUTE_SPARSE, np.uint8), op="spmm", n_rhs=n_rhs, min_tiles=1))
        xs.append(rt.DeviceArray.from_numpy(X))
        ys.append(rt.DeviceArray((plans[-1].nrows, n_rhs)))
        ref.append(_expect(A, X))
    print(f"case: group n={n_rhs}", flush=True)
    rt.Group(plans, xs, ys).launch()
    for y, r in zip(ys, ref):
        assert np.array_equal(y.numpy(), r, equal_nan=True)
