"""The FP32 SpMM kernel's tasks at the sizes where they can go wrong (marked
gpu): tile heights around the 16- and 32-row fragments, RHS widths around the
16-, 32- and 64-column groups, column ranges that end inside a step, dense
and sparse pieces in one tile, tiles without dense pieces, empty block rows
and infinities.

The tolerance is the kernel's own bound: K products of FP32 values summed in
FP32 differ from the exact sum by at most about K * 2^-24 of sum |a||x|; the
widest row here has 400 stored columns, so 400 * 2^-24 = 2.4e-5 covers the
worst case and the usual bar of 1e-5 the observed one."""
import numpy as np
import pytest

from oracle import c_oracle
from sable_amd.convert import ROUTE_DENSE, ROUTE_SPARSE, ROUTE_DENSE_MFMA
from sable_amd.vbr import VBR

pytestmark = pytest.mark.gpu

TOL = 1e-5


@pytest.fixture(scope="module")
def rt():
    from sable_amd import runtime
    runtime.init()
    return runtime


def _matrix(heights, widths, seed, empty=()):
    """Every block stored (but those of the block rows in ``empty``), half of
    its values zero."""
    rng = np.random.default_rng(seed)
    rows = [i for i in range(len(heights)) if i not in empty]
    size = [heights[i] * w for i in rows for w in widths]
    val = rng.standard_normal(sum(size)).astype(np.float32)
    val[rng.random(len(val)) < 0.5] = 0
    n = len(widths)
    begin = [-1 if i in empty else rows.index(i) * n for i in range(len(heights))]
    return VBR(val, np.concatenate([[0], np.cumsum(size)]).astype(np.int64),
               np.tile(np.arange(n), len(rows)).astype(np.int64),
               np.concatenate([[0], np.cumsum(heights)]).astype(np.int64),
               np.concatenate([[0], np.cumsum(widths)]).astype(np.int64), np.asarray(begin, np.int64),
               np.asarray([b if b < 0 else b + n for b in begin], np.int64))


def _check(vbr, X, Y):
    Y64, AY = c_oracle.spmm_f64_dense_blocks(vbr.val, vbr.indx, vbr.bindx, vbr.rpntr, vbr.cpntr, vbr.bpntrb,
                                             vbr.bpntre, X)
    assert c_oracle.scaled_error(Y.ravel(), Y64.ravel(), AY.ravel())["componentwise"] <= TOL


HEIGHTS = [1, 15, 16, 17, 31, 32, 33, 64, 3, 127, 128, 129, 200]
WIDTHS = [1, 7, 8, 9, 23, 24, 25, 100, 3, 200]


@pytest.mark.parametrize("use_rtc", [True, False])
@pytest.mark.parametrize("n_rhs", [4, 12, 16, 20, 32, 36, 60, 64, 68, 96, 100, 128, 132, 512])
def test_fragment_edges(rt, n_rhs, use_rtc):
    vbr = _matrix(HEIGHTS, WIDTHS, n_rhs, empty=(8,))
    rng = np.random.default_rng(n_rhs)
    X = rng.uniform(-1, 1, (int(vbr.cpntr[-1]), n_rhs)).astype(np.float32)
    nb = len(vbr.bindx)
    mixed = rng.choice([ROUTE_DENSE, ROUTE_SPARSE], nb)
    mixed[: 2 * len(WIDTHS)] = ROUTE_SPARSE               # two block rows without dense pieces
    for name, routes in (("dense", np.full(nb, ROUTE_DENSE)), ("sparse", np.full(nb, ROUTE_SPARSE)), ("mixed", mixed)):
        print(f"case: n={n_rhs} {name} rtc={use_rtc}", flush=True)
        plan = rt.Plan.from_vbr(vbr, routes.astype(np.uint8), op="spmm", n_rhs=n_rhs, wg=256, use_rtc=use_rtc)
        _check(vbr, X, plan.spmm(X))


@pytest.mark.parametrize("n_rhs", [16, 128])
def test_many_and_few_wavefronts(rt, n_rhs):
    """Both row counts per wavefront: a plan whose tiles leave the device's
    SIMDs empty takes 16 rows per wavefront, one that fills them 32."""
    for copies in (1, 150):
        vbr = _matrix([40, 97, 128] * copies, [5, 30, 61], copies)
        X = np.random.default_rng(3).uniform(-1, 1, (int(vbr.cpntr[-1]), n_rhs)).astype(np.float32)
        print(f"case: {copies} copies n={n_rhs}", flush=True)
        _check(vbr, X, rt.Plan.from_vbr(vbr, None, op="spmm", n_rhs=n_rhs).spmm(X))


@pytest.mark.parametrize("n_rhs", [16, 64])
@pytest.mark.parametrize("route", [ROUTE_DENSE, ROUTE_SPARSE])
def test_infinities_stay_in_their_rows(rt, n_rhs, route):
    """An infinity in X reaches exactly the rows whose products meet it: with
    the sparse route those with a nonzero there, with the dense route every
    row of the block (0 * inf is NaN), and no other block row, column or
    fragment padding."""
    vbr = _matrix([5, 33, 18], [6, 11, 9], 5)
    routes = np.full(len(vbr.bindx), route, np.uint8)
    if route == ROUTE_DENSE:
        routes[0] = ROUTE_SPARSE                           # block row 0: one sparse block among dense ones
    X = np.ones((26, n_rhs), np.float32)
    X[2, 1] = np.inf
    X[25, 3] = -np.inf                                     # the last column of the last step
    A = np.zeros((56, 26))
    for a in range(3):
        for k in range(vbr.bpntrb[a], vbr.bpntre[a]):
            c0, c1 = vbr.cpntr[vbr.bindx[k]], vbr.cpntr[vbr.bindx[k] + 1]
            r0, r1 = vbr.rpntr[a], vbr.rpntr[a + 1]
            blk = vbr.val[vbr.indx[k]:vbr.indx[k + 1]].reshape(c1 - c0, r1 - r0).T.astype(np.float64)
            if routes[k] == ROUTE_SPARSE:
                blk[blk == 0] = np.nan                     # not an entry: no product
            A[r0:r1, c0:c1] = blk
    with np.errstate(invalid="ignore"):
        P = A[:, :, None] * X[None].astype(np.float64)
    P[np.isnan(A)] = 0
    ref = P.sum(axis=1)
    print(f"case: infinities n={n_rhs} route={route}", flush=True)
    Y = rt.Plan.from_vbr(vbr, routes, op="spmm", n_rhs=n_rhs).spmm(X)
    assert np.array_equal(np.isnan(Y), np.isnan(ref))
    assert np.array_equal(np.isposinf(Y), np.isposinf(ref)) and np.array_equal(np.isneginf(Y), np.isneginf(ref))
    ok = np.isfinite(ref)
    assert np.max(np.abs(Y[ok] - ref[ok]) / np.maximum(np.abs(P).sum(axis=1)[ok], 1e-30)) <= TOL


def test_group_of_all_kinds(rt):
    """A group whose members take different routes gives the bits of their own
    launches."""
    rng = np.random.default_rng(8)
    plans, xs, ys, ref = [], [], [], []
    for k, routes in enumerate(([ROUTE_DENSE], [ROUTE_SPARSE], [ROUTE_DENSE, ROUTE_SPARSE, ROUTE_DENSE_MFMA])):
        vbr = _matrix(HEIGHTS[k:], WIDTHS, 40 + k, empty=(1,))
        X = rng.uniform(-1, 1, (int(vbr.cpntr[-1]), 32)).astype(np.float32)
        plan = rt.Plan.from_vbr(vbr, rng.choice(routes, len(vbr.bindx)).astype(np.uint8), op="spmm", n_rhs=32,
                                min_tiles=1)
        plans.append(plan)
        xs.append(rt.DeviceArray.from_numpy(X))
        ys.append(rt.DeviceArray((plan.nrows, 32)))
        ref.append(plan.spmm(X))
    print("case: group of three routings", flush=True)
    g = rt.Group(plans, xs, ys)
    for _ in range(2):
        g.launch()
        for y, r in zip(ys, ref):
            assert np.array_equal(y.numpy(), r)
