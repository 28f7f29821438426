"""The algorithmic bytes of a plan are those of the arrays its kernels read:
in SpMM 8 per sparse entry (value and X row) and the FP32 kernel's tasks."""
import numpy as np
import pytest

from sable_amd import synth
from sable_amd.convert import ROUTE_DENSE, ROUTE_DENSE_MFMA, ROUTE_SPARSE
from sable_amd.runtime import Plan

TILE, PIECE, RANGE, TASK, XCDS = 64, 48, 8, 40, 8


def _plan(kinds, host_only=True, **kw):
    vbr, _, _ = synth.mixed_vbr(900, 12, 10, 150, 0.4, 0.5, (0.8, 1.0), (0.05, 0.3), seed=5)
    routes = np.random.default_rng(5).choice(kinds, len(vbr.bindx)).astype(np.uint8)
    return Plan.from_vbr(vbr, routes, host_only=host_only, **kw)


@pytest.mark.parametrize("kinds", [[ROUTE_SPARSE], [ROUTE_DENSE], [ROUTE_DENSE_MFMA], [ROUTE_DENSE, ROUTE_SPARSE],
                                   [ROUTE_DENSE, ROUTE_SPARSE, ROUTE_DENSE_MFMA]])
@pytest.mark.parametrize("n_rhs", [16, 128])
def test_spmm(kinds, n_rhs):
    s = _plan(kinds, op="spmm", n_rhs=n_rhs).stats
    tasks = s["descriptor_bytes"] - TILE * s["ntiles_mfma"] - PIECE * s["npieces"] - RANGE * s["nxranges"]
    assert tasks % (TASK * XCDS) == 0 and (tasks > 0) == (s["ntiles"] > s["ntiles_mfma"])
    assert s["bytes_alg"] == (4 * (s["dense_values"] + s["mfma_values"] + s["rowptr_entries"]) + 8 * s["sparse_nnz"]
                              + s["descriptor_bytes"] + 4 * n_rhs * (s["nrows"] + s["ncols"]))


def test_spmv():
    s = _plan([ROUTE_DENSE, ROUTE_SPARSE]).stats
    assert s["descriptor_bytes"] == TILE * s["ntiles"] + PIECE * s["npieces"] + 4 * s["xmap_entries"]
    assert s["bytes_alg"] == (4 * (s["dense_values"] + s["rowptr_entries"]) + 6 * s["sparse_nnz"]
                              + s["descriptor_bytes"] + 4 * (s["nrows"] + s["ncols"]))


@pytest.mark.gpu
@pytest.mark.parametrize("op,n_rhs", [("spmv", 1), ("spmm", 16)])
def test_device_plan(op, n_rhs):
    """A device plan exports what the host plan does, and holds what its
    kernels read: no local columns in SpMM."""
    kinds = [ROUTE_DENSE, ROUTE_SPARSE]
    host, dev = _plan(kinds, op=op, n_rhs=n_rhs), _plan(kinds, host_only=False, op=op, n_rhs=n_rhs)
    for name in Plan._EXPORT:
        assert np.array_equal(host.export(name), dev.export(name)), name
    s = dev.stats
    held = 4 * (s["dense_padded"] + s["sparse_padded"] + s["rowptr_entries"]) + TILE * s["ntiles"] \
        + PIECE * s["npieces"] + RANGE * s["nxranges"]
    if op == "spmm":
        held += 4 * s["sparse_padded"] + s["descriptor_bytes"] - PIECE * s["npieces"] - RANGE * s["nxranges"]
    else:
        held += 2 * s["sparse_padded"] + 4 * s["xmap_entries"]
    assert s["device_bytes"] == held
