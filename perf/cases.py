"""The workloads this framework is timed on, through its public entry points.

Six kinds of work:

* ``spmv``   y = A x with a kept plan: device arrays, or numpy arrays in and
  out (``host``), as a program that has no device buffers calls it;
* ``spmm``   Y = A X with a kept plan, the dense blocks on the FP32 path, on
  MFMA with the exact three-term bf16 split (``bf16x6``) or with the hi+lo
  split (``bf16x3``);
* ``batch``  many matrices in one kept group, SpMV and SpMM of each;
* ``train``  a training step of the block router: forward, masked MSE
  gradient, backward, Adam;
* ``convert`` a SciPy matrix to partitioned, compressed VBR arrays on the GPU
  (``cut_indices2`` then ``sparse_to_vbrc_device``).

Matrices follow the laws of this repository's generators (``synth.py``):
``cuts`` partitions are drawn from uniform cut points (the reference's law,
so parts may be one row wide), ``bounded`` ones from sizes in [smin, smax].
``mix`` is the stored blocks' density: ``full`` all 1, ``half`` half of them
0.8-1.0 and half 0.01-0.2, ``mostly`` 70 % of them 0.9-1.0 and 30 % 0.02-0.1.
Values are N(0, 1), x and X uniform in [-1, 1].
"""
import numpy as np
import torch  # before the library: both then share one ROCm runtime

from sable_amd import autopartition, convert, runtime
from sable_amd.router import mlp
from sable_amd.router.router import Router

_MIX = {  # share of the denser class, its density range, the other class's
    "full": (1.0, (1.0, 1.0), (1.0, 1.0)),
    "half": (0.5, (0.8, 1.0), (0.01, 0.2)),
    "mostly": (0.7, (0.9, 1.0), (0.02, 0.1)),
}


def _matrix(m, n, rparts, cparts, smin, smax, frac, mix):
    """The fields that describe a matrix: m x n, its partition and blocks."""
    return dict(m=m, n=n, rparts=rparts, cparts=cparts, smin=smin, smax=smax, frac=frac, mix=mix)


def listed():
    return [
        # the smallest use: the reference's own 1,000-row synthetic (20 x 20
        # cut points, 10 % of the blocks, all dense); one call's latency
        dict(name="spmv_1k", kind="spmv", routes="dense", host=False, **_matrix(1000, 1000, 20, 20, 0, 0, 0.1, "full")),
        # a program that holds numpy arrays: x goes in and y comes out of host
        # memory on every call; odd sizes
        dict(name="spmv_20k_numpy", kind="spmv", routes="threshold", host=True,
             **_matrix(20011, 20011, 203, 203, 20, 200, 0.01, "half")),
        # ragged and rectangular: block rows of 8 to 75 rows
        dict(name="spmv_30k_short", kind="spmv", routes="threshold", host=False,
             **_matrix(30011, 27001, 800, 700, 8, 75, 0.01, "half")),
        # an ordinary matrix, its blocks routed by the trained router
        dict(name="spmv_40k_learned", kind="spmv", routes="learned", host=False,
             **_matrix(40000, 40000, 400, 400, 20, 200, 0.01, "half")),
        # the largest: the 100,000-row matrix of the repository's benchmark
        dict(name="spmv_100k", kind="spmv", routes="threshold", host=False,
             **_matrix(100000, 100000, 1000, 1000, 20, 200, 0.01, "half")),
        # the generated SpMM program's default: N = 512 on the FP32 path
        dict(name="spmm_3k_n512", kind="spmm", n_rhs=512, precision="fp32",
             **_matrix(3001, 3001, 30, 30, 20, 200, 0.1, "half")),
        # the 50,000-row SpMM of the benchmark at N = 128, FP32 path
        dict(name="spmm_50k_n128_fp32", kind="spmm", n_rhs=128, precision="fp32",
             **_matrix(50000, 50000, 500, 500, 32, 192, 0.02, "mostly")),
        # the same with its dense blocks on MFMA at FP32-level accuracy
        dict(name="spmm_50k_n128", kind="spmm", n_rhs=128, precision="bf16x6",
             **_matrix(50000, 50000, 500, 500, 32, 192, 0.02, "mostly")),
        # a narrow right-hand side (block solvers), ragged partition
        dict(name="spmm_20k_n16", kind="spmm", n_rhs=16, precision="bf16x6",
             **_matrix(20011, 20011, 203, 203, 20, 200, 0.02, "half")),
        # a matrix set served together: SpMV and SpMM at N = 16 of each
        dict(name="batch_16", kind="batch", count=16, n_rhs=16, nlo=2000, nhi=32000, plo=50, phi=400),
        # training the router on a mini-batch of measured blocks
        dict(name="train_4096", kind="train", batch=4096),
        # from a SciPy matrix to the compressed arrays a plan is built from
        dict(name="convert_6k", kind="convert", threshold=0.2, **_matrix(6007, 6007, 60, 60, 20, 200, 0.1, "half")),
    ]


def _log(rng, lo, hi):
    return int(round(lo * (hi / lo) ** rng.random()))


def _drawn_matrix(rng, nlo, nhi, frac, stored):
    """A square or rectangular matrix of nlo..nhi rows whose stored blocks
    hold about ``stored`` values at most."""
    m = _log(rng, nlo, nhi)
    n = m if rng.random() < 0.6 else max(nlo, int(m * rng.uniform(0.6, 1.0)))
    mean = rng.choice((30, 60, 100, 110))
    rp, cp = max(4, m // mean), max(4, n // mean)
    frac = min(max(frac, 16.0 / (rp * cp)), stored / (m * n))
    if m <= 4000 and rng.random() < 0.5:
        return _matrix(m, n, rp, cp, 0, 0, frac, rng.choice(("full", "half")))
    return _matrix(m, n, rp, cp, max(1, mean // 5), 2 * mean, frac, rng.choice(("half", "mostly")))


def draw(rng):
    kind = rng.choice(("spmv", "spmv", "spmv", "spmm", "spmm", "spmm", "batch", "train", "convert"))
    if kind == "spmv":
        case = dict(kind=kind, host=rng.random() < 0.25, **_drawn_matrix(rng, 1000, 90000, 0.01, 80e6))
        routes = ("threshold", "dense", "learned") if case["m"] * case["n"] * case["frac"] < 20e6 else ("threshold",)
        return dict(case, routes=rng.choice(routes))
    if kind == "spmm":
        precision = rng.choice(("fp32", "bf16x6", "bf16x6", "bf16x3"))
        n_rhs = rng.choice((4, 8, 16, 20, 32, 64, 72, 128, 256, 512) if precision == "fp32" else (16, 32, 64, 128, 256))
        # at most the 50k SpMM's products: 50e6 stored values times N = 128
        stored = min(40e6, 5e9 / n_rhs)
        return dict(kind=kind, n_rhs=n_rhs, precision=precision, **_drawn_matrix(rng, 1000, 45000, 0.02, stored))
    if kind == "batch":
        nhi = _log(rng, 6000, 24000)
        return dict(kind=kind, count=rng.randint(3, 16), n_rhs=rng.choice((16, 32)), nlo=2000, nhi=nhi,
                    plo=50, phi=rng.choice((200, 300, 400)))
    if kind == "train":
        return dict(kind=kind, batch=_log(rng, 256, 4096))
    return dict(kind=kind, threshold=0.2, **_drawn_matrix(rng, 1000, 6000, 0.1, 4e6))


# ---- matrices --------------------------------------------------------------

def _sizes(g, total, parts, smin, smax):
    """Partition sizes summing to total: uniform cut points (smin 0), else
    sizes in [smin, smax]."""
    if not smin:
        cuts = np.sort(g.choice(np.arange(1, total), parts - 1, replace=False))
        return np.diff(np.concatenate([[0], cuts, [total]])).astype(np.int64)
    s = g.integers(smin, smax + 1, parts).astype(np.float64)
    s = np.clip(np.floor(smin + (s - smin) * (total - parts * smin) / max(float((s - smin).sum()), 1.0)), smin, smax)
    s = s.astype(np.int64)
    while s.sum() != total:
        step = 1 if s.sum() < total else -1
        room = np.nonzero(s < smax if step > 0 else s > smin)[0]
        s[g.choice(room, min(len(room), abs(int(total - s.sum()))), replace=False)] += step
    return s


def _arrays(case, seed, pattern=None):
    """The VBR arrays (host, FP32 values) of a case's matrix; ``pattern``
    seeds its partition, blocks and zeros (default: ``seed``)."""
    pattern = seed if pattern is None else pattern
    g = np.random.Generator(np.random.PCG64([pattern, 11]))
    h = _sizes(g, case["m"], case["rparts"], case["smin"], case["smax"])
    w = _sizes(g, case["n"], case["cparts"], case["smin"], case["smax"])
    total = len(h) * len(w)
    chosen = np.sort(g.choice(total, max(1, int(round(case["frac"] * total))), replace=False))
    br, bc = chosen // len(w), chosen % len(w)
    size = h[br] * w[bc]
    indx = np.concatenate([[0], np.cumsum(size)]).astype(np.int64)
    share, hi, lo = _MIX[case["mix"]]
    first = g.random(len(size)) < share
    density = np.where(first, g.uniform(*hi, len(size)), g.uniform(*lo, len(size)))
    stored = int(indx[-1])
    val = torch.randn(stored, generator=torch.Generator("cuda").manual_seed(seed), device="cuda")
    if case["mix"] != "full":
        d = torch.repeat_interleave(torch.from_numpy(density.astype(np.float32)).cuda(),
                                    torch.from_numpy(size).cuda())
        val *= torch.rand(stored, generator=torch.Generator("cuda").manual_seed(pattern + 1), device="cuda") < d
    count = np.bincount(br, minlength=len(h))
    end = np.cumsum(count)
    return dict(val=val.cpu().numpy(), indx=indx, bindx=bc.astype(np.int64),
                rpntr=np.concatenate([[0], np.cumsum(h)]).astype(np.int64),
                cpntr=np.concatenate([[0], np.cumsum(w)]).astype(np.int64),
                bpntrb=np.where(count > 0, end - count, -1).astype(np.int64),
                bpntre=np.where(count > 0, end, -1).astype(np.int64))


def _rhs(case, seed, n_rhs):
    g = np.random.Generator(np.random.PCG64([seed, 12]))
    shape = (case["n"],) if n_rhs == 1 else (case["n"], n_rhs)
    return g.random(shape, dtype=np.float32) * np.float32(2) - np.float32(1)


def _members(case, seed):
    """The matrices of a batch: rows log-uniform, partition counts uniform,
    1 % of the blocks, parts of a fifth to twice the mean size.  The sizes
    are the case's own; the seed sets the values, as in a served set."""
    g = np.random.Generator(np.random.PCG64([case["count"], case["nhi"], case["phi"]]))
    out = []
    for i in range(case["count"]):
        n = _log(g, case["nlo"], case["nhi"])
        p = int(g.integers(case["plo"], case["phi"] + 1))
        lo = max(1, -(-n // (5 * p)))
        out.append((_matrix(n, n, p, p, lo, max(lo + 1, 2 * n // p), 0.01, "half"), seed * 1009 + i))
    return out


class _Device:
    """A device array of the framework, seen by torch without a copy."""

    def __init__(self, a):
        self.owner = a
        self.__cuda_array_interface__ = dict(shape=a.shape, typestr="<f4", data=(a.ptr, False), version=2)


def _seen(a):
    return torch.as_tensor(_Device(a), device="cuda")


# ---- states and passes -----------------------------------------------------

def _spmm_routes(a, precision):
    r = convert.threshold_routes(a["val"], a["indx"], convert.DEFAULT_DENSITY)
    if precision == "fp32":
        return r
    return np.where(r == convert.ROUTE_DENSE, convert.ROUTE_DENSE_MFMA, r).astype(np.uint8)


def prepare(case, seed):
    if case["kind"] == "spmv":
        a = _arrays(case, seed)
        if case["routes"] == "learned":
            routes = Router.load().route_blocks(**a)
        elif case["routes"] == "threshold":
            routes = convert.threshold_routes(a["val"], a["indx"], convert.DEFAULT_DENSITY)
        else:
            routes = None
        plan = runtime.Plan(**a, routes=routes)
        x = _rhs(case, seed, 1)
        if case["host"]:
            return dict(plan=plan, x=x)
        y = runtime.DeviceArray(plan.nrows)
        return dict(plan=plan, x=runtime.DeviceArray.from_numpy(x), y=y, out=_seen(y))
    if case["kind"] == "spmm":
        a = _arrays(case, seed)
        plan = runtime.Plan(**a, routes=_spmm_routes(a, case["precision"]), op="spmm", n_rhs=case["n_rhs"],
                            mfma_split=2 if case["precision"] == "bf16x3" else 3)
        y = runtime.DeviceArray((plan.nrows, case["n_rhs"]))
        return dict(plan=plan, x=runtime.DeviceArray.from_numpy(_rhs(case, seed, case["n_rhs"])), y=y, out=_seen(y))
    if case["kind"] == "batch":
        plans, xs, ys = [], [], []
        for c, s in _members(case, seed):
            a = _arrays(c, s)
            # the options the benchmark's batch gives its members
            r = convert.threshold_routes(a["val"], a["indx"], convert.DEFAULT_DENSITY)
            plans.append(runtime.Plan(**a, routes=r, wg=256, min_tiles=1))
            plans.append(runtime.Plan(**a, routes=_spmm_routes(a, "bf16x6"), op="spmm", n_rhs=case["n_rhs"], wg=128,
                                      min_tiles=1))
            xs += [runtime.DeviceArray.from_numpy(_rhs(c, s, 1)),
                   runtime.DeviceArray.from_numpy(_rhs(c, s, case["n_rhs"]))]
            ys += [runtime.DeviceArray(c["m"]), runtime.DeviceArray((c["m"], case["n_rhs"]))]
        return dict(group=runtime.Group(plans, xs, ys), keep=(plans, xs, ys), out=[_seen(y) for y in ys])
    if case["kind"] == "train":
        z, t, mask, p = _samples(case, seed)
        net = mlp.DeviceMLP(p)
        dev = [runtime.DeviceArray.from_numpy(v) for v in (z, t, mask)]
        return dict(net=net, dev=dev, n=case["batch"], scale=1.0 / float(mask.sum()), grad=_seen(net.g))
    # partitioned by its pattern (products of signed values would cancel),
    # which is the case's own; the seed sets the values
    A = convert.vbr_to_csc(**_arrays(case, seed, case["m"]))
    P = A.copy()
    P.data[:] = 1.0
    return dict(A=A, P=P, threshold=case["threshold"])


def run(state):
    if "group" in state:
        state["group"].launch()
        return state["out"]
    if "net" in state:
        net = state["net"]
        out = net.gradient(*state["dev"], state["n"], state["scale"])
        net.adam()
        return dict(out=_seen(out), grad=state["grad"])
    if "A" in state:
        cols, rows = autopartition.cut_indices2(state["P"], state["threshold"], autopartition.similarity2, device=True)
        rp, cp = np.asarray(rows, dtype=np.int64), np.asarray(cols, dtype=np.int64)
        return (rp, cp) + tuple(convert.sparse_to_vbrc_device(state["A"], rp, cp))
    call = state["plan"].spmm if state["plan"].op == "spmm" else state["plan"].spmv
    if "y" not in state:
        return call(state["x"])
    call(state["x"], state["y"])
    return state["out"]


def _samples(case, seed):
    """A mini-batch of standardised block features, log2 costs and the mask
    of the measured outputs, and the network's parameters."""
    g = np.random.Generator(np.random.PCG64([seed, 13]))
    n = case["batch"]
    z = g.standard_normal((n, mlp.N_FEATURES), dtype=np.float32)
    t = (g.standard_normal((n, mlp.N_OUT), dtype=np.float32) * 2 + 8).astype(np.float32)
    mask = (g.random((n, mlp.N_OUT)) < 0.8).astype(np.float32)
    return z, t, mask, mlp.init_params(seed)


# ---- what a pass cannot do without, and its result in 64 bits ----------------

def _counts(c):
    """Expected stored nonzeros of the denser and the sparser class."""
    stored = c["frac"] * c["m"] * c["n"]
    share, hi, lo = _MIX[c["mix"]]
    return stored * share * sum(hi) / 2, stored * (1 - share) * sum(lo) / 2


def _product(c, n_rhs):
    """Bytes (4 per nonzero, 2 more for the column of a sparse block's one; x
    and y once) and flops of one product."""
    d, s = _counts(c)
    return 4 * d + 6 * s + 4 * n_rhs * (c["m"] + c["n"]), 2 * (d + s) * n_rhs


def work(case):
    if case["kind"] in ("spmv", "spmm"):
        b, f = _product(case, case.get("n_rhs", 1))
    elif case["kind"] == "batch":
        each = [_product(c, n) for c, _ in _members(case, 0) for n in (1, case["n_rhs"])]
        b, f = sum(e[0] for e in each), sum(e[1] for e in each)
    elif case["kind"] == "train":
        n, p = case["batch"], mlp.n_params()
        # features, targets, mask in, outputs out; parameters, their two
        # moments read and written and the gradient written
        b = 4 * n * (mlp.N_FEATURES + 3 * mlp.N_OUT) + 4 * 7 * p
        f = 6 * n * p
    else:
        # the CSC matrix read for each axis and for the blocks, the
        # compressed values written
        nnz = sum(_counts(case))
        b, f = 3 * 12 * nnz + 8 * case["frac"] * case["m"] * case["n"], 6 * nnz
    return {"bytes": b, "flops": f}


def _exact_product(a, x):
    """A x in 64 bits, block by block."""
    xd = torch.from_numpy(x.astype(np.float64)).cuda().reshape(len(x), -1)
    val = torch.from_numpy(a["val"]).cuda()
    y = torch.zeros(int(a["rpntr"][-1]), xd.shape[1], dtype=torch.float64, device="cuda")
    rp, cp, ix, bx = (a[k].tolist() for k in ("rpntr", "cpntr", "indx", "bindx"))
    for i, (b, e) in enumerate(zip(a["bpntrb"].tolist(), a["bpntre"].tolist())):
        for k in range(max(b, 0), max(e, 0)):
            c0, c1 = cp[bx[k]], cp[bx[k] + 1]
            block = val[ix[k]:ix[k + 1]].double().reshape(c1 - c0, rp[i + 1] - rp[i])
            y[rp[i]:rp[i + 1]] += block.t().contiguous() @ xd[c0:c1]
    return y.reshape((len(y),) + x.shape[1:]).cpu()


def exact(case, seed):
    if case["kind"] in ("spmv", "spmm"):
        return _exact_product(_arrays(case, seed), _rhs(case, seed, case.get("n_rhs", 1)))
    if case["kind"] == "batch":
        out = []
        for c, s in _members(case, seed):
            a = _arrays(c, s)
            out += [_exact_product(a, _rhs(c, s, n)) for n in (1, case["n_rhs"])]
        return out
    if case["kind"] == "train":
        z, t, mask, p = (v.astype(np.float64) for v in _samples(case, seed))
        F, H, K = mlp.N_FEATURES, mlp.N_HIDDEN, mlp.N_OUT
        w1, b1, w2, b2 = np.split(p, np.cumsum([H * F, H, K * H]))
        h = np.maximum(z @ w1.reshape(H, F).T + b1, 0)
        out = h @ w2.reshape(K, H).T + b2
        d = 2 * (out - t) * mask / mask.sum()
        dh = (d @ w2.reshape(K, H)) * (h > 0)
        return dict(out=out, grad=np.concatenate([(dh.T @ z).ravel(), dh.sum(0), (d.T @ h).ravel(), d.sum(0)]))
    return None  # copies and whole numbers: held to be the same
