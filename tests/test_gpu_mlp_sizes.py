"""The router network's kernels at the edges of their work split (marked gpu):
batches around the 16 samples of a forward workgroup and the 1024 threads of
a backward one, more gradients per hidden unit than one workgroup holds, and
parameters on both sides of what forward keeps in LDS.

Tolerance: a gradient is a sum of n products of FP32 values; summed in FP32
its error is at most about (n + H + K + F) * 2^-24 of the sum of their
magnitudes, taken here against the FP64 oracle."""
import numpy as np
import pytest

from oracle import mlp_oracle as MO

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n,F,H,K", [(1, 6, 32, 6), (15, 6, 32, 6), (16, 1, 1, 1), (17, 6, 32, 6), (1023, 6, 32, 3),
                                     (1025, 6, 32, 6), (300, 9, 17, 6), (70, 64, 256, 64), (2100, 20, 33, 12)])
def test_gradient_and_separate_calls(n, F, H, K):
    from sable_amd import runtime as rt
    from sable_amd.router import mlp
    from sable_amd._lib import check, lib
    rng = np.random.default_rng(n)
    p = mlp.init_params(n, F, H, K)
    X, T = rng.normal(0, 1, (n, F)).astype(np.float32), rng.normal(0, 1, (n, K)).astype(np.float32)
    M = (rng.random((n, K)) < 0.8).astype(np.float32)
    net = mlp.DeviceMLP(p, F, H, K)
    Xd, Td, Md = (rt.DeviceArray.from_numpy(v) for v in (X, T, M))
    print(f"case: n={n} F={F} H={H} K={K}", flush=True)
    scale = 1.0 / n
    out = net.gradient(Xd, Td, Md, n, scale)
    o64, h64 = MO.forward(p, X, F, H, K)
    assert np.allclose(out.numpy(), o64, rtol=1e-4, atol=1e-4)
    W1, b1, W2, b2 = MO.unpack(p, F, H, K)
    d = np.abs(2 * scale * (o64 - T) * M)
    dh = d @ np.abs(W2)
    mag = np.concatenate([(dh.T @ np.abs(X)).ravel(), dh.sum(0), (d.T @ h64).ravel(), d.sum(0)])
    # the forward's own rounding reaches every residual (first term), then
    # the sums; a unit within rounding of its threshold may switch
    eps = 2.0 ** -24
    near = np.min(np.abs(X.astype(np.float64) @ W1.T + b1), initial=1.0) < 1e-5
    err = np.abs(net.g.numpy() - MO.grad(p, X, T, M, F, H, K, scale)[1])
    bound = (n + 4 * (F + H + K)) * eps * mag + 64 * eps * np.max(mag)
    assert near or np.all(err <= bound)
    # the separate calls give the same bits
    bufs = [rt.DeviceArray((n, K)), rt.DeviceArray((n, H)), rt.DeviceArray((n, K)), rt.DeviceArray(p.size)]
    o, h, dd, g = bufs
    check(lib.sable_mlp_forward(net.p.ptr, F, H, K, Xd.ptr, n, o.ptr, h.ptr))
    check(lib.sable_mlp_mse_grad(o.ptr, Td.ptr, Md.ptr, n * K, scale, dd.ptr))
    check(lib.sable_mlp_backward(net.p.ptr, F, H, K, Xd.ptr, n, h.ptr, dd.ptr, g.ptr))
    assert np.array_equal(o.numpy(), out.numpy()) and np.array_equal(g.numpy(), net.g.numpy())


def test_empty_batch_has_zero_gradient():
    from sable_amd import runtime as rt
    from sable_amd.router import mlp
    from sable_amd._lib import check, lib
    net = mlp.DeviceMLP(mlp.init_params(3))
    net.g.copy_from(np.ones(net.p.size, np.float32))
    x = rt.DeviceArray.zeros((1, 64))
    check(lib.sable_mlp_backward(net.p.ptr, net.F, net.H, net.K, x.ptr, 0, x.ptr, x.ptr, net.g.ptr))
    assert not np.any(net.g.numpy())
