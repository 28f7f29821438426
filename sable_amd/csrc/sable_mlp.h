// Router network kernels: a 2-layer MLP (FP32) with ReLU hidden layer.
//
//   hidden = relu(W1 x + b1)       W1: H x F, b1: H
//   out    = W2 hidden + b2        W2: K x H, b2: K
//
// Parameters live in one flat array [W1, b1, W2, b2].  The loss kernel forms
// the gradient of a masked mean squared error, so a whole training step
// (forward, loss gradient, backward, Adam) runs on the device.
//
// A mini-batch is tiny (4096 samples of 6 features: 0.4 MB), so both kernels
// are bound by their chains of dependent loads and by how many wavefronts
// share them.  Forward: 16 lanes per sample, the parameters in LDS (a thread
// per sample left 16 workgroups walking 400 loads each: 48 us, now 5).
// Backward: a workgroup per hidden unit, each thread summing every
// SB_MLP_BWG-th sample for all of the unit's gradients, then a fixed tree
// over the workgroup: deterministic, no atomics (a thread per parameter
// summing the samples one after another took 2796 us, now 24).
#pragma once

#include "sable_device.h"

#define SB_MLP_SPB 16           // forward: samples per workgroup (16 lanes each)
#define SB_MLP_LDS 4096         // forward: parameters held in LDS at most
#define SB_MLP_BWG 1024         // backward: threads per workgroup
#define SB_MLP_BOUT 16          // backward: gradients of a hidden unit per workgroup

// The forward pass of this workgroup's samples with the parameters at P; a
// sample's sums run in index order.  With target, also the loss gradient.
template <typename Ptr>
__device__ __forceinline__ void sb_mlp_forward_body(Ptr P, int F, int H, int K, const float *__restrict__ X, int n,
                                                    float *__restrict__ out, float *__restrict__ hidden,
                                                    const float *__restrict__ target, const float *__restrict__ mask,
                                                    float scale, float *__restrict__ dout, float *h)
{
    const Ptr W1 = P, b1 = W1 + H * F, W2 = b1 + H, b2 = W2 + K * H;
    const int l = threadIdx.x & 15;
    const int64_t i = (int64_t)blockIdx.x * SB_MLP_SPB + (threadIdx.x >> 4);
    h += (threadIdx.x >> 4) * H;
    if (i < n) {
        const float *x = X + i * F;
        for (int j = l; j < H; j += 16) {
            float s = b1[j];
            for (int f = 0; f < F; ++f) s += W1[j * F + f] * x[f];
            s = s > 0.f ? s : 0.f;
            h[j] = s;
            hidden[i * H + j] = s;
        }
    }
    __syncthreads();
    if (i < n) {
        for (int k = l; k < K; k += 16) {
            float s = b2[k];
#pragma unroll 8
            for (int j = 0; j < H; ++j) s += W2[k * H + j] * h[j];
            out[i * K + k] = s;
            if (target) dout[i * K + k] = scale * 2.f * (s - target[i * K + k]) * mask[i * K + k];
        }
    }
}

extern "C" __global__ void __launch_bounds__(256)
sb_mlp_forward_kernel(const float *__restrict__ P, int F, int H, int K, const float *__restrict__ X, int n,
                      float *__restrict__ out, float *__restrict__ hidden, const float *__restrict__ target,
                      const float *__restrict__ mask, float scale, float *__restrict__ dout)
{
    __shared__ float p[SB_MLP_LDS];
    __shared__ float h[SB_MLP_SPB * 256];        // H is at most 256
    const int np = H * F + H + K * H + K;
    if (np <= SB_MLP_LDS) {
        for (int q = threadIdx.x; q < np; q += 256) p[q] = P[q];
        __syncthreads();
        sb_mlp_forward_body((const __attribute__((address_space(3))) float *)p, F, H, K, X, n, out, hidden, target, mask,
                            scale, dout, h);
    } else {
        sb_mlp_forward_body(P, F, H, K, X, n, out, hidden, target, mask, scale, dout, h);
    }
}

// Workgroup (j, c): hidden unit j's gradients c * SB_MLP_BOUT .. of
// [dL/dW1[j][0..F), dL/db1[j], dL/dW2[0..K)[j]]; j = H: those of b2.
extern "C" __global__ void __launch_bounds__(SB_MLP_BWG)
sb_mlp_backward_kernel(const float *__restrict__ P, int F, int H, int K, const float *__restrict__ X, int n,
                       const float *__restrict__ hidden, const float *__restrict__ dout, float *__restrict__ G)
{
    __shared__ float part[SB_MLP_BWG / 64][SB_MLP_BOUT];
    const int nW1 = H * F;
    const float *W2 = P + nW1 + H;
    const int j = blockIdx.x, o0 = blockIdx.y * SB_MLP_BOUT;
    const int nout = j < H ? F + 1 + K : K;
    if (o0 >= nout) return;
    float g[SB_MLP_BOUT];
#pragma unroll
    for (int q = 0; q < SB_MLP_BOUT; ++q) g[q] = 0.f;
    for (int64_t i = threadIdx.x; i < n; i += SB_MLP_BWG) {
        const float *dk = dout + i * K, *x = X + i * F;
        if (j < H) {
            const float hv = hidden[i * H + j];
            float d = 0.f;                       // dL/d(hidden unit), zero where it is off
            if (o0 <= F)
                for (int k = 0; k < K; ++k) d += dk[k] * W2[k * H + j];
            const bool on = !(hv <= 0.f);
#pragma unroll
            for (int q = 0; q < SB_MLP_BOUT; ++q) {
                const int o = o0 + q;
                if (o < F) {
                    if (on) g[q] += d * x[o];
                } else if (o == F) {
                    if (on) g[q] += d;
                } else if (o < nout) {
                    g[q] += dk[o - F - 1] * hv;
                }
            }
        } else {
#pragma unroll
            for (int q = 0; q < SB_MLP_BOUT; ++q)
                if (o0 + q < nout) g[q] += dk[o0 + q];
        }
    }
#pragma unroll
    for (int q = 0; q < SB_MLP_BOUT; ++q) {
        for (int m = 1; m < 64; m <<= 1) g[q] += __shfl_xor(g[q], m, 64);
        if ((threadIdx.x & 63) == 0) part[threadIdx.x >> 6][q] = g[q];
    }
    __syncthreads();
    const int o = o0 + (int)threadIdx.x;
    if (threadIdx.x >= SB_MLP_BOUT || o >= nout) return;
    float s = 0.f;
    for (int w = 0; w < SB_MLP_BWG / 64; ++w) s += part[w][threadIdx.x];
    const int at = j == H ? nW1 + H + K * H + o : o < F ? j * F + o : o == F ? nW1 + j : nW1 + H + (o - F - 1) * H + j;
    G[at] = s;
}

// dout = scale * 2 * (out - target) * mask   (mask 0/1 per output)
extern "C" __global__ void __launch_bounds__(256)
sb_mlp_mse_grad_kernel(const float *__restrict__ out, const float *__restrict__ target,
                       const float *__restrict__ mask, int64_t n, float scale, float *__restrict__ dout)
{
    const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= n) return;
    dout[i] = scale * 2.f * (out[i] - target[i]) * mask[i];
}

extern "C" __global__ void __launch_bounds__(256)
sb_adam_kernel(float *__restrict__ P, const float *__restrict__ G, float *__restrict__ m, float *__restrict__ v,
               int64_t n, float lr, float b1, float b2, float eps, int step)
{
    const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= n) return;
    const float g = G[i];
    const float mi = b1 * m[i] + (1.f - b1) * g;
    const float vi = b2 * v[i] + (1.f - b2) * g * g;
    m[i] = mi;
    v[i] = vi;
    const float mhat = mi / (1.f - powf(b1, (float)step));
    const float vhat = vi / (1.f - powf(b2, (float)step));
    P[i] -= lr * mhat / (sqrtf(vhat) + eps);
}
