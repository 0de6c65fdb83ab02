"""The fused training pass of the 128x4 networks against the same step made
layer by layer from the exposed BF16 GEMM (one K chunk, so below 512 rows):
weight gradients bit for bit, bias gradients and loss to FP32 rounding, at row
counts around the 32 and 64 rows its waves and blocks take and at input widths
of one and two MFMA steps.  Larger batches (split over K) against each other
through a fresh network with the updated weights, which also pins the
transposed weight copy that Adam keeps."""
import ctypes

import numpy as np
import pytest

from casl_p4est_amd import _lib as L
from casl_p4est_amd import curvature as CV

pytestmark = pytest.mark.gpu


def bf16(torch, a):
    return a.to(torch.bfloat16).contiguous()


def gemm(torch, a, b, ta=0, tb=0, bias=None, relu=0):
    M, K = (a.shape[1], a.shape[0]) if ta else a.shape
    N = b.shape[0] if tb else b.shape[1]
    out = torch.empty((M, N), dtype=torch.float32, device=a.device)
    p = lambda t: ctypes.c_void_p(t.data_ptr()) if t is not None else None
    L.call("casl_bf16_gemm", M, N, K, p(a), a.shape[1], ta, p(b), b.shape[1], tb, p(bias), relu, p(out), None, N, None)
    return out


def make(torch, width, n, seed):
    net = CV.CurvatureNet((width, 128, 128, 128, 128, 1), seed=seed, zero_last_layer=False)
    rng = np.random.default_rng(seed)
    net.set_scaler(rng.normal(size=width) * 0.2, rng.uniform(0.5, 2.0, size=width))
    w, b = net.params()
    net.set_params(w, (rng.normal(size=b.size) * 0.05).astype(np.float32))
    x = torch.from_numpy(rng.normal(size=(n, width)).astype(np.float32)).cuda()
    t = torch.from_numpy(rng.normal(size=n).astype(np.float32)).cuda()
    return net, x, t


@pytest.mark.parametrize("width", [10, 17, 28, 32])
@pytest.mark.parametrize("n", [1, 31, 33, 64, 65, 300])
def test_matches_layer_by_layer(cuda, width, n):
    import torch
    net, x, t = make(torch, width, n, 7 * n + width)
    w, b = (torch.from_numpy(v).cuda() for v in net.params())
    loss = net.backward(x, t)
    gw, gb = net.grads()
    W, B, o, ob = [], [], 0, 0
    for i, k in zip(net.dims[:-1], net.dims[1:]):
        W.append(bf16(torch, w[o:o + i * k].view(i, k)))
        B.append(b[ob:ob + k].contiguous())
        o, ob = o + i * k, ob + k
    inv = torch.from_numpy(np.float32(1) / net.std).cuda()
    A = [bf16(torch, (x - torch.from_numpy(net.mean).cuda()) * inv)]
    for l in range(4):
        A.append(bf16(torch, gemm(torch, A[l], W[l], bias=B[l], relu=1)))
    e = gemm(torch, A[4], W[4], bias=B[4])[:, 0] - t
    assert loss == pytest.approx(float((e.double() ** 2).mean()), rel=1e-5)
    dz = (2.0 * e * (np.float32(1) / np.float32(n)))[:, None]
    o, ob = gw.size, gb.size
    for l in range(4, -1, -1):
        i, k = net.dims[l], net.dims[l + 1]
        o, ob = o - i * k, ob - k
        d16 = bf16(torch, dz)
        assert np.array_equal(gw[o:o + i * k].reshape(i, k), gemm(torch, A[l], d16, ta=1).cpu().numpy()), l
        np.testing.assert_allclose(gb[ob:ob + k], dz.double().sum(0).cpu().numpy(), rtol=1e-4,
                                   atol=1e-6 * float(dz.abs().sum(0).max()))
        if l > 0:
            dz = gemm(torch, d16, W[l], tb=1) * (A[l].float() > 0)


@pytest.mark.parametrize("width,n", [(10, 4096), (28, 5003)])
def test_updated_weights_reach_every_copy(cuda, width, n):
    import torch
    net, x, t = make(torch, width, n, 3)
    for _ in range(3):
        net.backward(x, t)
        net.adam_step(1e-2)
    fresh = CV.CurvatureNet(net.dims, seed=1)
    fresh.set_scaler(net.mean, net.std)
    fresh.set_params(*net.params())
    assert net.backward(x, t) == fresh.backward(x, t)
    for a, b in zip(net.grads(), fresh.grads()):
        assert np.array_equal(a, b)
    assert torch.equal(net.forward(x), fresh.forward(x))
