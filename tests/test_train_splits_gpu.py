"""The fused training pass over batches that are split over the rows: every
weight gradient equals, bit for bit, the sum in order of the split's products
made one by one with the exposed BF16 GEMM."""
import numpy as np
import pytest

from test_train_chain_gpu import bf16, gemm, make

pytestmark = pytest.mark.gpu


def splits(M, N, K):
    """The split-K rule of the layer by layer pass."""
    tiles, s = ((M + 63) // 64) * ((N + 63) // 64), 1
    while s < 64 and tiles * s < 512 and K // (2 * s) >= 256:
        s *= 2
    return s


@pytest.mark.parametrize("width,n", [(10, 513), (28, 1024), (10, 4096), (17, 5003), (10, 8192), (28, 16384), (10, 40001)])
def test_split_batches(cuda, width, n):
    import torch
    net, x, t = make(torch, width, n, n + width)
    w, b = (torch.from_numpy(v).cuda() for v in net.params())
    net.backward(x, t)
    gw, _ = net.grads()
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
    dz = (2.0 * e * (np.float32(1) / np.float32(n)))[:, None]
    sp = splits(128, 128, n)
    kc = (-(-n // sp) + 15) // 16 * 16 if sp > 1 else n
    o = gw.size
    for l in range(4, -1, -1):
        i, k = net.dims[l], net.dims[l + 1]
        o -= i * k
        d16, s = bf16(torch, dz), None
        for z in range(sp):
            part = torch.zeros((i, k), device=cuda)
            if z * kc < n:
                part = gemm(torch, A[l][z * kc:(z + 1) * kc], d16[z * kc:(z + 1) * kc], ta=1)
            s = part if s is None else s + part
        assert np.array_equal(gw[o:o + i * k].reshape(i, k), s.cpu().numpy()), l
        if l > 0:
            dz = gemm(torch, d16, W[l], tb=1) * (A[l].float() > 0)
