"""The fused network curvature kernel against normalisation + network + blend
as three calls, bit for bit, at sample counts around the 32 and 64 rows its
waves take and the rows its blocks spread over, from aligned and unaligned
feature arrays, with flat, symmetric and non-finite stencils among them."""
import numpy as np
import pytest

from casl_p4est_amd import curvature as CV

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dims", [CV.DIMS_2D, CV.DIMS_3D], ids=["2d", "3d"])
@pytest.mark.parametrize("n", [1, 15, 16, 17, 32, 33, 64, 65, 1000, 33000])
def test_fused_equals_three_calls(cuda, dims, n):
    import torch
    net = CV.CurvatureNet(dims, seed=n, zero_last_layer=False)
    net.set_scaler(np.linspace(-0.3, 0.3, dims[0]), np.linspace(0.5, 2.0, dims[0]))
    g = torch.Generator(device="cuda")
    g.manual_seed(n)
    for shift in (0, 1):
        f = torch.randn(n * dims[0] + shift, device=cuda, generator=g)[shift:].view(n, dims[0])
        f[:, -1] *= 0.02
        if n > 12:
            f[3] = 0.0
            f[5, :-1] = 1.0
            f[9, -1] = 0.005
            f[11] = float("nan")
            f[12, 4] = float("inf")
        assert (f.data_ptr() % 16 == 0) == (shift == 0)
        a = CV.hybrid_hk(net, f, fused=True).cpu().numpy()
        b = CV.hybrid_hk(net, f, fused=False).cpu().numpy()
        assert np.array_equal(a, b, equal_nan=True)
