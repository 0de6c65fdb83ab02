"""Stage kernels compiled for cubic dyadic cells and for any cells against the
two-pass kernels: FP64 reinitialization and advection bit for bit, the mixed
path within its bound of 1e-3 finest cells of the FP64 result, on small and
full-size tiles, cubes of edges other than 1 among them."""
import numpy as np
import pytest

import casl_p4est_amd as C
from casl_p4est_amd import levelset as ls

pytestmark = pytest.mark.gpu

BOXES = {2: [[1.0, 1.0], [0.25, 0.25], [8.0, 8.0], [2.0, 1.0]],
         3: [[1.0] * 3, [0.25] * 3, [8.0] * 3, [2.0, 1.0, 0.5], [1.0, 1.0, 2.0]]}


@pytest.mark.parametrize("lmax", [6, 8], ids=["small", "large"])
@pytest.mark.parametrize("dim,box", [(d, b) for d in BOXES for b in BOXES[d]], ids=str)
def test_tiled_equals_two_pass(cuda, dim, box, lmax):
    import torch
    lmax += 3 if dim == 2 else 0
    m = min(box)
    phi = ls.Sphere([0.45 * e for e in box], 0.3 * m)
    g = C.DeviceGrid(dim, phi, 2, lmax, lip=1.2, box_min=[0.0] * dim, box_max=box)
    st = g.device()
    assert st.tile_info()["tiled"]
    p0 = g.sample(phi)
    p0 = p0 * (1.0 + 0.4 * torch.sin(p0 * (20.0 / m)))
    v = torch.cos(p0 * (9.0 / m))
    out = {}
    for path in ("tiled", "two_pass"):
        st.set_path(path)
        for prec in (0, 1):
            a = p0.clone()
            st.reinit(a, 2, 2, 4, C.DBL_MAX, -C.DBL_MAX, prec)
            out[path, prec] = a.cpu().numpy()
        a = p0.clone()
        st.advect(a, v, 0.3 * m * 2.0 ** -lmax)
        out[path, "advect"] = a.cpu().numpy()
    for k in (0, "advect"):
        assert np.array_equal(out["tiled", k].view(np.uint64), out["two_pass", k].view(np.uint64))
    assert np.abs(out["tiled", 1] - out["tiled", 0]).max() <= 1e-3 * m * 2.0 ** -lmax
