"""casl_stencil_get_path names the path of mixed calls, so that setting the
path to what it returned changes no result."""
import pytest

import casl_p4est_amd as C
from casl_p4est_amd import levelset as ls

pytestmark = pytest.mark.gpu

GRIDS = [  # dim, box edge, finest level, the path of a default mixed call
    (2, 1.0, 8, "tiled"), (2, 3.0, 8, "two_pass"),
    (3, 1.0, 6, "tiled"), (3, 3.0, 6, "two_pass"), (3, 2.5, 5, "two_pass"),
]


@pytest.mark.parametrize("dim,box,lmax,path", GRIDS)
def test_setting_the_path_got_changes_nothing(cuda, dim, box, lmax, path):
    import torch
    shape = ls.Sphere([0.45 * box] * dim, 0.31 * box)
    g = C.DeviceGrid(dim, shape, 2, lmax, lip=2.4, box_min=[0.0] * dim, box_max=[box] * dim)
    ds = g.device()
    assert ds.tile_info()["tiled"]
    p0 = g.sample(shape)
    p0 = p0 * (1.0 + 0.4 * torch.sin(g.sample(ls.Plane([5.0 / box] * dim, 0.2))))

    def results():
        out = [ds.reinit(p0.clone(), space, 2, 5, C.DBL_MAX, -C.DBL_MAX, prec) for prec in (0, 1) for space in (1, 2)]
        nrm = ds.normals(p0)
        return out + [ds.advect(p0.clone(), p0, 1e-3 * box), nrm, ds.mean_curvature(nrm)]

    before = results()
    assert ds.path == path
    ds.set_path(ds.path)
    assert ds.path == path
    for a, b in zip(before, results()):
        assert torch.equal(a, b)
    for other in ("tiled", "two_pass"):
        ds.set_path(other)
        assert ds.path == other
