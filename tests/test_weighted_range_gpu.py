"""FP64 tiles of cubic cells whose edge is no power of two against those of
dyadic cubes, where every scaling is exact: the same grid on a box of edge 3
and one of edge 4, phi scaled alike, some nodes of it infinite or NaN.
A stage leaves infinities and NaN at the same nodes of both."""
import pytest

import casl_p4est_amd as C
from casl_p4est_amd import levelset as ls

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dim,lmin,lmax", [(2, 2, 8), (2, 9, 10), (3, 2, 5), (3, 5, 7)],
                         ids=["2d_small", "2d_full", "3d_small", "3d_full"])
@pytest.mark.parametrize("value", [float("inf"), float("-inf"), float("nan")])
def test_ends_of_the_range_spread_alike(cuda, dim, lmin, lmax, value):
    import torch
    out = []
    for box in (4.0, 3.0):
        shape = ls.Sphere([0.45 * box] * dim, 0.31 * box)
        g = C.DeviceGrid(dim, shape, lmin, lmax, lip=1.2, box_min=[0.0] * dim, box_max=[box] * dim)
        ds = g.device()
        ds.set_path("tiled")
        assert ds.tile_info()["tiled"]
        if box == 4.0:
            p4 = g.sample(shape)
            p4 = p4 * (1.0 + 0.4 * torch.sin(g.sample(ls.Plane([1.3] * dim, 0.2))))
            at = torch.randperm(g.num_nodes, device=cuda, generator=torch.Generator(cuda).manual_seed(3))
            at = at[:max(3, g.num_nodes // 500)]
        assert g.num_nodes == p4.numel()
        p = p4 * (box / 4.0)
        p[at] = value
        vn = torch.cos(p4)
        got = [ds.reinit(p.clone(), space, 1, 1, C.DBL_MAX, -C.DBL_MAX, 0) for space in (1, 2)]
        got.append(ds.advect(p.clone(), vn, 1e-3 * box))
        out.append(got)
    for a, b in zip(*out):
        assert torch.equal(a.isnan(), b.isnan())
        assert torch.equal(a.isposinf(), b.isposinf()) and torch.equal(a.isneginf(), b.isneginf())
