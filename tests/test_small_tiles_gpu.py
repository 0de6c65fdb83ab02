"""Grids below one full-size tile per compute unit: the small-tile kernels give
the CPU oracle's bits in FP64 and the grid-wide kernels' bits in mixed
precision, at tile counts from one to the largest grid they take, and the
device builder cuts the same tiles as the host's."""
import numpy as np
import pytest

import casl_p4est_amd as C
from casl_p4est_amd import levelset as ls
from oracle import pyoracle as O

pytestmark = pytest.mark.gpu

GRIDS = {  # dim, level set, min and max level
    "one_tile": (2, ls.Sphere([0.5, 0.5], 0.3), 3, 4),
    "uniform17": (2, ls.Sphere([0.4, 0.5], 0.2), 4, 4),
    "circle_jumps": (2, ls.Sphere([0.45, 0.5], 0.31), 1, 9),
    "star": (2, ls.Star(), 3, 10),
    "uniform9": (3, ls.Sphere([0.5, 0.5, 0.5], 0.3), 3, 3),
    "sphere_jumps": (3, ls.Sphere([0.45, 0.5, 0.55], 0.3), 1, 5),
    "gyroid_walls": (3, ls.Gyroid(), 3, 5),
    "spheres": (3, ls.random_spheres(10, seed=4), 2, 6),
}


@pytest.mark.parametrize("name", sorted(GRIDS))
def test_matches_oracle_and_grid_wide(cuda, name):
    import torch
    dim, shape, lmin, lmax = GRIDS[name]
    f = C.Forest(dim).refine_levelset(shape, lmin, lmax, lip=2.4).build_nodes()
    ngbd = C.NodeNeighbors(f).init_neighbors()
    _, xyz = f.nodes()
    phi0 = f.sample(shape) * (1.0 + 0.4 * np.sin(5 * xyz[:, 0]) * np.cos(4 * xyz[:, 1]))
    ds = ngbd.device()
    info = ds.tile_info()
    assert info["tiled"] and ds.path == "tiled"
    assert info["n_tiles"] >= (f.num_nodes + 255) // 256
    solver = C.LevelSet(ngbd)
    for space, time in ((2, 2), (2, 1), (1, 2), (1, 1)):
        out = {}
        for path in ("tiled", "two_pass"):
            ds.set_path(path)
            phi = torch.from_numpy(phi0).to(cuda)
            solver.reinitialize_within_range_of_phi_0(phi, space, time, C.DBL_MAX, -C.DBL_MAX, 5)
            assert np.array_equal(phi.cpu().numpy(), O.reinit(ngbd.tables, phi0, space, time, 5)), (path, space, time)
            phi = torch.from_numpy(phi0).to(cuda)
            solver.reinitialize_within_range_of_phi_0(phi, space, time, 0.2, -0.1, 5, precision="mixed")
            out[path] = phi
        assert torch.equal(out["tiled"], out["two_pass"]), (space, time)
    vn = np.cos(np.arange(f.num_nodes) * 0.01)
    ds.set_path("tiled")
    phi = torch.from_numpy(phi0).to(cuda)
    dt = solver.advect_in_normal_direction(torch.from_numpy(vn).to(cuda), phi)
    assert np.array_equal(phi.cpu().numpy(), O.advect(ngbd.tables, phi0, vn, dt))
    g = C.DeviceGrid(dim, shape, lmin, lmax, lip=2.4)
    if g.num_nodes == f.num_nodes:
        ok, why = g.device().tile_check(ngbd.tables)
        assert ok, why


@pytest.mark.parametrize("lmax", [12, 13])
def test_both_sides_of_the_size_rule(cuda, lmax):
    """119K nodes take small tiles, 237K full-size ones: the same bits as the
    grid-wide kernels on either side."""
    import torch
    shape = ls.Star()
    g = C.DeviceGrid(2, shape, 4, lmax, lip=2.4)
    ds = g.device()
    per_tile = g.num_nodes / ds.tile_info()["n_tiles"]
    assert (per_tile <= 256) == (g.num_nodes <= 3 << 16)
    phi0 = g.sample(shape)
    for prec in (0, 1):
        out = []
        for path in ("tiled", "two_pass"):
            ds.set_path(path)
            out.append(ds.reinit(phi0.clone(), 2, 2, 6, C.DBL_MAX, -C.DBL_MAX, prec))
        assert torch.equal(out[0], out[1]), prec
