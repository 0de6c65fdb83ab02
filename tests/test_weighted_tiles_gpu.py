"""FP64 on the tiled kernels over cubic cells whose edge is not a power of
two: reinitialization (every order, a mask) and advection equal the CPU oracle
bit for bit, as the grid-wide kernels do, and the host and device builders
agree on which grids may take that path."""
import numpy as np
import pytest

import casl_p4est_amd as C
from casl_p4est_amd import levelset as ls
from oracle import pyoracle as O

pytestmark = pytest.mark.gpu

BOXES = {  # dim, lower corner, upper corner, level
    "square3": (2, [0.0, 0.0], [3.0, 3.0], 8),
    "square2.5": (2, [-1.25, -1.25], [1.25, 1.25], 7),
    "cube3": (3, [0.0] * 3, [3.0] * 3, 6),
    "cube6": (3, [-3.0, 0.0, 1.0], [3.0, 6.0, 7.0], 6),
    "cube_shifted": (3, [0.1, 0.2, 0.3], [3.1, 3.2, 3.3], 5),
}


def problem(name):
    dim, lo, hi, lmax = BOXES[name]
    edge = hi[0] - lo[0]
    shape = ls.Sphere([a + 0.45 * edge for a in lo], 0.31 * edge)
    f = C.Forest(dim, lo, hi).refine_levelset(shape, 2, lmax, lip=2.4).build_nodes()
    phi0 = f.sample(shape)
    _, xyz = f.nodes()
    phi0 = phi0 * (1.0 + 0.4 * np.sin(5 * xyz[:, 0] / edge) * np.cos(4 * xyz[:, 1] / edge))
    return f, C.NodeNeighbors(f).init_neighbors(), phi0, shape


@pytest.mark.parametrize("name", sorted(BOXES))
def test_fp64_matches_oracle(cuda, name):
    import torch
    f, ngbd, phi0, shape = problem(name)
    tab = ngbd.tables
    ds = ngbd.device()
    solver = C.LevelSet(ngbd)
    tiled = ds.tile_info()["tiled"]
    assert tiled or name == "cube_shifted"
    rng = np.random.default_rng(5)
    mask = (rng.random(tab.n_nodes) < 0.8).astype(np.uint8)
    vn = np.sin(np.arange(tab.n_nodes) * 0.01) + 0.2
    for path in ("tiled", "two_pass"):
        ds.set_path(path)
        for space, time in ((2, 2), (2, 1), (1, 2), (1, 1)):
            phi = torch.from_numpy(phi0).to(cuda)
            solver.reinitialize_within_range_of_phi_0(phi, space, time, C.DBL_MAX, -C.DBL_MAX, 6)
            assert np.array_equal(phi.cpu().numpy(), O.reinit(tab, phi0, space, time, 6)), (path, space, time)
        phi = torch.from_numpy(phi0).to(cuda)
        solver.reinitialize_2nd_order_with_mask(phi, torch.from_numpy(mask).to(cuda), number_of_iterations=4)
        assert np.array_equal(phi.cpu().numpy(), O.reinit(tab, phi0, 2, 2, 4, mask=mask)), path
        phi = torch.from_numpy(phi0).to(cuda)
        dt = solver.advect_in_normal_direction(torch.from_numpy(vn).to(cuda), phi)
        assert np.array_equal(phi.cpu().numpy(), O.advect(tab, phi0, vn, dt)), path


@pytest.mark.parametrize("name", ["square3", "cube3", "cube6"])
def test_device_builder_agrees(cuda, name):
    dim, lo, hi, lmax = BOXES[name]
    f, ngbd, _, shape = problem(name)
    g = C.DeviceGrid(dim, shape, 2, lmax, lip=2.4, box_min=lo, box_max=hi)
    ok, why = g.device().tile_check(ngbd.tables)
    assert ok, why
