"""The device's refinement and node numbering against the host's where its
blocks, prefix tables and merged key lists have edges: minimum levels from 0
to past the prefix tables' cells, one cell, a leaf count around one block,
grids finer than a prefix and all hanging nodes on one side, spheres that
are culled, touch, coincide or lie far outside, and none at all."""
import numpy as np
import pytest

import casl_p4est_amd as C
from casl_p4est_amd import levelset as ls

pytestmark = pytest.mark.gpu

CASES = {
    "one cell 2d": (2, ls.Sphere([0.5, 0.5], 0.3), 0, 0, 1.2, None, None),
    "one cell 3d": (3, ls.Sphere([0.5, 0.5, 0.5], 0.3), 0, 0, 1.2, None, None),
    "from level 0 2d": (2, ls.Sphere([0.4, 0.6], 0.3), 0, 9, 1.2, None, None),
    "from level 0 3d": (3, ls.Sphere([0.4, 0.6, 0.5], 0.3), 0, 6, 1.2, None, None),
    "256 leaves 2d": (2, ls.Sphere([0.5, 0.5], 0.3), 4, 4, 1.2, None, None),
    "minimum past the maximum 3d": (3, ls.Sphere([0.5, 0.5, 0.5], 0.3), 4, 2, 1.2, None, None),
    "past the prefix 2d": (2, ls.Sphere([0.3, 0.7], 1e-3), 1, 16, 8.0, None, None),
    "past the prefix 3d": (3, ls.Sphere([0.3, 0.7, 0.4], 1e-3), 1, 12, 4.0, None, None),
    "at a corner 3d": (3, ls.Sphere([1.0, 1.0, 1.0], 0.01), 1, 10, 2.0, None, None),
    "distant box 3d": (3, ls.Spheres([[1e6 + 0.4, -2e6 + 0.5, 0.3], [1e6 + 0.8, -2e6 + 0.7, 0.6]], [0.2, 0.1], 0.0),
                       1, 6, 1.2, [1e6, -2e6, 0.0], [1e6 + 1.0, -2e6 + 1.0, 1.0]),
    "spheres 3d": (3, ls.Spheres([[0.3, 0.3, 0.3], [0.3, 0.3, 0.3], [0.5, 0.3, 0.3], [0.62, 0.55, 0.6], [9.0, 9.0, 9.0],
                                  [0.6, 0.5, 0.5]], [0.1, 0.1, 0.1, 0.2, 0.5, -0.1], 0.0), 2, 7, 1.2, None, None),
    "no band 3d": (3, ls.Spheres([[0.5, 0.5, 0.5]], [0.3], 0.0), 2, 6, 0.0, None, None),
}


@pytest.mark.parametrize("name", CASES)
def test_device_grid_equals_host(cuda, name):
    dim, phi, lmin, lmax, lip, lo, hi = CASES[name]
    f = C.Forest(dim, lo, hi).refine_levelset(phi, lmin, lmax, lip=lip).build_nodes()
    if f.sizes()[0] == 1:  # no cell beyond a wall node's: refused by both
        with pytest.raises(C.CaslError):
            C.flat_stencil_from_forest(f)
        with pytest.raises(C.CaslError):
            C.DeviceGrid(dim, phi, lmin, lmax, lip=lip, box_min=lo, box_max=hi)
        return
    g = C.DeviceGrid(dim, phi, lmin, lmax, lip=lip, box_min=lo, box_max=hi)
    print(f"[grid] {name}: {f.sizes()}", flush=True)
    assert g.sizes() == f.sizes()
    assert np.array_equal(g.node_ixyz(), f.nodes()[0])
    tab, dt = C.flat_stencil_from_forest(f), g.tables()
    for field in ("nbr", "wall"):
        assert np.array_equal(getattr(dt, field), getattr(tab, field))
    for field in ("d", "d_tr"):
        assert np.array_equal(getattr(dt, field).view(np.uint64), getattr(tab, field).view(np.uint64))
    assert np.array_equal(g.sample(phi).cpu().numpy().view(np.uint64), f.sample(phi).view(np.uint64))


def test_refinement_by_many_modulated_spheres(cuda):
    """Culled spheres and shared modulation factors on the device against every
    sphere at every corner on the host."""
    rng = np.random.default_rng(5)
    phi = ls.Spheres(rng.uniform(0.1, 0.9, (90, 3)).tolist(), rng.uniform(0.02, 0.15, 90).tolist(), 0.3)
    f = C.Forest(3).refine_levelset(phi, 2, 7, lip=1.2).build_nodes()
    g = C.DeviceGrid(3, phi, 2, 7, lip=1.2)
    # sin and cos may differ in the last place between host and device, which
    # moves no decision of this grid
    assert g.sizes() == f.sizes()
    assert np.array_equal(g.node_ixyz(), f.nodes()[0])
