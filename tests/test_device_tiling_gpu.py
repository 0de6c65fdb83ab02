"""The device's tiling against the host's, byte for byte, where its blocks
have something to get wrong: grids of a few nodes, a node count just past a
whole number of tiles, grids on both sides of the small tiles' limit, tiles
with many levels (grids refined to a point) and with hanging faces throughout
(thin shells)."""
import pytest

import casl_p4est_amd as C
from casl_p4est_amd import levelset as ls

pytestmark = pytest.mark.gpu

CASES = {
    "9 nodes": (2, ls.Sphere([0.5, 0.5], 0.3), 1, 1, 1.2),
    "27 nodes": (3, ls.Sphere([0.5, 0.5, 0.5], 0.3), 1, 1, 1.2),
    "17^2 = 256 + 33 nodes": (2, ls.Sphere([0.5, 0.5], 0.3), 4, 4, 1.2),
    "513^2 nodes, full tiles": (2, ls.Sphere([0.5, 0.5], 0.3), 9, 9, 1.2),
    "33^3 nodes": (3, ls.Sphere([0.5, 0.5, 0.5], 0.3), 5, 5, 1.2),
    "65^3 nodes, full tiles": (3, ls.Sphere([0.5, 0.5, 0.5], 0.3), 6, 6, 1.2),
    "to a point 2d": (2, ls.Sphere([0.3, 0.7], 1e-4), 2, 14, 8.0),
    "to a point 3d": (3, ls.Sphere([0.3, 0.7, 0.4], 1e-4), 1, 11, 4.0),
    "thin shell 3d, full tiles": (3, ls.Sphere([0.45, 0.5, 0.55], 0.3), 2, 8, 1.2),
    "thin curve 2d, full tiles": (2, ls.Sphere([0.45, 0.5], 0.3), 2, 15, 1.2),
}


@pytest.mark.parametrize("name", CASES)
def test_device_tiles_equal_host_tiles(cuda, name):
    dim, phi, lmin, lmax, lip = CASES[name]
    f = C.Forest(dim).refine_levelset(phi, lmin, lmax, lip=lip).build_nodes()
    tab = C.flat_stencil_from_forest(f)
    ds = C.DeviceGrid(dim, phi, lmin, lmax, lip=lip).device()
    info = ds.tile_info()
    print(f"[tiles] {name}: {f.sizes()} {info}", flush=True)
    assert info["tiled"], info
    ok, why = ds.tile_check(tab)
    assert ok, why
