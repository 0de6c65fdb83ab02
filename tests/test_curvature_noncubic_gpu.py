"""Normals and mean curvature on the tiles of cells that are not cubes equal
the grid-wide tables' bit for bit: boxes of 2:1 edges, and flat ones where the
test that drops a correction (its weight over the node's largest distance,
against 1e-13) is close to either side."""
import pytest

import casl_p4est_amd as C
from casl_p4est_amd import levelset as ls

pytestmark = pytest.mark.gpu

BOXES = [[2.0, 1.0], [1.0, 4.0], [2.0, 1.0, 0.5], [1.0, 1.0, 2.0]]
BOXES += [[1.0, 2.0 ** -k] for k in (19, 20, 21, 22)] + [[2.0 ** -k, 1.0] for k in (20, 21)]
BOXES += [[1.0, 1.0, 2.0 ** -21], [1.0, 2.0 ** -20, 2.0], [2.0 ** -21, 1.0, 0.5], [1.0, 2.0 ** -21, 2.0 ** -21]]


@pytest.mark.parametrize("box", BOXES, ids=str)
def test_tiles_equal_tables(cuda, box):
    import torch
    dim = len(box)
    # a plane through the middle of the box in its own coordinates; a small
    # Lipschitz constant, so that neighbouring leaves differ by several levels
    k = [1.0 / b for b in box]
    steep = max(k)
    shape = ls.Plane([a / steep for a in k], -0.47 * dim / steep)
    g = C.DeviceGrid(dim, shape, 1, 9 if dim == 2 else 6, lip=1e-3 * min(box) / max(box), box_min=[0.0] * dim, box_max=box)
    ds = g.device()
    assert ds.tile_info()["tiled"] and ds.tile_info()["n_irregular"] > 0
    s = g.sample(shape) * steep
    t = g.sample(ls.Plane([(1.7 + a) * q / steep for a, q in enumerate(k)], 0.1)) * steep
    phi = s + 0.3 * torch.sin(3.0 * t) * torch.cos(5.0 * s)
    out = []
    for path in ("two_pass", "tiled"):
        ds.set_path(path)
        nrm = ds.normals(phi)
        out.append((nrm, ds.mean_curvature(nrm), ds.mean_curvature(torch.stack([phi] * dim))))
    for a, b in zip(*out):
        assert torch.equal(a, b)
