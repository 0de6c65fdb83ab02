"""The default path of mixed calls on cubic cells whose edges are no powers of
two depends on how many full-size tiles the grid makes, halved ones counted:
nodes in an order that is not p4est's make many more tiles than N over the
tile size, in grids of small and of full-size tiles."""
import numpy as np
import pytest

import casl_p4est_amd as C
from casl_p4est_amd import levelset as ls

pytestmark = pytest.mark.gpu


def shuffled(tab, seed):
    """The same grid with its nodes renumbered at random; old[i] is new node i."""
    F, N = 2 * tab.dim, tab.n_nodes
    old = np.random.default_rng(seed).permutation(N)
    new = np.empty(N, dtype=np.int32)
    new[old] = np.arange(N, dtype=np.int32)
    nbr = new[np.asarray(tab.nbr).reshape(-1, N)[:, old]]
    d, dt = np.asarray(tab.d).reshape(F, N)[:, old], np.asarray(tab.d_tr).reshape(-1, N)[:, old]
    wall = np.asarray(tab.wall)[old]
    return C.FlatStencil(tab.dim, *(np.ascontiguousarray(a) for a in (nbr, d, dt, wall)), tab.zero_distance_threshold), old


@pytest.mark.parametrize("dim,lmin,lmax,lip", [(2, 3, 12, 2.4), (2, 9, 10, 1.2), (3, 2, 6, 2.4), (3, 4, 7, 2.4)],
                         ids=["2d_small", "2d_full", "3d_small", "3d_full"])
def test_default_path_counts_halved_tiles(cuda, dim, lmin, lmax, lip):
    import torch
    shape = ls.Sphere([1.35] * dim, 0.93)
    f = C.Forest(dim, [0.0] * dim, [3.0] * dim).refine_levelset(shape, lmin, lmax, lip=lip).build_nodes()
    tab = C.NodeNeighbors(f).init_neighbors().tables
    units = torch.cuda.get_device_properties(0).multi_processor_count
    _, xyz = f.nodes()
    phi0 = f.sample(shape) * (1.0 + 0.4 * np.sin(2 * xyz[:, 0]) * np.cos(3 * xyz[:, 1]))
    for t, old in ((tab, np.arange(tab.n_nodes)), shuffled(tab, 7)):
        ds = C.DeviceStencil(t)
        assert ds.tile_info()["tiled"]
        # in its own order the grid makes fewer full-size tiles than there are
        # compute units; at random (4 or 6 foreign nodes each) it makes more
        assert tab.n_nodes < 1536 * units
        default = "two_pass" if t is tab else "tiled"
        assert ds.path == default
        out = {}
        for path in (None, "tiled", "two_pass"):
            if path:
                ds.set_path(path)
            p = torch.from_numpy(phi0[old]).to(cuda)
            out[path] = ds.reinit(p, 2, 2, 4, C.DBL_MAX, -C.DBL_MAX, 1)
        assert not torch.equal(out["tiled"], out["two_pass"])
        assert torch.equal(out[None], out[default])
