"""Full-size tiles where the other tests' grids are cut into small ones: FP64
over cubic cells of an edge that is no power of two, and 2D cells that are not
cubes, bit for bit as the grid-wide kernels, mixed calls within 1e-3 finest
cells of FP64 near the interface; and a box whose origin rounds the offsets of
the cells, which stays on the grid-wide kernels in FP64."""
import ctypes

import numpy as np
import pytest

import casl_p4est_amd as C
from casl_p4est_amd import _lib as L
from casl_p4est_amd import levelset as ls
from oracle import pyoracle as O

pytestmark = pytest.mark.gpu


def problem(dim, box, lmin, lmax, lip=1.2):
    import torch
    m = min(box)
    shape = ls.Sphere([0.45 * e for e in box], 0.3 * m)
    g = C.DeviceGrid(dim, shape, lmin, lmax, lip=lip, box_min=[0.0] * dim, box_max=box)
    p0 = g.sample(shape)
    return g, p0 * (1.0 + 0.4 * torch.sin(g.sample(ls.Plane([7.0 / m] * dim, 0.3))))


@pytest.mark.parametrize("dim,box,lmin,lmax", [
    (2, [3.0, 3.0], 9, 11), (2, [2.5, 2.5], 3, 14), (3, [3.0] * 3, 5, 7), (3, [6.0] * 3, 3, 8), (2, [2.0, 1.0], 9, 11),
    (2, [1.0, 4.0], 3, 14)], ids=str)
def test_fp64_full_size_tiles(cuda, dim, box, lmin, lmax):
    import torch
    g, p0 = problem(dim, box, lmin, lmax)
    ds = g.device()
    info = ds.tile_info()
    assert info["tiled"] and g.num_nodes / info["n_tiles"] > 256 and info["n_irregular"] > 0
    mask = (torch.rand(g.num_nodes, device=cuda, generator=torch.Generator(cuda).manual_seed(5)) < 0.8).to(torch.uint8)
    vn, m = torch.cos(p0 * (9.0 / min(box))), min(box)
    out = []
    for path in ("tiled", "two_pass"):
        ds.set_path(path)
        got = [ds.reinit(p0.clone(), space, time, 4, C.DBL_MAX, -C.DBL_MAX, 0)
               for space, time in ((2, 2), (2, 1), (1, 2), (1, 1))]
        got.append(ds.reinit(p0.clone(), 2, 2, 3, 0.2 * m, -0.1 * m, 0, mask=mask))
        got.append(ds.advect(p0.clone(), vn, 0.3 * m * 2.0 ** -lmax))
        mixed = ds.reinit(p0.clone(), 2, 2, 4, C.DBL_MAX, -C.DBL_MAX, 1)
        h = m * 2.0 ** -lmax
        assert ds.band_linf(mixed, got[0], got[0], 3 * h) <= 1e-3 * h, path
        out.append(got)
    for k, (a, b) in enumerate(zip(*out)):
        assert torch.equal(a, b), k


def count(kernel):
    ms, n = ctypes.c_double(), ctypes.c_int64()
    L.call("casl_profile_query", kernel.encode(), ctypes.byref(ms), ctypes.byref(n))
    return n.value


def test_rounded_offsets_stay_grid_wide(cuda):
    """A box whose origin rounds the offsets of regular faces by less than the
    construction's threshold, each still exact in FP32: tiled, but the weights
    share no significand, so FP64 calls run the grid-wide kernels."""
    import torch
    lo, edge, level = 2.0 ** 26, 0.75 + 2.0 ** -24, 3
    shape = ls.Sphere([lo + 0.45 * edge] * 3, 0.31 * edge)
    f = C.Forest(3, [lo] * 3, [lo + edge] * 3).refine_levelset(shape, level, level).build_nodes()
    ngbd = C.NodeNeighbors(f).init_neighbors()
    tab = ngbd.tables
    q, offsets = edge * 2.0 ** -level, np.asarray(tab.d_tr)
    assert bool(((offsets != 0) & (offsets != q)).any())
    phi0 = f.sample(shape) * (1.0 + 0.4 * np.sin(np.arange(tab.n_nodes) * 0.7))
    ref = O.reinit(tab, phi0, 2, 2, 4)
    ds = ngbd.device()
    ds.set_path("tiled")
    assert ds.tile_info()["tiled"]
    L.call("casl_profile_enable", 1)
    L.call("casl_profile_reset")
    try:
        p = torch.from_numpy(phi0).to(cuda)
        out = ds.reinit(p, 2, 2, 4, C.DBL_MAX, -C.DBL_MAX, 0).cpu().numpy()
        vn = np.cos(np.arange(tab.n_nodes) * 0.01)
        p = torch.from_numpy(phi0).to(cuda)
        ds.advect(p, torch.from_numpy(vn).to(cuda), 0.01 * q)
        launches = {k: count(k) for k in ("k_tile_stage", "k_tile_prep", "k_tile_advect", "k_stage", "k_advect")}
    finally:
        L.call("casl_profile_enable", 0)
    assert launches["k_stage"] == 8 and launches["k_advect"] == 2, launches
    assert not any(v for k, v in launches.items() if k.startswith("k_tile")), launches
    assert np.array_equal(out, ref)
    assert np.array_equal(p.cpu().numpy(), O.advect(tab, phi0, vn, 0.01 * q))
