"""GPU: the kernels for rows of more than 4096 voxels where their blocks end: row counts on either side of a block's
end, blocks without a triangle beside others, rows in several tiles of pass 3, and enough rows for blocks of
sixteen of them; counts, offsets, Flying Edges and both Marching Cubes orders, run twice, bit for bit against
the oracle."""
import numpy as np
import pytest

from helpers import bits_equal

pytestmark = pytest.mark.gpu

# nx, ny, nz
SIZES = [(4097, 2, 2), (4097, 3, 3), (4160, 5, 2), (4100, 2, 7), (8192, 3, 4), (4101, 37, 29)]


def _same(mesh, points, normals, triangles):
    assert mesh.points.shape == points.shape and mesh.triangles.shape == triangles.shape
    assert bits_equal(mesh.points, points) and bits_equal(mesh.normals, normals) and bits_equal(mesh.triangles, triangles)


@pytest.mark.parametrize("field", ["noise", "few", "none"])
@pytest.mark.parametrize("nx,ny,nz", SIZES)
def test_wide_rows(oracle_mod, nx, ny, nz, field):
    import miniisosurface_amd as m
    rng = np.random.default_rng(nx + 31 * ny + 1009 * nz)
    v = rng.uniform(0, 1, (nz, ny, nx)).astype(np.float32)
    if field == "few":
        v *= np.float32(0.5)
        v[nz - 1, ny - 1, nx - 3] = v[0, 0, 0] = 0.9
    elif field == "none":
        v *= np.float32(0.5)
    print(f"[wide] {nx}x{ny}x{nz} {field}", flush=True)
    ref = oracle_mod.FEResult(v, 0.7, nthreads=4)
    algo = m.FlyingEdgesAlgorithm(m.Image3D(v), 0.7)
    for _ in range(2):
        algo.run()
        _same(algo.moveOutput(), ref.points, ref.normals, ref.triangles)
    rows = algo.rows()
    for key in ("xl", "xr", "xcount", "ycount", "zcount"):
        assert np.array_equal(rows[key].astype(np.uint64), ref.rows[key]), key
    per_row = sum(rows[k].astype(np.uint64) for k in ("xcount", "ycount", "zcount"))
    assert np.array_equal(rows["voffset"], np.cumsum(per_row) - per_row)
    assert np.array_equal(rows["toffset"], np.cumsum(rows["tcount"].astype(np.uint64)) - rows["tcount"])
    mc = oracle_mod.MCResult(v, 0.7)
    for order, want in (("first_visit", (mc.points, mc.normals, mc.triangles)), ("edge", mc.edge_order())):
        h = m._MC(m.Image3D(v), 0.7, order=order)
        for _ in range(2):
            h.run()
            _same(h.mesh(), *want)


def test_wide_rows_many(oracle_mod):
    """65,550 rows of 4097 voxels, a few voxels of each 37th row above the isovalue: sixteen rows a block of
    k_mc_count, the last block of 14; a host with that many rows sees the whole mesh"""
    import torch

    import miniisosurface_amd as m
    nx, ny, nz = 4097, 6555, 10
    v = torch.zeros((nz, ny, nx), device="cuda")
    gen = torch.Generator(device="cuda")
    gen.manual_seed(7)
    at = torch.arange(5, ny * nz, 37, device="cuda")
    cols = torch.randint(0, nx, (at.numel(), 3), generator=gen, device="cuda")
    v.view(ny * nz, nx)[at[:, None], cols] = torch.rand(cols.shape, generator=gen, device="cuda") * 0.5 + 0.5
    torch.cuda.synchronize()
    host = v.cpu().numpy()
    print(f"[wide] {nx}x{ny}x{nz}", flush=True)
    mc = oracle_mod.MCResult(host, 0.4)
    h = m._MC(m.DeviceVolume.from_tensor(v), 0.4)
    for _ in range(2):
        h.run()
        _same(h.mesh(), mc.points, mc.normals, mc.triangles)
