"""GPU: pass 3 where its tiles meet -- row counts at a tile's end and one beside it, enough rows for tiles
of more than 1024 rows, rows long enough for 64-bit step sums -- through Flying Edges (offsets and
mesh), both Marching Cubes orders, slabs, and batches whose jobs start inside a tile: bit for bit
against the oracle."""
import numpy as np
import pytest

from helpers import bits_equal

pytestmark = pytest.mark.gpu

# nx, ny, nz; rows = ny * nz
SIZES = [(3, 341, 3), (5, 512, 2), (4, 205, 5), (33, 31, 33), (70, 1025, 2), (4, 2051, 513), (524290, 3, 2)]


def _volume(nx, ny, nz):
    return np.random.default_rng(nx + 31 * ny + 1009 * nz).uniform(0, 1, (nz, ny, nx)).astype(np.float32)


def _same(mesh, ref):
    assert mesh.points.shape == ref.points.shape and mesh.triangles.shape == ref.triangles.shape
    assert bits_equal(mesh.points, ref.points) and bits_equal(mesh.normals, ref.normals)
    assert bits_equal(mesh.triangles, ref.triangles)


@pytest.mark.parametrize("nx,ny,nz", SIZES)
def test_scan_tiles(oracle_mod, nx, ny, nz):
    import miniisosurface_amd as m
    print(f"[scan] {nx}x{ny}x{nz}", flush=True)
    v = _volume(nx, ny, nz)
    ref = oracle_mod.FEResult(v, 0.7, nthreads=4)
    algo = m.FlyingEdgesAlgorithm(m.Image3D(v), 0.7)
    for _ in range(2):      # the second run starts from the first one's tile sums
        algo.run()
        _same(algo.moveOutput(), ref)
    rows = algo.rows()
    per_row = sum(rows[k].astype(np.uint64) for k in ("xcount", "ycount", "zcount"))
    assert np.array_equal(rows["voffset"], np.cumsum(per_row) - per_row)
    assert np.array_equal(rows["toffset"], np.cumsum(rows["tcount"].astype(np.uint64)) - rows["tcount"])
    _same(m.flying_edges_slabs(m.Image3D(v), 0.7, max(1, nz // 3)), ref)
    mc = oracle_mod.MCResult(v, 0.7)
    _same(m.MarchingCubes(m.Image3D(v), 0.7), mc)
    p, n, t = mc.edge_order()
    edge = m.MarchingCubes(m.Image3D(v), 0.7, order="edge")
    assert bits_equal(edge.points, p) and bits_equal(edge.normals, n) and bits_equal(edge.triangles, t)


@pytest.mark.parametrize("launch", ["graphs", "fused"])
def test_batch_jobs_inside_tiles(oracle_mod, launch):
    import torch

    import miniisosurface_amd as m
    from miniisosurface_amd.batch import BatchExtraction
    dims = [(5, 37, 29), (70, 3, 2), (130, 41, 27), (3, 501, 2), (300, 7, 9), (64, 64, 17), (2, 2, 2), (900, 11, 5)]
    vols = [_volume(*d) for d in dims]
    b = BatchExtraction([(m.DeviceVolume.from_tensor(torch.from_numpy(v).cuda()), 0.6) for v in vols])
    b.set_launch(launch)
    refs = [oracle_mod.FEResult(v, 0.6, nthreads=2, want_debug=False) for v in vols]
    for _ in range(3):
        b.run()
        for j, ref in enumerate(refs):
            _same(b.mesh(j), ref)
