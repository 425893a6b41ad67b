"""GPU: the lane-row kernels where a small volume's rows take more lanes than their words (fewer rows per
wavefront) -- volumes just below and at the number of wavefronts that ends it, one row per wavefront, every
width of a row -- through Flying Edges, both Marching Cubes orders, slabs and a batch, against the oracle,
bit for bit."""
import numpy as np
import pytest

from helpers import bits_equal

pytestmark = pytest.mark.gpu

# nx, ny, nz
SIZES = [(40, 8, 4), (64, 128, 16), (64, 512, 255), (64, 512, 256), (63, 300, 70), (130, 200, 160), (200, 91, 46),
         (257, 64, 60), (700, 60, 30), (1025, 20, 20), (2050, 9, 8), (4096, 8, 8)]


def _volume(nx, ny, nz):
    rng = np.random.default_rng(nx * 7 + ny * 1013 + nz * 10007)
    return rng.uniform(0, 1, (nz, ny, nx)).astype(np.float32)


def _same(mesh, points, normals, triangles):
    assert mesh.points.shape == points.shape and mesh.triangles.shape == triangles.shape
    assert bits_equal(mesh.points, points) and bits_equal(mesh.normals, normals)
    assert bits_equal(mesh.triangles, triangles)


@pytest.mark.parametrize("nx,ny,nz", SIZES)
def test_small_volume(oracle_mod, nx, ny, nz):
    import miniisosurface_amd as m
    print(f"[small] {nx}x{ny}x{nz}", flush=True)
    v, iso = _volume(nx, ny, nz), 0.85
    ref = oracle_mod.FEResult(v, iso, nthreads=4, want_debug=False)
    _same(m.flying_edges(m.Image3D(v), iso), ref.points, ref.normals, ref.triangles)
    whole = m.flying_edges_slabs(m.Image3D(v), iso, max(1, nz // 3))
    _same(whole, ref.points, ref.normals, ref.triangles)
    mc = oracle_mod.MCResult(v, iso)
    _same(m.MarchingCubes(m.Image3D(v), iso), mc.points, mc.normals, mc.triangles)
    _same(m.MarchingCubes(m.Image3D(v), iso, order="edge"), *mc.edge_order())


@pytest.mark.parametrize("count", [1, 3, len(SIZES)])
def test_small_batch(oracle_mod, count):
    import torch

    import miniisosurface_amd as m
    from miniisosurface_amd.batch import BatchExtraction
    print(f"[small batch] {count}", flush=True)
    vols = [_volume(nx, ny, nz) for nx, ny, nz in sorted(SIZES, key=np.prod)[:count]]
    b = BatchExtraction([(m.DeviceVolume.from_tensor(torch.from_numpy(v).cuda()), 0.85) for v in vols])
    for order in ("dispatch", "xcd"):
        b.set_queue_order(order)
        b.run()
        for j, v in enumerate(vols):
            ref = oracle_mod.FEResult(v, 0.85, nthreads=4, want_debug=False)
            _same(b.mesh(j), ref.points, ref.normals, ref.triangles)
