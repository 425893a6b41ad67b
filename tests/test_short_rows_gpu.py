"""GPU: pass 1 where rows are at most 256 voxels and a wavefront takes several -- rows that end on or beside
a word boundary, one voxel in the last word, row counts that leave the last wavefront some, one or no
rows, volumes whose last voxels fill no lane's eight -- alone and as jobs of a batch, in every block order
and launch, with one geometry or both: bit for bit against the oracle."""
import numpy as np
import pytest

from helpers import bits_equal

pytestmark = pytest.mark.gpu

PLACINGS = {"unit": [((1.0, 1.0, 1.0), (0.0, 0.0, 0.0))], "spaced": [((0.5, 0.75, 1.25), (-3.0, 4.0, 0.5))]}
PLACINGS["both"] = PLACINGS["unit"] + PLACINGS["spaced"]

# nx, ny, nz
SIZES = [(2, 67, 63), (63, 3, 5), (64, 91, 91), (65, 4, 4), (127, 128, 33), (128, 5, 13), (129, 47, 89), (191, 2, 9),
         (192, 65, 64), (193, 3, 7), (255, 91, 46), (256, 4, 4), (256, 130, 127), (257, 5, 4)]


def _volume(nx, ny, nz):
    return np.random.default_rng(nx * 10007 + ny * 101 + nz).uniform(0, 1, (nz, ny, nx)).astype(np.float32)


def _same(mesh, ref):
    assert mesh.points.shape == ref.points.shape and mesh.triangles.shape == ref.triangles.shape
    assert bits_equal(mesh.points, ref.points) and bits_equal(mesh.normals, ref.normals)
    assert bits_equal(mesh.triangles, ref.triangles)


@pytest.mark.parametrize("nx,ny,nz", SIZES)
def test_short_rows(oracle_mod, nx, ny, nz):
    import miniisosurface_amd as m
    print(f"[short] {nx}x{ny}x{nz}", flush=True)
    v = _volume(nx, ny, nz)
    _same(m.flying_edges(m.Image3D(v), 0.8), oracle_mod.FEResult(v, 0.8, nthreads=2, want_debug=False))


@pytest.mark.parametrize("placing", sorted(PLACINGS))
@pytest.mark.parametrize("order", ["dispatch", "xcd"])
@pytest.mark.parametrize("launch", ["graphs", "fused"])
def test_short_row_jobs(oracle_mod, placing, order, launch):
    import torch

    import miniisosurface_amd as m
    from miniisosurface_amd.batch import BatchExtraction
    print(f"[jobs] {placing} {order} {launch}", flush=True)
    vols = [_volume(*d) for d in SIZES if d[0] * d[1] * d[2] < 300000]
    places = [PLACINGS[placing][j % len(PLACINGS[placing])] for j in range(len(vols))]
    devs = [m.DeviceVolume.from_tensor(torch.from_numpy(v).cuda(), *p) for v, p in zip(vols, places)]
    jobs = [(d, iso) for d in devs for iso in (0.8, 0.3)]
    refs = [oracle_mod.FEResult(v, iso, *p, nthreads=2, want_debug=False)
            for v, p in zip(vols, places) for iso in (0.8, 0.3)]
    b = BatchExtraction(jobs)
    b.set_queue_order(order)
    b.set_launch(launch)
    for blocks, chunk in ((4, 4), (1, 3)):
        b.set_tuning(blocks, chunk)
        for _ in range(2):
            b.run()
            for j, ref in enumerate(refs):
                _same(b.mesh(j), ref)
