"""GPU: pass 4 of the row kernels at the sizes where its pieces meet -- rows of a few voxels (no inner
origin), rows that end on or beside a 32- and a 64-voxel boundary (the next half's bit, the next
lane's), rows that fill all lanes, wavefronts with more origins and cells than one round lists, and
slabs that begin and end inside a wavefront's rows -- bit for bit against the oracle."""
import numpy as np
import pytest

from helpers import bits_equal

pytestmark = pytest.mark.gpu

SPACED = ((0.5, 0.75, 1.25), (-3.0, 4.0, 0.5))
UNIT = ((1.0, 1.0, 1.0), (0.0, 0.0, 0.0))

# nx, ny, nz, field
SIZES = [(2, 2, 2, "rand"), (3, 4, 3, "rand"), (4, 3, 4, "rand"), (5, 5, 5, "rand"), (31, 6, 5, "rand"),
         (32, 5, 6, "checker"), (33, 7, 4, "rand"), (63, 9, 5, "checker"), (64, 70, 4, "checker"), (65, 5, 7, "rand"),
         (96, 6, 5, "rand"), (128, 37, 5, "checker"), (256, 17, 5, "rand"), (257, 9, 4, "checker"),
         (512, 9, 4, "checker"), (1024, 5, 4, "rand"), (2048, 3, 4, "checker"), (4096, 3, 3, "rand")]


def _volume(nx, ny, nz, field):
    if field == "checker":     # every edge cut
        return (np.indices((nz, ny, nx)).sum(0) % 2).astype(np.float32)
    return np.random.default_rng(nx * 10007 + ny * 101 + nz).uniform(0, 1, (nz, ny, nx)).astype(np.float32)


@pytest.mark.parametrize("placing", [UNIT, SPACED], ids=["unit", "spaced"])
@pytest.mark.parametrize("nx,ny,nz,field", SIZES)
def test_emit_sizes(oracle_mod, nx, ny, nz, field, placing):
    import miniisosurface_amd as m
    print(f"[emit] {nx}x{ny}x{nz} {field} {placing}", flush=True)
    v = _volume(nx, ny, nz, field)
    sp, org = placing
    ref = oracle_mod.FEResult(v, 0.5, sp, org, nthreads=2, want_debug=False)
    image = m.Image3D(v, sp, org)
    for planes in (None, 1, 2):
        mesh = m.flying_edges(image, 0.5) if planes is None else m.flying_edges_slabs(image, 0.5, planes)
        assert mesh.points.shape == ref.points.shape and mesh.triangles.shape == ref.triangles.shape
        assert bits_equal(mesh.points, ref.points) and bits_equal(mesh.normals, ref.normals)
        assert bits_equal(mesh.triangles, ref.triangles)
