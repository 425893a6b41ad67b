"""GPU: a Marching Cubes handle run again after its device volume has changed -- the same size of mesh, a
smaller one, none, a larger one than its buffers hold -- in both vertex orders, with unit and general
geometry, also where the order changes between runs: every run bit for bit against the oracle."""
import numpy as np
import pytest

from helpers import bits_equal

pytestmark = pytest.mark.gpu

PLACINGS = [((1.0, 1.0, 1.0), (0.0, 0.0, 0.0)), ((0.5, 0.75, 1.25), (-3.0, 4.0, 0.5))]
# nx, ny, nz: a few words per row and whole wavefronts; one word; a row per wavefront
SIZES = [(130, 37, 21), (33, 9, 70), (2100, 5, 4)]


@pytest.mark.parametrize("placing", PLACINGS, ids=["unit", "spaced"])
@pytest.mark.parametrize("nx,ny,nz", SIZES)
def test_mc_rerun(oracle_mod, nx, ny, nz, placing):
    import torch

    import miniisosurface_amd as m
    sp, org = placing
    rng = np.random.default_rng(nx + ny + nz)
    dev = torch.zeros((nz, ny, nx), dtype=torch.float32, device="cuda")
    mc = m._MC(m.DeviceVolume.from_tensor(dev, sp, org), 0.5)
    low = 0.5 + 0.4 * np.sin(np.arange(nx) / 5).astype(np.float32) * np.ones((nz, ny, 1), np.float32)
    noise = rng.uniform(0, 1, (nz, ny, nx)).astype(np.float32)
    for step, (field, order) in enumerate([(low, "first_visit"), (low, "first_visit"), (noise, "first_visit"),
                                           (noise, "edge"), (0 * low, "edge"), (low, "edge"), (noise, "first_visit"),
                                           (0 * low, "first_visit"), (1 - noise, "edge"), (low, "first_visit")]):
        print(f"[mc] {nx}x{ny}x{nz} {placing} step {step}", flush=True)
        dev.copy_(torch.from_numpy(np.ascontiguousarray(field)))
        torch.cuda.synchronize()
        mc.set_order(order)
        mc.run()
        mesh = mc.mesh()
        ref = oracle_mod.MCResult(np.ascontiguousarray(field), 0.5, sp, org)
        p, n, t = (ref.points, ref.normals, ref.triangles) if order == "first_visit" else ref.edge_order()
        assert mesh.points.shape == p.shape and mesh.triangles.shape == t.shape
        assert bits_equal(mesh.points, p) and bits_equal(mesh.normals, n) and bits_equal(mesh.triangles, t)
