"""GPU: miso_fe_run_noalloc at the last size its 64 MiB of row state take, for rows of one, two and eleven
mask words: the mesh of miso_fe_run, bit for bit; one more pair of rows is refused."""
import ctypes

import pytest

pytestmark = pytest.mark.gpu


# nx, ny: two planes of ny rows
@pytest.mark.parametrize("nx,ny", [(2, 698984), (65, 599136), (700, 262130)])
def test_noalloc_at_the_limit(nx, ny):
    import torch

    import miniisosurface_amd as m
    from miniisosurface_amd._lib import lib
    print(f"[noalloc limit] {nx}x{ny}x2", flush=True)
    gen = torch.Generator(device="cuda")
    gen.manual_seed(nx)
    flat = torch.rand(2 * (ny + 1) * nx, generator=gen, device="cuda")
    iso = 1.0 - 20000.0 / flat.numel()          # some 20,000 voxels above it

    def run(rows, pts, nrm, tri):
        vol = m.DeviceVolume.from_tensor(flat[:2 * rows * nx].view(2, rows, nx))
        st = m._volume_struct(vol)[0]
        nv, nt = ctypes.c_uint64(), ctypes.c_uint64()
        rc = lib().miso_fe_run_noalloc(ctypes.byref(st), ctypes.c_float(iso), None, pts.data_ptr(), nrm.data_ptr(),
                                       tri.data_ptr(), pts.shape[0], tri.shape[0], ctypes.byref(nv), ctypes.byref(nt))
        return rc, nv.value, nt.value

    cap = 200000
    bufs = [torch.empty((cap, 3), device="cuda"), torch.empty((cap, 3), device="cuda"),
            torch.empty((cap, 3), dtype=torch.int32, device="cuda")]
    torch.cuda.synchronize()
    rc, nv, nt = run(ny, *bufs)
    assert rc == 0, lib().miso_last_error()
    algo = m.FlyingEdgesAlgorithm(m.DeviceVolume.from_tensor(flat[:2 * ny * nx].view(2, ny, nx)), iso)
    algo.run()
    ref = algo.moveOutput()
    assert (nv, nt) == (ref.points.shape[0], ref.triangles.shape[0]) and nv > 1000
    got = [b[:n].cpu().numpy() for b, n in zip(bufs, (nv, nv, nt))]
    assert got[0].tobytes() == ref.points.tobytes() and got[1].tobytes() == ref.normals.tobytes()
    assert (got[2].astype("uint32") == ref.triangles).all()
    rc, _, _ = run(ny + 1, *bufs)
    assert rc == -3 and "scratch" in lib().miso_last_error().decode()
