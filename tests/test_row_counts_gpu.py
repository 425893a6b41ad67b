"""GPU: pass 2's per-row counts and trims -- rows of one to 64 words (every number of lanes a row takes),
the last word full, with one voxel and on either side of its middle, row counts that leave the last wavefront
part empty, signs that cut nearly every edge, few edges, and fill whole rows or all but their ends --
against the oracle, bit for bit."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

# nx, ny, nz
SIZES = [(2, 5, 3), (31, 70, 4), (33, 9, 11), (64, 66, 3), (65, 33, 5), (96, 7, 9), (97, 7, 9), (128, 5, 5),
         (129, 3, 21), (300, 4, 7), (512, 5, 5), (545, 3, 4), (1000, 4, 4), (1024, 3, 5), (1025, 2, 4), (1600, 3, 3),
         (2048, 2, 3), (2081, 3, 3), (4033, 2, 3), (4096, 3, 2)]


def _fields(nx, ny, nz):
    rng = np.random.default_rng(nx + 131 * ny + 1009 * nz)
    noise = rng.uniform(0, 1, (nz, ny, nx)).astype(np.float32)
    yield "half", noise
    yield "sparse", noise * noise * noise * np.float32(0.52)
    full = np.ones_like(noise)
    full[:, :, 0] = noise[:, :, 0]
    full[:, :, -1] = noise[:, :, -1]
    yield "full but its ends", full
    # body diagonals below, the other corners above: the two-corner rings and their complements
    k, j, i = np.meshgrid(np.arange(nz), np.arange(ny), np.arange(nx), indexing="ij")
    yield "rings", np.where((i + j + k) % 3 == 0, np.float32(0), np.float32(1)) + noise * np.float32(0.25)


@pytest.mark.parametrize("nx,ny,nz", SIZES)
def test_row_counts(oracle_mod, nx, ny, nz):
    import miniisosurface_amd as m
    for name, v in _fields(nx, ny, nz):
        print(f"[rows] {nx}x{ny}x{nz} {name}", flush=True)
        algo = m.FlyingEdgesAlgorithm(m.Image3D(v), 0.5)
        algo.run()
        rows = algo.rows()
        ref = oracle_mod.FEResult(v, 0.5, nthreads=2).rows
        for key in ("xl", "xr", "xcount", "ycount", "zcount"):
            assert np.array_equal(rows[key].astype(np.uint64), ref[key]), (name, key)
        cells = [j + ny * k for k in range(nz - 1) for j in range(ny - 1)]
        assert np.array_equal(rows["tcount"][cells].astype(np.uint64), ref["tcount"]), name
        assert int(rows["tcount"].sum()) == int(ref["tcount"].sum()), name
