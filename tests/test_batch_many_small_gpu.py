"""GPU: a batch of many more jobs than blocks, each of one or a few items (2 to 9 voxels a side): the meshes of
the graph launch against the oracle for some jobs, and of the fused launch, whose blocks go from chunk to chunk
across many jobs, against the graph launch's, byte for byte, with chunks of one, four and sixteen items in both
queue orders. And the fused launch takes at most four times as long: beside the same passes it has three grid
barriers and fewer blocks, twice the time when measured; eight times if a block walks to its chunks job by job."""
import numpy as np
import pytest

from helpers import bits_equal

pytestmark = pytest.mark.gpu

N = 20000


def _output(b):
    import torch
    v, t = b.totals()
    p, n, tri = b.device_output(0)

    class Mem:
        def __init__(self, ptr, count, typestr):
            self.__cuda_array_interface__ = {"shape": (3 * count,), "typestr": typestr, "data": (ptr, False), "version": 2}

    return [torch.as_tensor(Mem(*a), device="cuda").clone() for a in ((p, v, "<i4"), (n, v, "<i4"), (tri, t, "<i4"))]


def test_many_small_jobs(oracle_mod):
    import torch

    from miniisosurface_amd import DeviceVolume
    from miniisosurface_amd.batch import BatchExtraction
    rng = np.random.default_rng(11)
    dims = rng.integers(2, 10, size=(N, 3))
    dims[::500] = (70, 9, 40)                     # some jobs of several items among them
    at = np.concatenate([[0], np.cumsum(dims.prod(1))])
    host = rng.uniform(0, 1, int(at[-1])).astype(np.float32)
    flat = torch.from_numpy(host).cuda()
    isos = rng.uniform(0.3, 0.95, N).astype(np.float32)
    b = BatchExtraction([(DeviceVolume.from_tensor(flat[at[q]:at[q + 1]].view(*map(int, dims[q]))), float(isos[q]))
                         for q in range(N)])

    def timed():
        return min(b.run().time_ms() for _ in range(12))

    b.set_launch("graphs")
    graphs = timed()
    ref = _output(b)
    for q in list(range(0, N, 500)) + list(range(1, N, 701)):
        r = oracle_mod.FEResult(host[at[q]:at[q + 1]].reshape(dims[q]), float(isos[q]), want_debug=False)
        got = b.mesh(q)
        assert bits_equal(got.points, r.points) and bits_equal(got.normals, r.normals), q
        assert np.array_equal(got.triangles, r.triangles), q
    b.set_launch("fused")
    fused = timed()
    print(f"[many small] graphs {graphs:.3f} ms, fused {fused:.3f} ms", flush=True)
    for chunk in (4, 1, 16):
        b.set_tuning(b.tuning()[0], chunk)
        for order in ("dispatch", "xcd"):
            b.set_queue_order(order)
            b.run()                               # sizes nothing new, captures the graphs again
            b.run()
            for a, c in zip(ref, _output(b)):
                assert torch.equal(a, c), (chunk, order)
    b.close()
    assert fused < 4 * graphs, (graphs, fused)
