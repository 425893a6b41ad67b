"""GPU: handles without a caller's stream, whose streams and pinned pages pass from one to the next -- fewer
alive at once than are kept, as many, and more, made and destroyed in changing order, volumes of several sizes
and of no cells, from one thread and from several: every mesh bit for bit against the oracle."""
import threading

import numpy as np
import pytest

from helpers import bits_equal

pytestmark = pytest.mark.gpu

SIZES = [(33, 21, 17), (1, 5, 4), (64, 64, 9), (130, 7, 11), (5, 300, 3)]     # nx, ny, nz


def _volume(q):
    nx, ny, nz = SIZES[q % len(SIZES)]
    return np.random.default_rng(q).uniform(0, 1, (nz, ny, nx)).astype(np.float32)


def _check(mesh, ref):
    assert mesh.points.shape == ref.points.shape and mesh.triangles.shape == ref.triangles.shape
    assert bits_equal(mesh.points, ref.points) and bits_equal(mesh.normals, ref.normals)
    assert bits_equal(mesh.triangles, ref.triangles)


def _turns(refs, alive, seed):
    import miniisosurface_amd as m
    rng = np.random.default_rng(seed)
    held = []
    for turn in range(24):
        q = int(rng.integers(len(refs)))
        kind = turn % 3
        h = m._MC(m.Image3D(_volume(q)), 0.5) if kind == 2 else m.FlyingEdgesAlgorithm(m.Image3D(_volume(q)), 0.5)
        held.append((h, kind, q))
        rng.shuffle(held)
        while len(held) >= alive:
            h, kind, q = held.pop()
            h.run()
            _check(h.mesh() if kind == 2 else h.moveOutput(), refs[q][kind == 2])
            del h


@pytest.mark.parametrize("alive", [1, 4, 7])
def test_handles_in_turn(oracle_mod, alive):
    refs = [(oracle_mod.FEResult(_volume(q), 0.5, want_debug=False), oracle_mod.MCResult(_volume(q), 0.5))
            for q in range(2 * len(SIZES))]
    print(f"[handles] {alive} alive, one thread", flush=True)
    _turns(refs, alive, alive)
    errors = []

    def work(seed):
        try:
            _turns(refs, alive, seed)
        except BaseException as e:
            errors.append(e)

    print(f"[handles] {alive} alive each, three threads", flush=True)
    threads = [threading.Thread(target=work, args=(100 + t,)) for t in range(3)]
    for t in threads:
        t.start()
    for t in threads:
        t.join()
    assert not errors, errors
