"""The work that a user of this package has it do, as timing cases.

listed() names the cases, draw(rng) gives others of the same ranges, prepare(case, seed) makes what
a program holds before the call (a volume, and the handle it keeps), run(state) is one pass through
the public entry points, work(case) its compulsory bytes and operations, exact(case, seed) the
points and normals in 64 bits from torch alone.

The kinds of a case:
  handle       FlyingEdgesAlgorithm kept on a device volume: run(), the mesh left on the device
  noalloc      miso_fe_run_noalloc into buffers of the caller (the call for loops that may not allocate)
  host         flying_edges() on a host volume, whole call: copy in, four passes, copy the mesh out
  mc_first     Marching Cubes kept on a device volume, the serial reference's vertex order
  mc_edge      the same in global edge order
  batch_mixed  BatchExtraction of many small volumes of mixed sizes, each with its own isovalue
  batch_iso    BatchExtraction of one volume at many isovalues
  slabs        FlyingEdgesSlabs over a device volume, every part copied off as it comes
  serve        IsosurfaceServer: requests that wait together, delivered on the device
"""
from __future__ import annotations

import ctypes
import math

import numpy as np
import torch

import miniisosurface_amd as miso
from miniisosurface_amd import serve, synth
from miniisosurface_amd._lib import check, lib
from miniisosurface_amd.batch import BatchExtraction

SPACED = ((0.5, 0.75, 1.25), (-10.0, 4.0, 0.5))     # spacing and origin of a case with "spaced"
UNIT = ((1.0, 1.0, 1.0), (0.0, 0.0, 0.0))


def listed():
    return [
        # the smallest call: a volume of a tight loop or a tile, where launches and waits count
        dict(name="noalloc_64", kind="noalloc", field="gaussians", nx=64, ny=64, nz=64, iso=0.5, spaced=False),
        # the miniapp's own run, a 128^3 Gaussian volume in host memory, mesh back in host memory
        dict(name="host_128", kind="host", field="gaussians", nx=128, ny=128, nz=128, iso=0.5, spaced=False),
        # an ordinary scan: ragged rows, unequal spacing, an origin off zero
        dict(name="handle_ragged", kind="handle", field="noise", nx=333, ny=257, nz=190, iso=0.5, spaced=True),
        # a dense surface at an ordinary size
        dict(name="handle_gyroid_512", kind="handle", field="gyroid", nx=512, ny=512, nz=512, iso=0.0, spaced=False),
        # the benchmark's volume, the largest
        dict(name="handle_noise_1024", kind="handle", field="noise", nx=1024, ny=1024, nz=1024, iso=0.5,
             spaced=False),
        # a high isovalue in a large volume whose sides are no powers of two: little surface
        dict(name="handle_sparse", kind="handle", field="noise", nx=1000, ny=900, nz=700, iso=0.8, spaced=False),
        # Marching Cubes in the reference's order at an ordinary size
        dict(name="mc_first_512", kind="mc_first", field="gyroid", nx=512, ny=512, nz=512, iso=0.0, spaced=False),
        # Marching Cubes without duplicates (edge order), ragged and spaced
        dict(name="mc_edge_ragged", kind="mc_edge", field="noise", nx=400, ny=300, nz=280, iso=0.45, spaced=True),
        # many small volumes of mixed sizes, each with its own isovalue
        dict(name="batch_mixed_256", kind="batch_mixed", count=256, lo=32, hi=256),
        # one volume at many isovalues (a sweep)
        dict(name="batch_sweep_16", kind="batch_iso", field="gyroid", nx=256, ny=256, nz=256, count=16, spaced=False),
        # a volume cut into slabs to bound the output held at once
        dict(name="slabs_500", kind="slabs", field="noise", nx=500, ny=480, nz=420, iso=0.5, spaced=False, planes=100),
        # a serving step: requests on resident volumes that wait together
        dict(name="serve_12", kind="serve", count=12, pool=6),
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    most = work(next(c for c in listed() if c["name"] == "handle_noise_1024"))["bytes"]
    while True:
        kind = rng.choice(["noalloc", "host", "handle", "handle", "handle", "mc_first", "mc_edge", "batch_mixed",
                           "batch_iso", "slabs", "serve"])
        if kind == "batch_mixed":
            return dict(kind=kind, count=_log_int(rng, 32, 256), lo=32, hi=_log_int(rng, 96, 256))
        if kind == "serve":
            return dict(kind=kind, count=rng.randint(2, 16), pool=rng.randint(2, 8))
        hi = {"noalloc": 512, "host": 192, "handle": 1024, "mc_first": 512, "mc_edge": 512, "batch_iso": 256,
              "slabs": 512}[kind]
        case = dict(kind=kind, field=rng.choice(["gaussians", "noise", "gyroid"]), nx=_log_int(rng, 48, hi),
                    ny=_log_int(rng, 48, hi), nz=_log_int(rng, 48, hi), spaced=rng.random() < 0.4)
        if kind == "batch_iso":
            case["count"] = rng.randint(4, 16)
        else:
            case["iso"] = {"gaussians": rng.uniform(0.2, 0.8), "noise": rng.uniform(0.35, 0.9),
                           "gyroid": rng.uniform(-0.6, 0.6)}[case["field"]]
        if kind == "slabs":
            case["planes"] = _log_int(rng, 16, 128)
        if work(case)["bytes"] < 0.8 * most:
            return case


# ---------------------------------------------------------------------------- inputs
#
# A case's field is fixed; the seed mirrors it along x and y and moves every value within the
# isovalues around it. So volumes, points, normals and ids are other ones with another seed, while
# the number of vertices and triangles, which a mirror leaves as it is, belongs to the case.

FIELD_SEED = 0


def _vary(v, isos, seed):
    """The volume of `seed`: v mirrored, and its values moved by up to a quarter of their distance to the
    nearest isovalue, never onto the other side of one."""
    rng = np.random.default_rng(seed)
    v = v.flip([q for q in (1, 2) if rng.random() < 0.5]).contiguous()
    gen = torch.Generator(device=v.device)
    gen.manual_seed(seed)
    levels = torch.tensor(sorted(set(isos)), dtype=torch.float32, device=v.device)
    inf = torch.full((1,), math.inf, device=v.device)
    below, above = torch.cat([-inf, levels]), torch.cat([levels, inf])
    step = max(1, (1 << 26) // (v.shape[1] * v.shape[2]))
    for c in v.split(step):
        band = torch.bucketize(c, levels, right=True, out_int32=True)
        room = torch.minimum(c - below[band], above[band] - c)
        new = c + room * (torch.rand(c.shape, generator=gen, device=c.device) - 0.5) * 0.5
        c.copy_(torch.where(torch.bucketize(new, levels, right=True, out_int32=True) == band, new, c))
    return v


def _gyroid(nx, ny, nz, seed):
    """sin x cos y + sin y cos z + sin z cos x, 8 periods along x, and noise of 0.05 (synth.gyroid
    with the noise drawn on the GPU)"""
    dev = torch.device("cuda")
    k = 2.0 * math.pi * 8 / nx
    gen = torch.Generator(device=dev)
    gen.manual_seed(seed)
    x, y, z = (torch.arange(n, dtype=torch.float32, device=dev) * k for n in (nx, ny, nz))
    out = torch.rand((nz, ny, nx), generator=gen, dtype=torch.float32, device=dev).mul_(0.1).sub_(0.05)
    out += torch.sin(x)[None, None, :] * torch.cos(y)[None, :, None]
    out += torch.sin(y)[None, :, None] * torch.cos(z)[:, None, None]
    out += torch.sin(z)[:, None, None] * torch.cos(x)[None, None, :]
    return out


def _volume(case, seed):
    """the case's volume as a device tensor (nz, ny, nx)"""
    dims = (case["nx"], case["ny"], case["nz"])
    isos = _sweep(case) if case["kind"] == "batch_iso" else [float(np.float32(case["iso"]))]
    if case["field"] == "gyroid":
        v = _gyroid(*dims, FIELD_SEED)
    elif case["field"] == "noise":
        v = synth.value_noise(dims, FIELD_SEED, device="cuda")
    else:
        scale = min(dims) / 128.0
        v = synth.gaussians(dims, 4, FIELD_SEED, sigma_range=(8.0 * scale, 20.0 * scale), device="cuda")
    return _vary(v, isos, seed)


def _placing(case):
    return SPACED if case.get("spaced") else UNIT


def _sweep(case):
    """the isovalues of a sweep, over the middle of the field's range"""
    lo, hi = {"gaussians": (0.1, 0.9), "noise": (0.3, 0.7), "gyroid": (-1.0, 1.0)}[case["field"]]
    return [float(np.float32(lo + (hi - lo) * q / (case["count"] - 1))) for q in range(case["count"])]


SERVE_DIMS = (64, 96, 128, 160, 192, 256)


def _pool(case, seed):
    """a serving pool of volumes and the (volume index, isovalue) of its requests"""
    rng = np.random.default_rng(FIELD_SEED)
    pool = []
    for q in range(case["pool"]):
        n = SERVE_DIMS[q % len(SERVE_DIMS)]
        s = int(rng.integers(1 << 30))
        v = _gyroid(n, n, n, s) if q % 2 else synth.gaussians(n, 4, s, sigma_range=(n / 16.0, n / 6.4), device="cuda")
        pool.append((v, (float(v.min()), float(v.max()))))
    asked = []
    for q in range(case["count"]):
        p = q % case["pool"]
        lo, hi = pool[p][1]
        asked.append((p, float(np.float32(lo + (hi - lo) * rng.uniform(0.2, 0.8)))))
    isos = [[iso for p, iso in asked if p == q] or [0.5] for q in range(case["pool"])]
    return [_vary(v, isos[q], seed + q) for q, (v, _) in enumerate(pool)], asked


def _mixed(case, seed):
    """the volumes of a mixed batch, each with its isovalue"""
    jobs = synth.batch_volumes(case["count"], FIELD_SEED, case["lo"], case["hi"], device="cuda")
    return [(_vary(v, [float(np.float32(iso))], seed + q), float(np.float32(iso))) for q, (v, iso) in enumerate(jobs)]


def prepare(case, seed):
    kind = case["kind"]
    if kind == "batch_mixed":
        jobs = _mixed(case, seed)
        torch.cuda.synchronize()
        return dict(kind=kind, b=BatchExtraction([(miso.DeviceVolume.from_tensor(v), iso) for v, iso in jobs]))
    if kind == "serve":
        pool, asked = _pool(case, seed)
        srv = serve.IsosurfaceServer([miso.DeviceVolume.from_tensor(v) for v in pool], budget_bytes=20e9,
                                     deliver="device")
        return dict(kind=kind, srv=srv, asked=asked)
    t = _volume(case, seed)
    sp, org = _placing(case)
    if kind == "host":
        return dict(kind=kind, image=miso.Image3D(t.cpu().numpy(), sp, org), iso=case["iso"])
    vol = miso.DeviceVolume.from_tensor(t, sp, org)
    torch.cuda.synchronize()
    if kind == "batch_iso":
        return dict(kind=kind, b=BatchExtraction([(vol, iso) for iso in _sweep(case)]))
    if kind == "slabs":
        return dict(kind=kind, s=miso.FlyingEdgesSlabs(vol, case["iso"], case["planes"]), iso=case["iso"])
    if kind in ("mc_first", "mc_edge"):
        return dict(kind=kind, mc=miso._MC(vol, case["iso"], order="edge" if kind == "mc_edge" else "first_visit"))
    if kind == "noalloc":
        # buffers for the mesh, sized by counting once as a program with a loop over such volumes does
        nv, nt = ctypes.c_uint64(), ctypes.c_uint64()
        st = miso._volume_struct(vol)[0]
        lib().miso_fe_run_noalloc(ctypes.byref(st), case["iso"], None, None, None, None, 0, 0, ctypes.byref(nv),
                                  ctypes.byref(nt))
        cv, ct = nv.value + nv.value // 4 + 64, nt.value + nt.value // 4 + 64
        buf = (torch.empty((cv, 3), device="cuda"), torch.empty((cv, 3), device="cuda"),
               torch.empty((ct, 3), dtype=torch.int32, device="cuda"))
        return dict(kind=kind, vol=vol, st=st, iso=case["iso"], buf=buf, cap=(cv, ct))
    return dict(kind=kind, algo=miso.FlyingEdgesAlgorithm(vol, case["iso"]))


# ---------------------------------------------------------------------------- a pass

class _Device:
    """Device memory of a handle as torch sees it; keeps the handle."""

    def __init__(self, owner, ptr, shape, typestr):
        self.owner = owner
        self.__cuda_array_interface__ = {"shape": shape, "typestr": typestr, "data": (ptr, False), "version": 2}


def _tensor(owner, ptr, n, typestr):
    if not n:
        return torch.empty((0, 3), dtype={"<f4": torch.float32, "<i4": torch.int32, "<i8": torch.int64}[typestr],
                           device="cuda")
    return torch.as_tensor(_Device(owner, ptr, (n, 3), typestr), device="cuda")


def run(state):
    kind = state["kind"]
    if kind == "handle":
        algo = state["algo"]
        algo.run()
        p, n, t, bits, v, nt = algo.device_output()
        return _tensor(algo, p, v, "<f4"), _tensor(algo, n, v, "<f4"), _tensor(algo, t, nt, "<i%d" % (bits // 8))
    if kind == "noalloc":
        nv, nt = ctypes.c_uint64(), ctypes.c_uint64()
        p, n, t = state["buf"]
        check(lib().miso_fe_run_noalloc(ctypes.byref(state["st"]), state["iso"], None, p.data_ptr(), n.data_ptr(),
                                        t.data_ptr(), *state["cap"], ctypes.byref(nv), ctypes.byref(nt)), "noalloc")
        return p[:nv.value], n[:nv.value], t[:nt.value]
    if kind == "host":
        mesh = miso.flying_edges(state["image"], state["iso"])
        return mesh.points, mesh.normals, mesh.triangles
    if kind in ("mc_first", "mc_edge"):
        mc = state["mc"]
        mc.run()
        v, nt = mc.counts()
        p, n, t = ctypes.c_void_p(), ctypes.c_void_p(), ctypes.c_void_p()
        bits = ctypes.c_int()
        check(lib().miso_mc_device_output(mc._h, ctypes.byref(p), ctypes.byref(n), ctypes.byref(t),
                                          ctypes.byref(bits)), "output")
        return (_tensor(mc, p.value, v, "<f4"), _tensor(mc, n.value, v, "<f4"),
                _tensor(mc, t.value, nt, "<i%d" % (bits.value // 8)))
    if kind in ("batch_mixed", "batch_iso"):
        b = state["b"].run()
        v, nt = b.totals()
        p, n, t = b.device_output(0)       # the jobs' meshes lie one after another in one buffer
        return _tensor(b, p, v, "<f4"), _tensor(b, n, v, "<f4"), _tensor(b, t, nt, "<i4")
    if kind == "slabs":
        s = state["s"]
        s.restart(state["iso"])
        parts = []
        while s.next():
            q = s.part()
            p, n, t = s.device_part()
            parts.append((_tensor(s, p, q["nverts"], "<f4").clone(), _tensor(s, n, q["nverts"], "<f4").clone(),
                          _tensor(s, t, q["ntris"], "<i8").clone()))
            # the parts are reused by the library's own streams
            torch.cuda.current_stream().synchronize()
        return parts
    done = state["srv"].run([serve.Request(volume=p, iso=iso, rid=q) for q, (p, iso) in enumerate(state["asked"])])
    out = []
    for r in sorted(done, key=lambda r: r.rid):
        out.append(r.result)
        r.release()
    return out


# ---------------------------------------------------------------------------- work

def _cut_edges(case):
    """About the vertices of the mesh: the surface's cut edges, from the fields' mean crossings of a grid
    line (measured at 512^3 and 1024^3; a triangle mesh of a closed surface has about twice as many triangles)."""
    nx, ny, nz = case["nx"], case["ny"], case["nz"]
    iso = case.get("iso")
    if case["field"] == "gyroid":
        spread = 1.0 if iso is None else max(0.0, 1.0 - abs(iso) / 1.5)
        return 1.717 * 8 / nx * 3 * nx * ny * nz * spread
    if case["field"] == "noise":
        per_line = 12.5 * math.exp(-(((0.5 if iso is None else iso) - 0.5) / 0.13) ** 2 / 2)
        return per_line * (ny * nz + nx * nz + nx * ny)
    s2 = 208.0 * (min(nx, ny, nz) / 128.0) ** 2
    return 0.5 * 4 * 6 * math.pi * 2.0 * math.log(1.0 / (iso or 0.5)) * s2


def work(case):
    """Bytes: the volume read once (4 a voxel), 24 a vertex (point and normal), 12 a triangle of 32-bit
    ids (24 where they are 64-bit). Operations: a comparison a voxel and about 40 a vertex."""
    kind = case["kind"]
    if kind == "batch_mixed":
        side = (case["hi"] - case["lo"]) / math.log(case["hi"] / case["lo"])
        n, v = case["count"] * side ** 3, case["count"] * 0.9 * side ** 2
    elif kind == "serve":
        n = v = 0.0
        for q in range(case["count"]):
            side = SERVE_DIMS[(q % case["pool"]) % len(SERVE_DIMS)]
            n += side ** 3
            v += (20.0 if (q % case["pool"]) % 2 else 0.6) * side ** 2
    else:
        n, v = float(case["nx"] * case["ny"] * case["nz"]), _cut_edges(case)
        v *= case.get("count", 1)
    ids = 8 if kind in ("slabs", "host") else 4
    return {"bytes": 4.0 * n + 24.0 * v + 3 * ids * 2.0 * v, "flops": n + 40.0 * v}


# ---------------------------------------------------------------------------- the values in 64 bits

def _gradient(d, pos, axis, spacing):
    """-(central difference) along `axis` (0 x, 1 y, 2 z) at grid positions pos = (i, j, k), one-sided at the faces"""
    n = d.shape[2 - axis]
    up, lo = [p.clone() for p in pos], [p.clone() for p in pos]
    up[axis] = torch.clamp(pos[axis] + 1, max=n - 1)
    lo[axis] = torch.clamp(pos[axis] - 1, min=0)
    run_ = (up[axis] - lo[axis]).double() * spacing
    return (d[lo[2], lo[1], lo[0]].double() - d[up[2], up[1], up[0]].double()) / run_


def _vertices(d, iso, sp, org, axes=(0, 1, 2)):
    """Points and normals of the cut edges along `axes` in 64 bits, rows (k, j) in order and within a row
    by axis, then by i; and the plane k of each."""
    nz, ny, nx = d.shape
    iso = float(np.float32(iso))
    sp, org = [float(np.float32(s)) for s in sp], [float(np.float32(o)) for o in org]
    points, normals, planes = [], [], []
    step = max(1, (1 << 27) // (nx * ny))
    for k0 in range(0, nz, step):
        k1 = min(nz, k0 + step)
        s = d[k0:min(nz, k1 + 1)] >= iso
        m = s[:k1 - k0]
        cut = torch.zeros((k1 - k0, ny, len(axes), nx), dtype=torch.bool, device=d.device)
        for q, a in enumerate(axes):
            if a == 0:
                cut[:, :, q, :-1] = m[:, :, 1:] ^ m[:, :, :-1]
            elif a == 1:
                cut[:, :-1, q] = m[:, 1:] ^ m[:, :-1]
            else:
                cut[:s.shape[0] - 1, :, q] = s[1:] ^ s[:-1]
        k, j, q, i = cut.nonzero(as_tuple=True)
        k = k + k0
        axis = torch.tensor(axes, device=d.device)[q]
        a = [i, j, k]
        b = [p + (axis == c) for c, p in enumerate(a)]
        va, vb = d[k, j, i].double(), d[b[2], b[1], b[0]].double()
        w = (iso - va) / (vb - va)
        points.append(torch.stack([org[c] + (a[c].double() + w * (axis == c)) * sp[c] for c in range(3)], 1))
        ga = torch.stack([_gradient(d, a, c, sp[c]) for c in range(3)], 1)
        gb = torch.stack([_gradient(d, b, c, sp[c]) for c in range(3)], 1)
        normals.append(ga + w[:, None] * (gb - ga))
        planes.append(k)
    return torch.cat(points), torch.cat(normals), torch.cat(planes)


def exact(case, seed):
    """Points and normals; the triangles are whole numbers and stay equal. First-visit Marching Cubes has
    its vertices in the order of the case table's triangles, which only the library holds: no value here."""
    kind = case["kind"]
    if kind == "mc_first":
        return None
    if kind == "batch_mixed":
        jobs = [(v, iso, *UNIT) for v, iso in _mixed(case, seed)]
    elif kind == "serve":
        pool, asked = _pool(case, seed)
        jobs = [(pool[p], iso, *UNIT) for p, iso in asked]
    elif kind == "batch_iso":
        v = _volume(case, seed)
        jobs = [(v, iso, *_placing(case)) for iso in _sweep(case)]
    else:
        jobs = [(_volume(case, seed), case["iso"], *_placing(case))]
    if kind == "mc_edge":
        got = [_vertices(*jobs[0], axes=(a,)) for a in (0, 1, 2)]
        return torch.cat([g[0] for g in got]), torch.cat([g[1] for g in got]), None
    if kind == "serve":
        return [(*_vertices(*job)[:2], None) for job in jobs]
    if kind == "slabs":
        p, n, k = _vertices(*jobs[0])
        ends = [int((k < min(k1, case["nz"])).sum()) for k1 in
                range(0, case["nz"] + case["planes"], case["planes"])]
        return [(p[u:v], n[u:v], None) for u, v in zip(ends, ends[1:])]
    got = [_vertices(*job)[:2] for job in jobs]
    p, n = torch.cat([g[0] for g in got]), torch.cat([g[1] for g in got])
    if kind == "host":
        return p.cpu().numpy(), n.cpu().numpy(), None
    return p, n, None
