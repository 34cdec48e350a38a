"""The calls whose speed is tracked, at the sizes that real use of the
accelerators has: what a renderer does per frame, per animation step and per
optimisation step, through the public Python classes.

A case is a dict of plain values with a "kind":

  tri     TriangleAccel over a heightfield: Traverse (rebuild: Build32 first)
  tet     TetraAccel over a jittered grid: Build32, then TraverseTetra with a
          vertex scalar (time-varying simulation data)
  sph     ParticleAccel over a Plummer sphere: Traverse (rebuild: Build32 first)
  ao      ParticleAccel: TraverseAnySorted over ambient-occlusion rays
  sol     SolidAccel over pyramids / prisms / hexahedra: TraverseSolid
  lin     LineAccel over random-walk polylines: TraverseLines
  scene   Scene (two-level) over rigidly placed triangle meshes: Trace
  march   Volume.march: the emission-absorption forward march
  train   volume.render and its backward: gradients of voxels and transfer
          function

Geometry, cameras and gradients are made on the GPU from the seed alone.
Rays come in 8x8 pixel tiles ("tile") or in row order ("row"); frames whose
sides are no multiples of 8 end in ragged tiles.
"""
import math

import torch

from surface_amd import accel as A
from surface_amd import volume as V

DEV = "cuda"


def listed():
    return [
        # a shader's small ray queue on a small mesh (picking, probes): one
        # launch, latency only
        {"name": "tri_queue", "kind": "tri", "grid": 64, "w": 61, "h": 33, "order": "row",
         "view": "above", "rebuild": False},
        # a full frame of primary rays on a half-million triangle terrain, the
        # grid-512 heightfield of the benchmark
        {"name": "tri_frame", "kind": "tri", "grid": 512, "w": 1024, "h": 1024, "order": "tile",
         "view": "camera", "rebuild": False},
        # an animation step: a million deforming triangles rebuilt, then a
        # ragged preview frame
        {"name": "tri_rebuild", "kind": "tri", "grid": 725, "w": 333, "h": 251, "order": "tile",
         "view": "camera", "rebuild": True},
        # the benchmark's tetra step: 64^3 cells rebuilt and one frame with the
        # interpolated scalar
        {"name": "tet_step", "kind": "tet", "cells": 64, "w": 1024, "h": 1024, "order": "tile"},
        # the benchmark's particle set: 16 million spheres, 2048^2 primary rays
        {"name": "sph_frame", "kind": "sph", "count": 1 << 24, "w": 2048, "h": 2048,
         "order": "tile", "rebuild": False},
        # a particle simulation's step: 2 million spheres rebuilt, a preview frame
        {"name": "sph_step", "kind": "sph", "count": 2_000_003, "w": 512, "h": 384,
         "order": "tile", "rebuild": True},
        # ambient occlusion of a particle frame: incoherent short rays
        {"name": "sph_ao", "kind": "ao", "count": 4_000_000, "rays": 8_000_000, "bits": 30},
        # a frame over 64^3 hexahedra, the benchmark's solid set
        {"name": "hex_frame", "kind": "sol", "nv": 8, "cells": 64, "w": 768, "h": 768,
         "order": "tile"},
        # a frame over a million capped segments (streamlines, hair), rows of
        # pixels as a scanline renderer sends them
        {"name": "line_frame", "kind": "lin", "curves": 16384, "segs": 64, "w": 1000, "h": 750,
         "order": "row"},
        # two-level scene of instanced meshes, as a draw list makes it
        {"name": "scene_frame", "kind": "scene", "meshes": 24, "grid": 200, "w": 1280, "h": 720,
         "order": "tile"},
        # volume rendering: the benchmark's 256^3 volume, one frame
        {"name": "vol_frame", "kind": "march", "dim": 256, "w": 1024, "h": 1024, "tf": 256,
         "order": "tile"},
        # an optimisation step on a volume: forward and adjoint
        {"name": "vol_train", "kind": "train", "dim": 128, "w": 512, "h": 512, "tf": 256,
         "order": "tile"},
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["tri", "tri", "tet", "sph", "ao", "sol", "lin", "scene", "march", "train"])
    w, h = _log(rng, 40, 1024), _log(rng, 40, 1024)
    c = {"kind": kind, "w": w, "h": h, "order": rng.choice(["tile", "tile", "row"])}
    if kind == "tri":
        c.update(grid=_log(rng, 40, 725), view=rng.choice(["camera", "above"]),
                 rebuild=rng.random() < 0.4)
    elif kind == "tet":
        c.update(cells=_log(rng, 8, 64))
    elif kind == "sph":
        c.update(count=_log(rng, 2000, 1 << 22), rebuild=rng.random() < 0.4)
    elif kind == "ao":
        c = {"kind": kind, "count": _log(rng, 20_000, 4_000_000),
             "rays": _log(rng, 2000, 4_000_000), "bits": rng.choice([0, 15, 21, 30])}
    elif kind == "sol":
        c.update(nv=rng.choice([5, 6, 8]), cells=_log(rng, 12, 48))
    elif kind == "lin":
        c.update(curves=_log(rng, 40, 16384), segs=rng.randint(30, 64))
    elif kind == "scene":
        c.update(meshes=rng.randint(2, 40), grid=_log(rng, 40, 250))
    else:
        c.update(dim=_log(rng, 24, 160), tf=rng.choice([16, 64, 256]))
        if kind == "train":
            c.update(w=_log(rng, 32, 400), h=_log(rng, 32, 400))
    return c


# ------------------------------------------------------------------ inputs


def _gen(seed):
    return torch.Generator(device=DEV).manual_seed(int(seed))


def _uniform(g, *shape, lo=0.0, hi=1.0):
    return torch.rand(*shape, generator=g, device=DEV, dtype=torch.float64) * (hi - lo) + lo


def _tiles(w, h):
    """Pixel indices in 8x8-tile order."""
    y, x = torch.meshgrid(torch.arange(h, device=DEV), torch.arange(w, device=DEV), indexing="ij")
    key = ((y // 8) * ((w + 7) // 8) + x // 8) * 64 + (y % 8) * 8 + x % 8
    return torch.argsort(key.reshape(-1))


def _rays(org, d):
    n = d.shape[0]
    r = torch.empty((n, 8), dtype=torch.float32, device=DEV)
    r[:, 0:3] = org.to(torch.float32)
    r[:, 4:7] = d.to(torch.float32)
    bits = r.view(torch.int32)
    bits[:, 3] = 1  # double sided
    bits[:, 7] = -1  # no previous primitive
    return r


def _camera(eye, target, fov, c, up=(0.0, 0.0, 1.0)):
    """One ray per pixel centre of a pinhole camera."""
    w, h = c["w"], c["h"]
    eye, target, up = (torch.tensor(v, dtype=torch.float64, device=DEV) for v in (eye, target, up))
    fwd = target - eye
    fwd = fwd / fwd.norm()
    right = torch.linalg.cross(fwd, up)
    right = right / right.norm()
    upv = torch.linalg.cross(right, fwd)
    s = math.tan(math.radians(fov) * 0.5)
    x = ((torch.arange(w, device=DEV, dtype=torch.float64) + 0.5) / w * 2 - 1) * s * w / h
    y = (1 - (torch.arange(h, device=DEV, dtype=torch.float64) + 0.5) / h * 2) * s
    d = fwd + x[None, :, None] * right + y[:, None, None] * upv
    d = (d / d.norm(dim=-1, keepdim=True)).reshape(-1, 3)
    if c["order"] == "tile":
        d = d[_tiles(w, h)]
    return _rays(eye, d)


def _heightfield(grid, g, jitter=0.01):
    amp = _uniform(g, 8, lo=0.02, hi=0.06).tolist()
    freq = _uniform(g, 8, 2, lo=0.5, hi=6.0).tolist()
    phase = _uniform(g, 8, hi=2 * math.pi).tolist()
    t = torch.linspace(0, 1, grid, device=DEV, dtype=torch.float64)
    y, x = torch.meshgrid(t, t, indexing="ij")
    z = torch.randn(grid, grid, generator=g, device=DEV, dtype=torch.float64) * jitter
    for k in range(8):
        z = z + amp[k] * torch.sin(2 * math.pi * (freq[k][0] * x + freq[k][1] * y) + phase[k])
    vert = torch.stack([x, y, z], -1).reshape(-1, 3).to(torch.float32)
    i = torch.arange(grid - 1, device=DEV)
    j, i = torch.meshgrid(i, i, indexing="ij")
    a = (j * grid + i).reshape(-1)
    b, c, d = a + 1, a + grid, a + grid + 1
    face = torch.stack([a, b, d, a, d, c], -1).reshape(-1, 3).to(torch.int32)
    return vert.contiguous(), face.contiguous()


def _above(c, g):
    """Rays straight down onto the heightfield's inside, slightly tilted."""
    n = c["w"] * c["h"]
    o = torch.empty((n, 3), dtype=torch.float64, device=DEV)
    o[:, :2] = _uniform(g, n, 2, lo=0.2, hi=0.8)
    o[:, 2] = 1.5
    d = torch.empty_like(o)
    d[:, :2] = _uniform(g, n, 2, lo=-0.05, hi=0.05)
    d[:, 2] = -1.0
    return _rays(o, d / d.norm(dim=-1, keepdim=True))


def _lattice(cells, g, jitter=0.2):
    n1 = cells + 1
    t = torch.arange(n1, device=DEV, dtype=torch.float64)
    z, y, x = torch.meshgrid(t, t, t, indexing="ij")
    p = torch.stack([x, y, z], -1).reshape(-1, 3)
    p = p + _uniform(g, *p.shape, lo=-jitter, hi=jitter)
    k = torch.arange(cells, device=DEV)
    cz, cy, cx = torch.meshgrid(k, k, k, indexing="ij")
    return p, (cz * n1 * n1 + cy * n1 + cx).reshape(-1), n1


def _scalars(q, cells, g, count=8):
    s = torch.zeros(len(q), dtype=torch.float64, device=DEV)
    cen = _uniform(g, count, 3, hi=cells)
    sig = _uniform(g, count, 3, lo=0.1, hi=0.3) * cells
    for k in range(count):
        s = s + torch.exp(-0.5 * (((q - cen[k]) / sig[k]) ** 2).sum(-1))
    return s.to(torch.float32).contiguous()


# six tetrahedra per cube along its 0-7 diagonal; corner c lies at
# (c & 1, c >> 1 & 1, c >> 2 & 1)
_SIX = ((0, 1, 3, 7), (0, 3, 2, 7), (0, 2, 6, 7), (0, 6, 4, 7), (0, 4, 5, 7), (0, 5, 1, 7))


def _tets(cells, g):
    p, base, n1 = _lattice(cells, g)
    corner = [(k & 1) + (k >> 1 & 1) * n1 + (k >> 2 & 1) * n1 * n1 for k in range(8)]
    six = torch.tensor([[corner[k] for k in t] for t in _SIX], device=DEV)
    f = (base[:, None, None] + six[None]).reshape(-1, 4)
    a, b, c, d = (p[f[:, k]] for k in range(4))
    turn = (torch.linalg.cross(b - a, c - a) * (d - a)).sum(-1) > 0
    f = torch.where(turn[:, None], f[:, [0, 2, 1, 3]], f)
    return (p.to(torch.float32).contiguous(), f.to(torch.int32).contiguous(),
            _scalars(p, cells, g))


# a hexahedron's corners (lower face, then the face above it) and faces
_HEX = ((0, 0, 0), (1, 0, 0), (1, 1, 0), (0, 1, 0), (0, 0, 1), (1, 0, 1), (1, 1, 1), (0, 1, 1))
_FACES = ((0, 3, 2, 1), (4, 5, 6, 7), (0, 1, 5, 4), (1, 2, 6, 5), (2, 3, 7, 6), (0, 4, 7, 3))


def _solids(cells, nv, g):
    p, base, n1 = _lattice(cells, g)
    hexa = base[:, None] + torch.tensor([x + y * n1 + z * n1 * n1 for x, y, z in _HEX], device=DEV)
    if nv == 8:
        f = hexa
    elif nv == 6:
        f = torch.cat([hexa[:, [0, 1, 2, 4, 5, 6]], hexa[:, [0, 2, 3, 4, 6, 7]]], 1).reshape(-1, 6)
    else:
        apex = len(p) + torch.arange(len(hexa), device=DEV)
        p = torch.cat([p, p[hexa].mean(1)])
        sides = hexa[:, torch.tensor(_FACES, device=DEV)][:, :, [0, 3, 2, 1]]
        f = torch.cat([sides, apex[:, None, None].expand(-1, 6, 1)], 2).reshape(-1, 5)
    return (p.to(torch.float32).contiguous(), f.to(torch.int32).contiguous(),
            _scalars(p[f.reshape(-1)], cells, g))


def _polylines(curves, segs, g, step=0.02):
    at = _uniform(g, curves, 3, lo=-1.0, hi=1.0)
    d = torch.randn(curves, 3, generator=g, device=DEV, dtype=torch.float64)
    p = [at]
    for _ in range(segs):
        d = d + 0.6 * torch.randn(curves, 3, generator=g, device=DEV, dtype=torch.float64)
        d = d / d.norm(dim=-1, keepdim=True)
        at = at + step * d
        p.append(at)
    p = torch.stack(p, 1).reshape(-1, 3).to(torch.float32)
    a = (torch.arange(curves, device=DEV)[:, None] * (segs + 1)
         + torch.arange(segs, device=DEV)).reshape(-1)
    return p.contiguous(), torch.stack([a, a + 1], -1).to(torch.int32).contiguous()


def _plummer(count, g):
    """Centres of a unit Plummer sphere, lognormal radii; the radii shrink
    with the mean distance of a smaller or larger set."""
    m = _uniform(g, count, lo=1e-6, hi=0.999)
    r = (1.0 / torch.sqrt(m ** (-2.0 / 3.0) - 1.0)).clamp_(max=50.0)
    ct = _uniform(g, count, lo=-1.0, hi=1.0)
    ph = _uniform(g, count, hi=2 * math.pi)
    st = torch.sqrt(1.0 - ct * ct)
    p = torch.stack([r * st * torch.cos(ph), r * st * torch.sin(ph), r * ct], -1)
    mu = -6.0 + math.log((1 << 24) / count) / 3.0
    rad = torch.exp(mu + 0.5 * torch.randn(count, generator=g, device=DEV, dtype=torch.float64))
    return p.to(torch.float32).contiguous(), rad.to(torch.float32).contiguous()


def _volume(dim, g, count=48):
    ax = torch.linspace(0, 1, dim, device=DEV, dtype=torch.float64)
    cen = _uniform(g, count, 3, lo=0.15, hi=0.85)
    sig = _uniform(g, count, 3, lo=0.03, hi=0.15)
    w = _uniform(g, count, lo=0.3, hi=1.0)
    e = torch.exp(-0.5 * ((ax[None, None] - cen[..., None]) / sig[..., None]) ** 2)
    vol = torch.zeros(dim, dim, dim, device=DEV, dtype=torch.float64)
    for k in range(count):
        vol += w[k] * e[k, 2][:, None, None] * e[k, 1][None, :, None] * e[k, 0][None, None, :]
    return (vol / vol.max()).to(torch.float32).reshape(-1).contiguous()


def _transfer(size, g):
    x = torch.linspace(0, 1, size, device=DEV, dtype=torch.float64)
    f, ph = _uniform(g, 3, lo=0.5, hi=2.0), _uniform(g, 3, hi=2 * math.pi)
    tf = torch.empty(size, 4, device=DEV, dtype=torch.float64)
    tf[:, :3] = 0.5 + 0.5 * torch.sin(2 * math.pi * f * x[:, None] + ph)
    tf[:, 3] = 0.05 * (x - 0.1).clamp(min=0) ** 1.5 / 0.9 ** 1.5
    return tf.to(torch.float32).contiguous()


def _volume_inputs(c, g):
    rays = _camera((1.8, -1.2, 1.5), (0.5, 0.5, 0.5), 35.0, c)
    return {"vox": _volume(c["dim"], g), "tf": _transfer(c["tf"], g), "rays": rays,
            "dims": (c["dim"],) * 3, "step": 0.5 / c["dim"]}


def _rotation(g):
    q = torch.randn(4, generator=g, device=DEV, dtype=torch.float64)
    w, x, y, z = (q / q.norm()).tolist()
    return [[1 - 2 * (y * y + z * z), 2 * (x * y - z * w), 2 * (x * z + y * w)],
            [2 * (x * y + z * w), 1 - 2 * (x * x + z * z), 2 * (y * z - x * w)],
            [2 * (x * z - y * w), 2 * (y * z + x * w), 1 - 2 * (x * x + y * y)]]


def _scene(c, g):
    """Heightfield patches of several sizes, each with a rotation and a place
    on a jittered lattice; an orbiting camera that frames them all."""
    n = c["meshes"]
    side = math.ceil(n ** (1.0 / 3.0))
    meshes, place = [], []
    shift = torch.tensor([0.5, 0.5, 0.0], device=DEV)
    for i in range(n):
        v, f = _heightfield(max(32, int(c["grid"] * (0.4 + 0.6 * ((i * 7) % n) / n))), g)
        meshes.append(((v - shift).contiguous(), f))
        cell = torch.tensor([i % side, i // side % side, i // (side * side)], dtype=torch.float64)
        at = 1.5 * (cell + (torch.rand(3, generator=g, device=DEV, dtype=torch.float64)
                            * 0.3 - 0.15).cpu())
        m = torch.eye(4, dtype=torch.float64)
        m[:3, :3] = torch.tensor(_rotation(g), dtype=torch.float64).T
        m[3, :3] = at
        place.append(m)
    t = torch.stack(place)
    mid = t[:, 3, :3].mean(0)
    span = float((t[:, 3, :3].max(0).values - t[:, 3, :3].min(0).values).max()) + 1.0
    eye = mid + span * torch.tensor([1.3, 0.5, 0.6], dtype=torch.float64)
    return meshes, t.numpy(), _camera(eye.tolist(), mid.tolist(), 40.0, c)


def _ao_rays(c, p, rad, g):
    """Cosine-weighted short rays that leave particles chosen at random, in
    runs of 8 per particle, each told to skip its own."""
    n = c["rays"]
    k = (n + 7) // 8
    at = torch.randint(0, c["count"], (k,), generator=g, device=DEV)
    near = torch.argsort(p[at, 0], stable=True)  # neighbours in a run of hits lie near each other
    at = at[near]
    nrm = torch.randn(k, 3, generator=g, device=DEV, dtype=torch.float64)
    nrm = nrm / nrm.norm(dim=-1, keepdim=True)
    o = p[at].double() + (rad[at].double() * 1.001)[:, None] * nrm
    d = torch.randn(k, 8, 3, generator=g, device=DEV, dtype=torch.float64)
    d = nrm[:, None] + d / d.norm(dim=-1, keepdim=True) * 0.999
    d = d / d.norm(dim=-1, keepdim=True)
    r = _rays(o[:, None].expand(-1, 8, -1).reshape(-1, 3), d.reshape(-1, 3))
    r.view(torch.int32)[:, 7] = at.to(torch.int32).repeat_interleave(8)
    return r[:n].contiguous(), torch.full((n,), 0.05, dtype=torch.float32, device=DEV)


def prepare(case, seed):
    c, g, kind = case, _gen(seed), case["kind"]
    s = {"kind": kind}
    if kind == "tri":
        v, f = _heightfield(c["grid"], g)
        s["rays"] = (_above(c, g) if c["view"] == "above" else
                     _camera((0.5, -0.1, 1.0), (0.5, 0.45, 0.0), 48.0, c))
        s["geo"] = (v, f) if c["rebuild"] else None
        s["acc"] = A.TriangleAccel()
        s["acc"].Build32(v, f)
    elif kind == "tet":
        v, f, s["scalars"] = _tets(c["cells"], g)
        n = float(c["cells"])
        s["rays"] = _camera((1.6 * n, -0.6 * n, 1.3 * n), (0.5 * n, 0.5 * n, 0.5 * n), 36.0, c)
        s["geo"] = (v, f)
        s["acc"] = A.TetraAccel()
        s["acc"].Build32(v, f)
    elif kind in ("sph", "ao"):
        p, r = _plummer(c["count"], g)
        s["acc"] = A.ParticleAccel()
        s["acc"].Build32(p, r)
        if kind == "sph":
            s["rays"] = _camera((0.0, -6.0, 1.0), (0.0, 0.0, 0.0), 30.0, c)
            s["geo"] = (p, r) if c["rebuild"] else None
        else:
            s["rays"], s["tmax"] = _ao_rays(c, p, r, g)
            s["bits"] = c["bits"]
    elif kind == "sol":
        v, f, s["scalars"] = _solids(c["cells"], c["nv"], g)
        n = float(c["cells"])
        s["rays"] = _camera((1.6 * n, -0.7 * n, 1.3 * n), (0.5 * n, 0.5 * n, 0.45 * n), 45.0, c)
        s["acc"] = A.SolidAccel()
        s["acc"].Build32(v, f, c["nv"])
    elif kind == "lin":
        p, f = _polylines(c["curves"], c["segs"], g)
        s["rays"] = _camera((0.3, -3.2, 0.8), (0.0, 0.0, 0.0), 40.0, c)
        s["acc"] = A.LineAccel()
        s["acc"].Build(p, f, constant_radius=0.004)
    elif kind == "scene":
        meshes, place, s["rays"] = _scene(c, g)
        s["scene"] = A.Scene(A.build_triangles_batch(meshes), place)
    else:
        s.update(_volume_inputs(c, g))
        if kind == "march":
            s["vol"] = V.Volume(s["vox"], s["dims"], (V.CLAMP_TO_EDGE,) * 3)
        else:
            s["grad"] = torch.randn(len(s["rays"]), 4, generator=g, device=DEV)
            s["vox"].requires_grad_(True)
            s["tf"].requires_grad_(True)
    return s


def run(state):
    kind = state["kind"]
    if kind in ("tri", "sph"):
        if state["geo"] is not None:
            state["acc"].Build32(*state["geo"])
        return state["acc"].Traverse(state["rays"])
    if kind == "tet":
        state["acc"].Build32(*state["geo"])
        return state["acc"].TraverseTetra(state["rays"], state["scalars"])
    if kind == "ao":
        return state["acc"].TraverseAnySorted(state["rays"], state["tmax"], state["bits"],
                                              "persistent")
    if kind == "sol":
        return state["acc"].TraverseSolid(state["rays"], state["scalars"])
    if kind == "lin":
        return state["acc"].TraverseLines(state["rays"])
    if kind == "scene":
        return state["scene"].Trace(state["rays"])
    if kind == "march":
        return state["vol"].march(state["tf"], state["step"], state["rays"])
    rgba = V.render(state["vox"], state["tf"], state["dims"], state["step"], state["rays"])
    gv, gt = torch.autograd.grad(rgba, (state["vox"], state["tf"]), state["grad"])
    return rgba.detach(), gv, gt


# --------------------------------------------------------- work and accuracy


def _prims(c):
    """(primitives, bytes of one primitive's own geometry, flops of its test)"""
    kind = c["kind"]
    if kind == "tri":
        return 2 * (c["grid"] - 1) ** 2, 48, 50
    if kind == "tet":
        return 6 * c["cells"] ** 3, 64, 200
    if kind in ("sph", "ao"):
        return c["count"], 16, 30
    if kind == "sol":
        return {5: 6, 6: 2, 8: 1}[c["nv"]] * c["cells"] ** 3, 16 * c["nv"], 400
    if kind == "lin":
        return c["curves"] * c["segs"], 32, 100
    return int(c["meshes"] * (c["grid"] * 0.7) ** 2 * 2), 48, 50


def work(case):
    """Rays read and hits written once, the geometry that rays can touch read
    once, one descent of a binary tree and one primitive test per ray; a
    rebuild reads the geometry and writes nodes and primitives. Marches: each
    voxel once, and a trilinear fetch, table lookup and blend per sample."""
    c, kind = case, case["kind"]
    n = c["rays"] if kind == "ao" else c["w"] * c["h"]
    if kind in ("march", "train"):
        vox = c["dim"] ** 3
        samples = n * 1.0 * c["dim"]  # about half a voxel per step over half the diagonal
        if kind == "march":
            return {"bytes": 4.0 * vox + 48.0 * n, "flops": 45.0 * samples}
        return {"bytes": 4.0 * vox * 3 + 48.0 * n * 3, "flops": 160.0 * samples}
    prims, size, test = _prims(c)
    out = {"tet": 48, "sol": 80, "lin": 48, "ao": 4, "scene": 20}.get(kind, 16)
    b = n * (32.0 + out) + min(prims, n) * float(size)
    f = n * (24.0 * math.log2(max(2, prims)) + test)
    if kind == "tet" or c.get("rebuild"):
        b += prims * (2.0 * size + 24.0)
        f += prims * 60.0
    return {"bytes": b, "flops": f}


def tolerance(case):
    """Hits, weights and occlusion flags are defined bit by bit (they follow
    one fixed order of float operations); marched colours and gradients are
    32-bit sums, the gradients in an order that changes from run to run."""
    if case["kind"] == "march":
        return {"rel": 1e-5}
    if case["kind"] == "train":
        return {"rel": 4e-5, "max": 4e-3}
    return "exact"


def _exact_tri(c, s, v, f):
    """Closest hits by testing every triangle in 64 bits (small sizes)."""
    rays, n = s["rays"], len(s["rays"])
    o, d = rays[:, 0:3].double(), rays[:, 4:7].double()
    p0, p1, p2 = (v[f[:, k].long()].double() for k in range(3))
    e1, e2 = p1 - p0, p2 - p0
    out = torch.empty(n, 4, dtype=torch.float64, device=DEV)
    step = max(1, 8_000_000 // len(f))
    for i in range(0, n, step):
        oo, dd = o[i:i + step, None], d[i:i + step, None]
        pv = torch.linalg.cross(dd.expand(-1, len(f), -1), e2[None].expand(len(oo), -1, -1))
        det = (e1 * pv).sum(-1)
        sv = oo - p0
        u = (sv * pv).sum(-1) / det
        q = torch.linalg.cross(sv, e1[None].expand_as(sv))
        w = (q * dd).sum(-1) / det
        t = (q * e2).sum(-1) / det
        t = torch.where((u >= 0) & (w >= 0) & (u + w <= 1) & (t >= 0), t, float("inf"))
        best, at = t.min(-1)
        hit = torch.isfinite(best)
        pick = torch.where(hit, at, -1).to(torch.int32).view(torch.float32).double()
        r = torch.arange(len(at), device=DEV)
        miss = torch.finfo(torch.float32).max
        out[i:i + step] = torch.stack(
            [torch.where(hit, best, miss), torch.where(hit, u[r, at], 0.0),
             torch.where(hit, w[r, at], 0.0), pick], -1)
    return out


def _exact_march(c, s):
    """The march in 64 bits, all samples of a chunk of rays at once; the
    gradients by autograd."""
    d3, dim, size = torch.float64, c["dim"], c["tf"]
    vox = s["vox"].detach().double().requires_grad_(c["kind"] == "train")
    tf = s["tf"].detach().double().requires_grad_(c["kind"] == "train")
    # entry, exit and sample count from the float rays the march is given
    o, d = s["rays"][:, 0:3].double(), s["rays"][:, 4:7].double()
    inv = 1.0 / d
    a, b = (0.0 - o) * inv, (1.0 - o) * inv
    t0 = torch.minimum(a, b).max(-1).values.clamp(min=0.0)
    t1 = torch.maximum(a, b).min(-1).values
    step = float(torch.tensor(s["step"], dtype=torch.float32))
    count = torch.ceil((t1 - t0) / step - 0.5).clamp(min=0).to(torch.int64)
    n, most = len(o), int(count.max())
    out = torch.empty(n, 4, dtype=d3, device=DEV)
    gv, gt = torch.zeros_like(vox), torch.zeros_like(tf)
    chunk = max(64, 3_000_000 // max(1, most))
    k = torch.arange(max(1, most), device=DEV, dtype=d3) + 0.5
    for i in range(0, n, chunk):
        j = slice(i, min(n, i + chunk))
        t = t0[j, None] + k * step
        live = torch.arange(len(k), device=DEV) < count[j, None]
        val = 0.0
        idx, frac = [], []
        for x in range(3):
            p = (o[j, x, None] + t * d[j, x, None]) * (dim - 1)
            lo = p.floor().clamp(0, dim - 1)
            frac.append(p - lo)
            lo = lo.long()
            idx.append((lo, (lo + 1).clamp(max=dim - 1)))
        for m in range(8):
            x, y, z = m & 1, m >> 1 & 1, m >> 2
            wgt = ((frac[0] if x else 1 - frac[0]) * (frac[1] if y else 1 - frac[1])
                   * (frac[2] if z else 1 - frac[2]))
            val = val + wgt * vox[(idx[2][z] * dim + idx[1][y]) * dim + idx[0][x]]
        pos = (val * (size - 1)).clamp(0, size - 1)
        bin_ = pos.detach().floor().clamp(max=size - 2).long()
        fr = (pos - bin_)[..., None]
        rgba = tf[bin_] * (1 - fr) + tf[bin_ + 1] * fr
        alpha = torch.where(live, rgba[..., 3], 0.0)
        past = torch.cumprod(1 - alpha, -1)
        before = torch.cat([torch.ones_like(past[:, :1]), past[:, :-1]], -1)
        col = ((before * alpha)[..., None] * rgba[..., :3]).sum(1)
        res = torch.cat([col, 1 - past[:, -1:]], -1)
        out[j] = res.detach()
        if c["kind"] == "train":
            x, y = torch.autograd.grad(res, (vox, tf), s["grad"][j].double())
            gv += x
            gt += y
    return out if c["kind"] == "march" else (out, gv, gt)


def exact(case, seed):
    if case["kind"] in ("march", "train"):
        s = _volume_inputs(case, g := _gen(seed))
        if case["kind"] == "train":
            s["grad"] = torch.randn(len(s["rays"]), 4, generator=g, device=DEV)
        return _exact_march(case, s)
    # closest hits of the other kinds: brute force would take too long, or
    # follows the float tests bit by bit (spheres, lines)
    if case["kind"] == "tri" and case["view"] == "above":
        g = _gen(seed)
        v, f = _heightfield(case["grid"], g)
        if len(f) * case["w"] * case["h"] < 3e10:
            return _exact_tri(case, {"rays": _above(case, g)}, v, f)
    return None
