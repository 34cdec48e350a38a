"""Inputs at which the wavefront walks' shortcuts stop or must not matter, on
the GPU against the oracle bit for bit:

- trees with a box so large that its bounds' sum overflows: the short box test
  is not for them, and the walks take the comparisons instead;
- equally near crossings (duplicated lines and solids, a line's cap on
  another's side), within a round of 64 queued tests and across rounds: the
  last side wins, else the first cap; of solids the first;
- rays that start on what they hit (t = 0): leaves tested as pairs go back to
  the one-by-one test.

Rays come in frames, and a few among many that see nothing, so that few lanes
reach a leaf.
"""
from __future__ import annotations

import numpy as np
import pytest

pytestmark = pytest.mark.gpu

from oracle.oracle import Oracle  # noqa: E402
from surface_amd import workloads as W  # noqa: E402


@pytest.fixture(scope="module")
def S():
    import torch
    assert torch.cuda.is_available(), "no GPU visible"
    from surface_amd import accel
    return accel


@pytest.fixture(scope="module")
def orc():
    return Oracle()


def as_rays(org, dirs):
    rays = np.zeros(len(org), W.RAY_DTYPE)
    rays["org"], rays["dir"] = org, dirs
    rays["flags"] = 1
    rays["prev_prim_id"] = W.NO_PRIM
    return rays


def sparse(rays, away):
    """Each of a few rays first of 64; the others see nothing."""
    out = np.repeat(rays, 64)
    k = np.arange(len(out)) % 64 != 0
    out["org"][k] += np.float32(away)
    return out


def check(got, want):
    want = want[0] if isinstance(want, tuple) else want
    assert np.array_equal(got["prim_id"], want["prim_id"])
    assert np.array_equal(got["t"].view(np.uint32), want["t"].view(np.uint32))
    assert np.array_equal(got["u"], want["u"]) and np.array_equal(got["v"], want["v"])
    return want


# ------------------------------------------------------- overflowing boxes

BIG = np.float32(3e38)


def huge(kind):
    """Ordinary geometry and one primitive that reaches to (3e38, 3e38, 0)."""
    if kind == "tri":
        V, F = W.heightfield(40)
        V = np.concatenate([V, np.float32([[BIG, BIG, 0.0]])])
        F = np.concatenate([F, np.uint32([[0, 1, len(V) - 1]])])
        return V, F, ((0.5, -0.1, 1.0), (0.5, 0.45, 0.0), (0, 0, 1))
    if kind == "lin":
        P, segs, _ = W.polylines(60, 40)
        P = np.concatenate([P, np.float32([[BIG, BIG, 0.0]])])
        segs = np.concatenate([segs.reshape(-1, 2), np.uint32([[0, len(P) - 1]])])
        return P, segs, ((0.0, -3.0, 0.5), (0.0, 0.0, 0.0), (0, 0, 1))
    nv = int(kind[3:])
    V, F, _ = W.solid_grid(12, nv=nv)
    F = F.reshape(-1, nv)
    V = np.concatenate([V, np.float32([[BIG, BIG, 0.0]])])
    last = F[-1].copy()
    last[-1] = len(V) - 1
    return V, np.concatenate([F, last[None]]), ((18.0, -8.0, 15.0), (6.0, 6.0, 5.0), (0, 0, 1))


@pytest.mark.parametrize("kind", ["tri", "lin", "sol5", "sol6", "sol8"])
def test_a_box_whose_bounds_overflow(S, orc, kind):
    A, B, (eye, at, up) = huge(kind)
    rays = W.pinhole_rays(eye, at, up, 40.0, 61, 43)
    if kind == "tri":
        a, tree = S.TriangleAccel(), orc.build_tri(A, B)
        a.Build32(S.device_tensor(A), S.device_tensor(B))
        trace = lambda r: orc.trace_tri(tree, A, B, r)  # noqa: E731
    elif kind == "lin":
        a, tree = S.LineAccel(), orc.build_lin(A, B, None, 0.02)
        a.Build(S.device_tensor(A), S.device_tensor(B), None, 0.02, True)
        trace = lambda r: orc.trace_lin(tree, A, B, None, 0.02, r)  # noqa: E731
    else:
        nv = int(kind[3:])
        a, tree = S.SolidAccel(), orc.build_sol(A, B, nv)
        a.Build32(S.device_tensor(A), S.device_tensor(B), nv)
        trace = lambda r: orc.trace_sol(tree, A, B, r)  # noqa: E731
    nodes = tree["nodes"]
    with np.errstate(over="ignore"):
        span = np.abs(nodes["bmin"]).astype(np.float32).reshape(len(nodes), -1).sum(
            1, dtype=np.float32) + np.abs(nodes["bmax"]).reshape(len(nodes), -1).sum(
            1, dtype=np.float32)
    assert not np.isfinite(span).all()  # the tree has such a box
    for r in (rays, sparse(rays[::40], (0.0, 0.0, 1e4))):
        want = check(S.hits_to_numpy(a.Traverse(S.device_tensor(r))), trace(r))
        assert (want["prim_id"] != W.NO_PRIM).any()


# --------------------------------------------------------------- equal hits


@pytest.mark.parametrize("copies", [2, 5])
def test_equal_line_crossings(S, orc, copies):
    # upright capped cylinders of radius 1 whose caps lie in z = 0, and lying
    # ones whose highest side touches z = 0: straight down, a cap of one and
    # the side of the other are both 4 away
    P, segs = [], []
    for k in range(130):
        x = 4.0 * k
        P += [(x, 0, -1), (x, 0, 0), (x - 1.5, 0, -1), (x + 1.5, 0, -1)]
        for _ in range(copies):
            segs += [(4 * k, 4 * k + 1), (4 * k + 2, 4 * k + 3)]
    P, segs = np.float32(P), np.uint32(segs)
    segs = segs[np.random.default_rng(1).permutation(len(segs))]
    fill = np.float32([[0, 50 + k, 60] for k in range(1100)])
    at = len(P) + np.arange(0, 1099, dtype=np.uint32)
    P, segs = np.concatenate([P, fill]), np.concatenate([segs, np.stack([at, at + 1], 1)])
    tree = orc.build_lin(P, segs, None, 1.0)
    a = S.LineAccel()
    a.Build(S.device_tensor(P), S.device_tensor(segs), None, 1.0, True)
    x = np.repeat(4.0 * np.arange(130), 4) + np.tile([0.0, 0.25, -0.5, 0.75], 130)
    down = as_rays(np.stack([x, np.zeros_like(x), np.full_like(x, 4.0)], 1).astype(np.float32),
                   np.float32([[0, 0, -1]]))
    # along the lying cylinders' axes: their caps, one behind the other, tie
    along = as_rays(np.float32([[-4, 0.25 * k, -0.75] for k in range(-2, 3)]),
                    np.float32([[1, 0, 0]]))
    for rays in (down, np.tile(down[:4], 40), sparse(down[::16], (0, 1e4, 0)), along,
                 np.tile(along, 30)):
        want = check(S.hits_to_numpy(a.Traverse(S.device_tensor(rays))),
                     orc.trace_lin(tree, P, segs, None, 1.0, rays))
        assert (want["prim_id"] != W.NO_PRIM).any()
    assert (orc.trace_lin(tree, P, segs, None, 1.0, down)[0]["t"] == 4.0).all()


@pytest.mark.parametrize("nv", [5, 6, 8])
def test_equal_solid_crossings(S, orc, nv):
    V, F, _ = W.solid_grid(10, nv=nv, jitter=0.0)
    F = np.repeat(F.reshape(-1, nv), 3, axis=0)
    F = F[np.random.default_rng(2).permutation(len(F))]
    tree = orc.build_sol(V, F, nv)
    a = S.SolidAccel()
    a.Build32(S.device_tensor(V), S.device_tensor(F), nv)
    rng = np.random.default_rng(3)
    xy = rng.uniform(0, 10, (300, 2)).astype(np.float32)
    up = as_rays(np.concatenate([xy, np.full((300, 1), -3, np.float32)], 1),
                 np.float32([[0.0, 0.0, 1.0]]))
    skew = as_rays(np.concatenate([xy, np.full((300, 1), -3, np.float32)], 1),
                   np.float32([[0.25, 0.125, 1.0]]))
    for rays in (up, skew, sparse(skew[:40], (0, 0, 1e4))):
        want = check(S.hits_to_numpy(a.Traverse(S.device_tensor(rays))),
                     orc.trace_sol(tree, V, F, rays))
        assert (want["prim_id"] != W.NO_PRIM).mean() > 0.01


# -------------------------------------------------------------------- t = 0


def test_triangles_at_the_origin_of_the_ray(S, orc):
    # a flat lattice, each triangle twice: rays that start in it, on its
    # vertices and its edges, and some above it
    n = 24
    y, x = np.mgrid[0:n, 0:n]
    V = np.stack([x, y, np.zeros_like(x)], -1).reshape(-1, 3).astype(np.float32)
    i = (y[:-1, :-1] * n + x[:-1, :-1]).reshape(-1)
    F = np.concatenate([np.stack([i, i + 1, i + n + 1], 1), np.stack([i, i + n + 1, i + n], 1)])
    F = np.concatenate([F, F]).astype(np.uint32)
    F = F[np.random.default_rng(5).permutation(len(F))]
    tree = orc.build_tri(V, F)
    a = S.TriangleAccel()
    a.Build32(S.device_tensor(V), S.device_tensor(F))
    rng = np.random.default_rng(6)
    xy = rng.uniform(0, n - 1, (600, 2))
    xy[::3] = np.round(xy[::3])
    xy[1::3, 0] = np.round(xy[1::3, 0])
    z = np.where(rng.random(600) < 0.7, 0.0, rng.uniform(-1, 1, 600))
    org = np.concatenate([xy, z[:, None]], 1).astype(np.float32)
    zero = 0
    for d in ((0.0, 0.0, 1.0), (0.25, 0.5, -1.0), (0.125, -0.25, 0.5)):
        rays = as_rays(org, np.float32([d]))
        for r in (rays, sparse(rays[:60], (0, 0, 1e4 * np.sign(d[2]))), rays[:8], rays[:1]):
            want = check(S.hits_to_numpy(a.Traverse(S.device_tensor(r))),
                         orc.trace_tri(tree, V, F, r))
            zero += int((want["t"] == 0).sum())
    assert zero > 300


def test_spheres_at_the_origin_of_the_ray(S, orc):
    # rays that leave a sphere's surface at its axis points, in and out
    rng = np.random.default_rng(7)
    P = rng.integers(-12, 13, (1500, 3)).astype(np.float32)
    R = rng.choice(np.float32([0.5, 1.0, 2.0]), 1500)
    tree = orc.build_sph(P, R)
    a = S.ParticleAccel()
    a.Build32(S.device_tensor(P), S.device_tensor(R))
    at = rng.integers(0, 1500, 400)
    side = np.eye(3, dtype=np.float32)[rng.integers(0, 3, 400)] * rng.choice([-1, 1], (400, 1))
    org = (P[at] + R[at, None] * side).astype(np.float32)
    d = np.eye(3, dtype=np.float32)[rng.integers(0, 3, 400)] * rng.choice([-1, 1], (400, 1))
    rays = as_rays(org, d.astype(np.float32))
    seen = 0
    for r in (rays, sparse(rays[:60], 1e4), rays[:8], rays[:1]):
        got = S.hits_to_numpy(a.Traverse(S.device_tensor(r)))
        want = orc.trace_sph(tree, P, R, 0.0, r)
        want = want[0] if isinstance(want, tuple) else want
        assert np.array_equal(got["prim_id"], want["prim_id"])
        assert np.array_equal(got["t"].view(np.uint32), want["t"].view(np.uint32))
        seen += int((want["t"] == 0).sum())
    assert seen > 100
