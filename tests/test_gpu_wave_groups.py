"""Wavefronts whose rays do not share direction signs, on the GPU: the walks
per group of nearby lanes and the lanes traced alone, against the oracle's
closest hits bit for bit (triangles, tetrahedra, spheres, solids, lines) and
its occlusion.

The rays: frames seen along an axis (the signs change inside the frame) with
sides that are no multiples of the 8x8 tile, in tile and in row order; one
camera per ray (every lane alone); and both mixed ray by ray, so that groups
of all sizes and lanes in no group share wavefronts.
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


# kind: geometry, the frame's eye, target and up, half extent of the scene
def geometry(kind):
    if kind == "tri":
        V, F = W.heightfield(72)
        return (V, F), ((0.5, 0.5, 2.0), (0.5, 0.5, 0.0), (0, 1, 0)), 0.5
    if kind == "tet":
        V, F, _ = W.tet_grid(12)
        return (V, F), ((6.0, 6.0, 30.0), (6.0, 6.0, 6.0), (0, 1, 0)), 6.0
    if kind == "sph":
        P, R, _ = W.clustered_spheres(8_000, 4, 600)
        return (P, R), ((0.0, -4.0, 0.0), (0.0, 0.0, 0.0), (0, 0, 1)), 1.0
    if kind == "lin":
        P, segs, _ = W.polylines(120, 40)
        return (P, segs), ((0.0, -3.0, 0.0), (0.0, 0.0, 0.0), (0, 0, 1)), 1.0
    V, F, _ = W.solid_grid(12, nv=int(kind[3:]))
    return (V, F), ((6.0, 6.0, 30.0), (6.0, 6.0, 6.0), (0, 1, 0)), 6.0


def ray_sets(view, half):
    eye, at, up = view
    tile = W.pinhole_rays(eye, at, up, 35.0, 101, 67)
    row = W.pinhole_rays(eye, at, up, 35.0, 77, 45, tiled=False)
    rng = np.random.default_rng(7)
    n = 1500
    single = np.zeros(n, W.RAY_DTYPE)
    single["org"] = (np.array(at) + rng.uniform(-half, half, (n, 3))).astype(np.float32)
    d = rng.normal(size=(n, 3))
    single["dir"] = (d / np.linalg.norm(d, axis=1, keepdims=True)).astype(np.float32)
    single["flags"] = 1
    single["prev_prim_id"] = W.NO_PRIM
    mix = tile[:n].copy()
    take = rng.random(n) < np.repeat(rng.uniform(0, 0.3, n // 50), 50)
    mix[take] = single[take]
    return {"tile": tile, "row": row, "single": single, "mix": mix}


def build(S, orc, kind, geo):
    A, B = geo
    if kind == "tri":
        a, tree = S.TriangleAccel(), orc.build_tri(A, B)
    elif kind == "tet":
        a, tree = S.TetraAccel(), orc.build_tet(A, B)
    elif kind == "sph":
        a, tree = S.ParticleAccel(), orc.build_sph(A, B)
    elif kind == "lin":
        a, tree = S.LineAccel(), orc.build_lin(A, B, None, 0.01)
        a.Build(S.device_tensor(A), S.device_tensor(B), None, 0.01, True)
        return a, lambda rays: orc.trace_lin(tree, A, B, None, 0.01, rays)
    else:
        nv = int(kind[3:])
        a, tree = S.SolidAccel(), orc.build_sol(A, B, nv)
        a.Build32(S.device_tensor(A), S.device_tensor(B), nv)
        return a, lambda rays: orc.trace_sol(tree, A, B, rays)
    a.Build32(S.device_tensor(A), S.device_tensor(B))
    if kind == "sph":
        return a, lambda rays: orc.trace_sph(tree, A, B, 0.0, rays)
    trace = orc.trace_tri if kind == "tri" else orc.trace_tet
    return a, lambda rays: trace(tree, A, B, rays)


@pytest.mark.parametrize("kind", ["tri", "tet", "sph", "lin", "sol8", "sol6", "sol5"])
def test_mixed_sign_wavefronts_match_oracle(S, orc, kind):
    geo, view, half = geometry(kind)
    a, oracle = build(S, orc, kind, geo)
    for name, rays in ray_sets(view, half).items():
        print(kind, name, len(rays), flush=True)
        want = oracle(rays)
        want = want[0] if isinstance(want, tuple) else want
        dev = S.device_tensor(rays)
        got = S.hits_to_numpy(a.Traverse(dev))
        assert np.array_equal(got["prim_id"], want["prim_id"])
        assert np.array_equal(got["t"].view(np.uint32), want["t"].view(np.uint32))
        if kind != "sph":  # a sphere's u, v come from atan2 / acos
            assert np.array_equal(got["u"], want["u"]) and np.array_equal(got["v"], want["v"])
        hit = want["prim_id"] != W.NO_PRIM
        assert hit.any()
        tmax = np.where(hit, np.nextafter(want["t"], np.float32(0 if len(rays) % 2 else 1e30)),
                        np.float32(1e30)).astype(np.float32)
        occ = a.TraverseAny(dev, S.device_tensor(tmax)).cpu().numpy()
        assert np.array_equal(occ != 0, hit & (want["t"] < tmax))


# launches that carry 8, 16, 32 and 64 rays per wavefront, coherent and not
# (random rays that a kernel traces one by one itself share wavefronts of 32
# from 65,552 and of 64 from 131,104 rays on), at sizes around a run of 64 and a
# block
@pytest.mark.parametrize("kind", ["tri", "sph", "lin", "tet", "sol8"])
@pytest.mark.parametrize("n", [1, 63, 65, 127, 129, 40_007, 150_001, 280_000])
def test_launch_sizes_match_oracle(S, orc, kind, n):
    geo, (eye, at, up), half = geometry(kind)
    a, oracle = build(S, orc, kind, geo)
    side = int(np.ceil(np.sqrt(n)))
    frame = W.pinhole_rays(eye, at, up, 35.0, side, side)[:n]
    rng = np.random.default_rng(n)
    rand = frame.copy()
    rand["org"] = (np.array(at) + rng.uniform(-half, half, (n, 3))).astype(np.float32)
    d = rng.normal(size=(n, 3))
    rand["dir"] = (d / np.linalg.norm(d, axis=1, keepdims=True)).astype(np.float32)
    half_rand = frame.copy()
    mix = (np.arange(n) // 64) % 3 == 1
    half_rand[mix] = rand[mix]
    check = np.arange(n) if n < 1000 else np.unique(np.r_[0:200, n - 200:n,
                                                          rng.integers(0, n, 4000)])
    for rays in (frame, rand, half_rand):
        got = S.hits_to_numpy(a.Traverse(S.device_tensor(rays)))
        assert len(got) == n
        want = oracle(np.ascontiguousarray(rays[check]))
        want = want[0] if isinstance(want, tuple) else want
        assert np.array_equal(got["prim_id"][check], want["prim_id"])
        assert np.array_equal(got["t"][check].view(np.uint32), want["t"].view(np.uint32))


# spheres and solids mark the rays that no group takes in the hits themselves:
# what the caller's buffer held before must not matter, nor a launch of none
@pytest.mark.parametrize("kind", ["sph", "sol5", "sol6", "sol8"])
def test_marks_in_the_hits_are_the_call_s_own(S, orc, kind):
    import torch
    geo, view, half = geometry(kind)
    a, oracle = build(S, orc, kind, geo)
    for name, rays in ray_sets(view, half).items():
        want = oracle(rays)
        want = want[0] if isinstance(want, tuple) else want
        dev = S.device_tensor(rays)
        for fill in (-1.0, float("nan"), 0.0):
            hits = torch.full((len(rays) + 64, 4), fill, device="cuda")
            got = S.hits_to_numpy(a.Traverse(dev, hits=hits)[:len(rays)].contiguous())
            assert np.array_equal(got["prim_id"], want["prim_id"]), (name, fill)
            assert np.array_equal(got["t"].view(np.uint32), want["t"].view(np.uint32))
            tail = hits[len(rays):]
            assert bool((torch.isnan(tail) if fill != fill else tail == fill).all())


@pytest.mark.parametrize("kind", ["sph", "sol8"])
def test_two_launch_traces_in_a_graph(S, orc, kind):
    # rays in groups, lone ones and both mixed take turns in one captured call
    import torch
    geo, view, half = geometry(kind)
    a, oracle = build(S, orc, kind, geo)
    sets = [r[:1500] for r in ray_sets(view, half).values()]
    rays = S.device_tensor(sets[0]).clone()
    hits = torch.empty((len(rays), 4), device="cuda")
    side = torch.cuda.Stream()
    side.wait_stream(torch.cuda.current_stream())
    with torch.cuda.stream(side):
        a.Traverse(rays, hits=hits)
    torch.cuda.current_stream().wait_stream(side)
    g = torch.cuda.CUDAGraph()
    with torch.cuda.graph(g):
        a.Traverse(rays, hits=hits)
    for r in sets + sets[::-1]:
        rays.copy_(S.device_tensor(np.ascontiguousarray(r)))
        g.replay()
        torch.cuda.synchronize()
        got = S.hits_to_numpy(hits)
        eager = S.hits_to_numpy(a.Traverse(rays))
        want = oracle(np.ascontiguousarray(r))
        want = want[0] if isinstance(want, tuple) else want
        assert np.array_equal(got["prim_id"], want["prim_id"])
        assert np.array_equal(got["t"].view(np.uint32), want["t"].view(np.uint32))
        assert got.tobytes() == eager.tobytes()
