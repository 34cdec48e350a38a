"""Hits at a distance of zero on the GPU, against the oracle bit for bit.

A ray that starts on a sphere and is tangent to it has a discriminant and a
linear term of zero, and the float test reports t = -0.5 * (b / a) = -0.0
(SphereIsect, render/render_accel_particle.cc:2423-2512). Nothing may replace
such a hit, whatever the leaves visited after it hold; leaves that few lanes
reach are tested as (ray, sphere) pairs whose order is that of t's bits, so
the kept distance's sign must not enter it.

The rays start on sphere 0 inside sphere 1, whose exit lies at a positive t.
They come alone, 8 to a launch, and among 63 rays of the same signs that see
nothing, so that their leaves are paired at each size.
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


def spheres(seed, big):
    """Sphere 0 (unit, at the origin) and sphere 1 (radius 4, around its
    surface) among small ones; `big`: all in one Morton cell below the depth cap,
    so that they share one leaf, which has a secondary tree."""
    rng = np.random.default_rng(seed)
    n = 140 if big else 24
    P = rng.uniform(-3, 3, (n, 3)).astype(np.float32)
    R = np.full(n, 0.05, np.float32)
    P[0], R[0] = 0, 1
    P[1], R[1] = rng.choice([-2.0, 2.0], 3), 4.5
    fill = rng.uniform(-3, 3, (1000, 3))  # out of the way: Build32 takes 1,024 and more
    P = np.concatenate([P, (fill + (1.023e6 if big else 300.0)).astype(np.float32)])
    R = np.concatenate([R, np.full(1000, 0.05, np.float32)])
    if big:
        # a Morton cell is 1,000 wide, and the path to this one branches at
        # each of 30 levels: the depth cap
        far = [[1e3 * (1 << k // 3) if c == k % 3 else 0.0 for c in range(3)] for k in range(30)]
        P = np.concatenate([P, np.array(far, np.float32)])
        R = np.concatenate([R, np.full(30, 0.05, np.float32)])
    return P, R


def tangents():
    """Rays along the axes, tangent to sphere 0 where they start."""
    rays = np.zeros(24, W.RAY_DTYPE)
    k = 0
    for a in range(3):
        for b in range(3):
            for so in (1, -1):
                for sd in (1, -1):
                    if a != b:
                        rays["org"][k, a], rays["dir"][k, b] = so, sd
                        k += 1
    rays["flags"] = 1
    rays["prev_prim_id"] = W.NO_PRIM
    return rays


def launches(rays):
    """Each ray alone, 8 of the same signs, and one among 63 that see nothing."""
    for i, r in enumerate(rays):
        yield rays[i:i + 1]
        yield np.repeat(rays[i:i + 1], 8)
        away = np.repeat(rays[i:i + 1], 64)
        away["org"][1:] += np.float32(3e7) * (rays["dir"][i] + rays["org"][i])
        yield away


@pytest.mark.parametrize("big", [False, True], ids=["small_leaves", "secondary_tree"])
def test_a_tangent_start_keeps_its_sphere(S, big):
    orc = Oracle()
    zero = 0
    for seed in range(6):
        P, R = spheres(seed, big)
        tree = orc.build_sph(P, R)
        leaves = tree["nodes"][tree["nodes"]["flag"] == 1]["data"][:, 0]
        assert leaves.max() >= 140 if big else leaves.max() <= 64
        a = S.ParticleAccel()
        a.Build32(S.device_tensor(P), S.device_tensor(R))
        for rays in launches(tangents()):
            want = orc.trace_sph(tree, P, R, 0.0, rays)
            want = want[0] if isinstance(want, tuple) else want
            got = S.hits_to_numpy(a.Traverse(S.device_tensor(rays)))
            assert np.array_equal(got["prim_id"], want["prim_id"]), (seed, rays[:1])
            assert np.array_equal(got["t"].view(np.uint32), want["t"].view(np.uint32))
            zero += int((want["t"].view(np.uint32) == 0x80000000).any())
    assert zero > 6 * 24
