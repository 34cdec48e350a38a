"""The slab test of the secondary sphere trees (sph_slab / sph_box in
surface_amd/csrc/srf_trace.hip), restated in numpy float32 and checked on the
CPU: no sphere that the float sphere test reports at t may lie in a box that
the slab test skips at the kept distance t. The spheres, rays and sphere test
are test_sphere_pad's (tiny spheres seen from far away, grazing rays, origins
just outside the surface, unnormalised and axis-parallel directions), moved
away from the origin of the coordinates as well.
"""
from __future__ import annotations

import numpy as np
import pytest

from test_sphere_pad import PAD, PAD_ORIGIN, adversarial, f32, f64, sphere_test

FLT_MAX, FLT_MIN = np.finfo(f32).max, np.finfo(f32).tiny


def fma(a, b, c):
    return (a.astype(f64) * b.astype(f64) + c.astype(f64)).astype(f32)


def enters(o, d, lo_box, hi_box, t):
    """Whether a ray enters its box no later than t, as the kernel tests it
    for a leaf whose only box this is."""
    with np.errstate(all="ignore"):
        far = np.maximum(np.abs(o - lo_box), np.abs(o - hi_box)).astype(f32)
        dist = np.sqrt((far * far).sum(1, dtype=f32))
        pad = f32(PAD) * dist + f32(PAD_ORIGIN) * np.abs(o).sum(1, dtype=f32)
        a = (d * d).sum(1, dtype=f32)
        sign = d < 0
        mag = np.minimum(np.abs(f32(1) / d), f32(1e30))
        lim = np.where(sign, -mag, mag).astype(f32)
        grow = np.where(sign, -pad[:, None], pad[:, None]).astype(f32)
        on, of = (o + grow) * lim, (o - grow) * lim
        ok = (a >= FLT_MIN)[:, None] & (np.abs(on) <= FLT_MAX) & (np.abs(of) <= FLT_MAX)
        inv = np.where(ok, lim, f32(0))
        on, of = np.where(ok, on, FLT_MAX), np.where(ok, of, -FLT_MAX)
        tn = fma(np.where(sign, hi_box, lo_box), inv, -on.astype(f32))
        tf = fma(np.where(sign, lo_box, hi_box), inv, -of.astype(f32))
        first = np.fmax(np.fmax(np.fmax(tn[:, 0], tn[:, 1]), tn[:, 2]), f32(0))
        last = np.fmin(np.fmin(np.fmin(tf[:, 0], tf[:, 1]), tf[:, 2]), t)
    return first <= last


@pytest.mark.parametrize("shift", [0.0, 30.0, 5e3])
def test_no_reported_hit_is_culled(shift):
    rng = np.random.default_rng(31)
    hits = 0
    for k in range(4):
        o, d, c, r = adversarial(rng, 200_000)
        if k == 3:  # components far too small to matter, and signed zeros
            d[:, 0] *= f32(1e-35)
            d[::2, 1] = f32(-0.0)
        move = rng.uniform(-shift, shift, (1, 3)).astype(f32)
        o, c = (o + move).astype(f32), (c + move).astype(f32)
        hit, t = sphere_test(o, d, c, r)
        keep = hit & np.isfinite(t) & (np.abs(d).sum(1) > 0)
        o, d, c, r, t = o[keep], d[keep], c[keep], r[keep], t[keep]
        # the build's box of a sphere contains its extents
        lo_box, hi_box = (c - r[:, None]).astype(f32), (c + r[:, None]).astype(f32)
        bad = ~enters(o, d, lo_box, hi_box, t)
        assert not bad.any(), (o[bad][:3], d[bad][:3], c[bad][:3], r[bad][:3], t[bad][:3])
        hits += len(t)
    assert hits > 100_000


def test_the_slab_test_culls():
    # boxes beside, behind and beyond the kept distance are skipped
    z = np.zeros((1, 3), f32)
    d = np.array([[0.0, 0.0, 1.0]], f32)
    box = lambda x, y, s: (np.array([[x, y, s]], f32), np.array([[x + 1, y + 1, s + 1]], f32))  # noqa: E731
    far = np.array([1e9], f32)
    assert enters(z, d, *box(-0.5, -0.5, 5.0), far)[0]
    assert not enters(z, d, *box(0.5, -0.5, 5.0), far)[0]
    assert not enters(z, d, *box(-0.5, -0.5, -5.0), far)[0]
    assert not enters(z, d, *box(-0.5, -0.5, 5.0), np.array([4.9], f32))[0]
