"""The short box test (box_plain in surface_amd/csrc/srf_trace_dev.h) against
the reference's comparisons (IntersectRayAABB,
render/render_accel_triangle.cc:1815-1861), both restated in numpy float32 on
the CPU: the same answer for every finite box and every ray that plain_ray
passes, products that overflow, touching planes, flat boxes and signed zeros
included.
"""
from __future__ import annotations

import numpy as np
import pytest

f32 = np.float32
MAX = np.finfo(f32).max
TINY = np.array(1, np.uint32).view(f32)


def planes(lo, hi, inv):
    neg = inv < 0
    return np.where(neg, hi, lo), np.where(neg, lo, hi)


def reference(o, inv, lo, hi, maxt):
    near, far = planes(lo, hi, inv)
    a, b = (near - o) * inv, (far - o) * inv
    tmin = np.where(a[:, 0] > a[:, 1], a[:, 0], a[:, 1])
    tmax = np.where(b[:, 0] < b[:, 1], b[:, 0], b[:, 1])
    tmin = np.where(tmin > a[:, 2], tmin, a[:, 2])
    tmax = np.where(tmax < b[:, 2], tmax, b[:, 2])
    clamped = np.where(maxt < tmax, maxt, tmax)
    two = (clamped > 0) & (tmin <= clamped)  # two-box nodes
    own = (tmax > 0) & (tmin <= tmax) & (tmin <= maxt)  # one box per node, maxt = FLT_MAX
    return two, own


def plain(o, inv, lo, hi, maxt):
    near, far = planes(lo, hi, inv)
    a, b = (near - o) * inv, (far - o) * inv
    enter = np.fmax(np.fmax(np.fmax(a[:, 0], a[:, 1]), a[:, 2]), TINY)
    return enter <= np.fmin(np.fmin(np.fmin(b[:, 0], b[:, 1]), b[:, 2]), maxt)


@pytest.mark.parametrize("scale", [1.0, 1e-20, 1e18, 1e37])
def test_same_answer_as_the_comparisons(scale):
    rng = np.random.default_rng(5)
    n = 400_000
    o = (rng.normal(size=(n, 3)) * scale).astype(f32)
    lo = (rng.normal(size=(n, 3)) * scale).astype(f32)
    hi = (lo + np.abs(rng.normal(size=(n, 3)) * scale)).astype(f32)
    hi[::7] = lo[::7]
    touch = rng.random((n, 3)) < 0.1
    o[touch] = np.where(rng.random(touch.sum()) < 0.5, lo[touch], hi[touch])
    d = rng.normal(size=(n, 3)).astype(f32)
    small = rng.random((n, 3)) < 0.1
    d[small] *= f32(1e-38)
    with np.errstate(all="ignore"):
        inv = (f32(1) / d).astype(f32)
    maxt = np.where(rng.random(n) < 0.3, MAX, np.abs(rng.normal(size=n) * scale)).astype(f32)
    maxt[::11] = 0
    ok = (np.isfinite(inv) & (inv != 0) & np.isfinite(o) & np.isfinite(hi)).all(1)
    o, inv, lo, hi, maxt = o[ok], inv[ok], lo[ok], hi[ok], maxt[ok]
    assert len(o) > n // 4
    with np.errstate(all="ignore"):
        two, _ = reference(o, inv, lo, hi, maxt)
        assert np.array_equal(plain(o, inv, lo, hi, maxt), two)
        top = np.full(len(o), MAX, f32)
        _, own = reference(o, inv, lo, hi, top)
        assert np.array_equal(plain(o, inv, lo, hi, top), own)
    assert two.any() and not two.all()
