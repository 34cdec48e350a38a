"""The float filter of the solid walk (sol_may_hit in
surface_amd/csrc/srf_trace.hip), restated in numpy float32 and checked on the
CPU against the oracle's FP64 crossings (or_solid_isect, the reference's
Intersect{Pyramid,Prism,Hexa}D): a solid that the filter drops at tb has no
crossing at a distance of zero or more below tb. tb is put on, just above and
just below the crossings; solids are warped, flat and far from the origin,
rays graze edges, and directions have lengths from 0.2 to 100.
"""
from __future__ import annotations

import numpy as np
import pytest

from oracle.oracle import Oracle
from surface_amd import workloads as W

f32 = np.float32
MAX = np.finfo(f32).max
EDGES = {5: [(i & 3, (i + 1) & 3 if i < 4 else 4) for i in range(8)],
         6: [(i if i < 6 else i - 6, (i + 1) % 3 if i < 3 else 3 + (i - 2) % 3 if i < 6 else i - 3)
             for i in range(9)],
         8: [(i if i < 8 else i - 8, (i + 1) & 3 if i < 4 else 4 + ((i + 1) & 3) if i < 8 else i - 4)
             for i in range(12)]}
# kind, corners v0 v1 v2, side products w0..w3, edges e2 e3 (~i: negated)
FACES = {5: [(0, 0, 1, 2, 0, 1, 2, 3, 2, 3), (1, 4, 1, 0, 0, 4, 5, 0, 0, 0),
             (1, 4, 2, 1, 1, 5, 6, 0, 0, 0), (1, 4, 3, 2, 2, 6, 7, 0, 0, 0),
             (1, 4, 0, 3, 3, 7, 4, 0, 0, 0)],
         6: [(2, 2, 0, 1, 0, 1, 2, 0, 0, 0), (2, 5, 3, 4, 3, 4, 5, 0, 0, 0),
             (0, 2, 0, 3, 2, 6, ~5, ~8, 5, 8), (0, 0, 1, 4, 0, 7, ~3, ~6, 3, 6),
             (0, 1, 2, 5, 1, 8, ~4, ~7, 4, 7)],
         8: [(0, 0, 1, 2, 0, 1, 2, 3, 2, 3), (0, 4, 5, 6, 4, 5, 6, 7, 6, 7),
             (0, 0, 1, 5, 0, 9, ~4, ~8, 4, 8), (0, 1, 2, 6, 1, 10, ~5, ~9, 5, 9),
             (0, 2, 3, 7, 2, 11, ~6, ~10, 6, 10), (0, 3, 0, 4, 3, 8, ~7, ~11, 7, 11)]}


def face(nv, A, B):
    """sol_face: the face of the masks A, B (boolean edge lists)."""
    bits = lambda m: sum(1 << i for i, x in enumerate(m) if x)  # noqa: E731
    A, B = bits(A), bits(B)
    has = lambda m, b: (m & b) == b  # noqa: E731
    if nv == 5:
        Mi, Mn = B, A
        rules = [(0, 0xF), (0x21, 0x10), (0x42, 0x20), (0x84, 0x40), (0x18, 0x80)]
        for f, (n, i) in enumerate(rules):
            if has(Mn, n) and has(Mi, i):
                return f
    else:
        Mi, Mn = A, B
        rules = ([(0x7, 0), (0, 0x38), (0x120, 0x44), (0x48, 0x81), (0x90, 0x102)] if nv == 6 else
                 [(0xF, 0), (0, 0xF0), (0x110, 0x201), (0x220, 0x402), (0x440, 0x804),
                  (0x880, 0x108)])
        for f, (n, i) in enumerate(rules):
            if has(Mn, n) and has(Mi, i):
                return f
    return -1


def may_hit(nv, V, o, d, tb, cext):
    """sol_may_hit for one solid (float32 arithmetic throughout)."""
    with np.errstate(all="ignore"):
        ln = np.sqrt((d * d).sum(dtype=f32))
        x, y, z = d / ln
        e1 = np.array([-y, x, 0], f32) if abs(x) > abs(z) else np.array([0, -z, y], f32)
        e1 = (e1 / np.sqrt((e1 * e1).sum(dtype=f32))).astype(f32)
        dn = np.array([x, y, z], f32)
        e2 = np.array([y * e1[2] - z * e1[1], z * e1[0] - x * e1[2], x * e1[1] - y * e1[0]], f32)
        C = f32(cext) + np.abs(o).max()
        r = (V - o).astype(f32)
        px, py, pz = ((r * e).sum(1, dtype=f32) for e in (e1, e2, dn))
        P, Z = (np.abs(px) + np.abs(py)).max(), np.abs(pz).max()
        eta = f32(1e-6) * (Z + P)
        E = (f32(2) * eta * (P + eta) + f32(2.4e-7) * P * P) + f32(1e-14) * (Z + P) * C
        w = np.array([px[b] * py[a] - py[b] * px[a] for a, b in EDGES[nv]], f32)
        if not (np.abs(w).min() > E) or ln > 1e4:
            return True
        m0 = w > 0
        f0, f1 = face(nv, m0, ~m0), face(nv, ~m0, m0)
        if f0 < 0 or f1 < 0:
            return False
        far = ln * f32(tb)
        zt = far + f32(4e-6) * ln * (C + far)
        serr = E * (f32(32) * (Z + abs(zt)) + f32(10) * P)

        def beyond(f):
            k, v0, v1, v2, w0, w1, w2, w3, g, h = FACES[nv][f]
            wt = lambda i: -w[~i] if i < 0 else w[i]  # noqa: E731
            if k == 0:
                (a2, b2), (a3, b3) = EDGES[nv][g], EDGES[nv][h]
                cr = ((px[b2] - px[a2]) * (py[b3] - py[a3])
                      - (py[b2] - py[a2]) * (px[b3] - px[a3]))
                a, b, c = wt(w1), (wt(w2) + wt(w3)) + cr, wt(w0)
            elif k == 1:
                a, b, c = -wt(w0), wt(w1), -wt(w2)
            else:
                a, b, c = wt(w0), wt(w1), wt(w2)
            D = (a + b) + c
            S = ((pz[v0] - zt) * a + (pz[v1] - zt) * b) + (pz[v2] - zt) * c
            return (D > 20 * E and S > serr) or (D < -20 * E and S < -serr)

        return not (beyond(f0) and beyond(f1))


@pytest.mark.parametrize("nv", [5, 6, 8])
@pytest.mark.parametrize("shift", [0.0, 500.0])
def test_dropped_solids_have_no_nearer_crossing(nv, shift):
    orc = Oracle()
    rng = np.random.default_rng(nv)
    dropped = crossed = 0
    for warp in (0.05, 0.3):
        P, F, _ = W.solid_grid(4, nv=nv, seed=nv, jitter=warp)
        P = (P * rng.uniform(0.3, 3.0, 3) + shift).astype(f32)
        cext = np.abs(P).max()
        for _ in range(1000):
            V = P[F[rng.integers(len(F))]]
            o = (V.mean(0) + rng.normal(size=3) * 10.0 ** rng.uniform(-0.5, 2)).astype(f32)
            wgt = rng.dirichlet(np.ones(nv))
            if rng.random() < 0.3:  # through an edge, nearly
                a, b = EDGES[nv][rng.integers(len(EDGES[nv]))]
                wgt = np.zeros(nv)
                wgt[a] = rng.random()
                wgt[b] = 1 - wgt[a]
            aim = (V * wgt[:, None]).sum(0) + rng.normal(size=3) * 10.0 ** rng.uniform(-8, 0)
            d = aim - o
            d = (d / np.linalg.norm(d) * 10.0 ** rng.uniform(-0.7, 2)).astype(f32)
            axis = [j for j in range(3) if abs(float(d[j])) > 0.1]
            if not axis:
                continue
            n, ts, pos, _ = orc.solid_isect(nv, o.astype(np.float64), d.astype(np.float64),
                                            V.astype(np.float64))
            near = np.inf
            if n:
                ts = np.asarray(ts, f32).reshape(-1)[:2]
                ok = ts[ts >= 0]
                near = float(ok.min()) if len(ok) else np.inf
            crossed += n != 0
            for tb in (MAX, near, near * (1 + 1e-6), near * (1 - 1e-6), near * 0.5, near * 2):
                tb = f32(min(tb, MAX))
                if not may_hit(nv, V, o, d, tb, cext):
                    dropped += 1
                    assert not near < tb, (V, o, d, near, tb)
    assert dropped > 1000 and crossed > 200
