"""The matrix pre-test of the tiles of 16 (swift_amd/csrc/sph_tile.h and the
chunk engine) never rejects a pair that the pair contract accepts, nor does
the box cull before it.

The test forms |x_j|^2 - 2 x_i . x_j + (|x_i|^2 - R) on float positions in
the tile frame -- relative to the centre of the tile's box, in units of its
largest radius -- with the squares taken 2^-18 low and the radii 2^-20 high;
a negative value passes.  Emulated with float32 in both extremes of the
matrix unit's accumulation: every product and sum rounded, and one fused
chain in either order.
"""
from __future__ import annotations

import numpy as np

from parity import contract_dx
from test_pretest import _pretest_radius2, _r2

f32 = np.float32
SQ_LO = f32(1.0 - 2.0 ** -18)
RAD_UP = f32(1.0 + 2.0 ** -20)


def _fma(a, b, c):
    return (a.astype(np.float64) * b.astype(np.float64) + c).astype(f32)


def _forms(vi, vj, sqj, c):
    """The accumulated value in three orders (lists of float32 arrays)."""
    b = [(f32(-2.0) * vi[:, k]).astype(f32) for k in range(3)]
    terms = [(vj[:, k], b[k]) for k in range(3)] + [(sqj, np.ones_like(sqj))]
    out = []
    for order in ((0, 1, 2, 3), (3, 2, 1, 0)):
        acc = c
        for k in order:
            acc = _fma(terms[k][0], terms[k][1], acc)
        out.append(acc)
    acc = np.zeros_like(c)
    for x, y in terms:
        acc = (acc + (x * y).astype(f32)).astype(f32)
    out.append((acc + c).astype(f32))
    return out


def _case(rng, symmetric, n_tiles=150):
    missed = culled = missed_bare = total = 0
    for _ in range(n_tiles):
        w = 10 ** rng.uniform(-3, 3)
        eps = f32(1.5 * w * 2.0 ** -19)
        H = w * 10 ** rng.uniform(-2.5, 0)
        a = min(H * 10 ** rng.uniform(-1, 1.5), w)  # tile extent
        ct = rng.uniform(0, 1, 3) * (w - a) + w + a / 2
        xi = ct + rng.uniform(-a / 2, a / 2, (16, 3))
        Hi = H * rng.uniform(0.5, 1.0, 16)
        Hi[0] = H
        hg2 = (f32(Hi) * f32(Hi)).astype(f32)
        invR = f32(1.0) / np.sqrt(hg2.max()).astype(f32)
        invR2 = ((invR * invR).astype(f32) * RAD_UP).astype(f32)
        corner_i = np.floor(ct / w) * w
        rel = (xi - corner_i).astype(f32)
        cen = corner_i + (f32(0.5) * (rel.min(0) + rel.max(0))).astype(np.float64)
        fi = (xi - cen).astype(f32)
        half = np.abs(fi).max(0)
        n = 3000
        k = rng.integers(0, 16, n)
        d = rng.normal(size=(n, 3))
        d /= np.linalg.norm(d, axis=1)[:, None]
        # radius of the pair: H_i, or H_j where that is the larger
        Hj = Hi[k] * (rng.uniform(0.3, 3.0, n) if symmetric else 1.0)
        Hj = np.minimum(Hj, w)
        hj2 = (f32(Hj) * f32(Hj)).astype(f32)
        R = np.maximum(hg2[k], hj2) if symmetric else hg2[k]
        r = np.sqrt(R.astype(np.float64)) * (1 - rng.uniform(-1e-6, 1e-5, n))
        xj = xi[k] + d * r[:, None]
        cj = np.floor(xj / w)
        ok = np.all((cj >= 0) & (cj <= 3), axis=1)
        k, xj, cj, hj2, R = k[ok], xj[ok], cj[ok], hj2[ok], R[ok]
        pj = (xj - cj * w).astype(f32)
        qoff = (cj * w - cen).astype(f32)
        vj = ((pj + qoff).astype(f32) * invR).astype(f32)
        vi = (fi[k] * invR).astype(f32)
        sqi = (_r2(vi[:, 0], vi[:, 1], vi[:, 2]) * SQ_LO).astype(f32)
        sqj = (_r2(vj[:, 0], vj[:, 1], vj[:, 2]) * SQ_LO).astype(f32)
        pre = _pretest_radius2(hg2[k], eps)
        ci = _fma(-(pre * RAD_UP).astype(f32), np.full_like(pre, invR2), sqi)
        val = _forms(vi, vj, sqj, ci)
        passed = [v < 0 for v in val]
        box_r = _pretest_radius2(np.full_like(R, hg2.max()), eps)
        if symmetric:
            prej = _pretest_radius2(hj2, eps)
            sj = _fma(-(prej * RAD_UP).astype(f32),
                      np.full_like(prej, invR2), sqj)
            passed = [p | (v < 0) for p, v in zip(passed,
                                                  _forms(vi, vj, sj, sqi))]
            box_r = np.maximum(box_r, prej)
        # the box of one candidate
        gap = np.maximum(f32(0), np.maximum((pj + qoff).astype(f32) - half,
                                            -half - (pj + qoff).astype(f32)))
        gap2 = _r2(*[gap[:, q].astype(f32) for q in range(3)])
        dc = contract_dx(xi[k], xj, np.floor(xi[k] / w).astype(np.int64),
                         cj.astype(np.int64), w)
        inside = _r2(dc[:, 0], dc[:, 1], dc[:, 2]) < R
        bare = _r2(*[(vi - vj)[:, q].astype(f32) for q in range(3)]) < (
            R * (invR * invR).astype(f32)).astype(f32)
        missed += int((inside & ~np.all(passed, axis=0)).sum())
        culled += int((inside & ~(gap2 < box_r)).sum())
        missed_bare += int((inside & ~bare).sum())
        total += int(inside.sum())
    return missed, culled, missed_bare, total


def test_matrix_pretest_never_rejects_a_contract_neighbour():
    for symmetric in (False, True):
        missed, culled, missed_bare, total = _case(
            np.random.default_rng(21 + symmetric), symmetric)
        assert total > 100000
        assert missed == 0
        assert culled == 0
        assert missed_bare > 0  # the widening is needed
