"""Separable interpolation and anterpolation by row windows against the 9-tap stencil table
(mlfma_get_interp) on single boxes' workspaces, on trees whose grids reach every form: rows of up to 64
samples (groups of 4 rows), up to 192 (2 rows) and up to 256 (1 row), rows longer than a wavefront,
beyond 256 (the 9-tap interpolation) and beyond 340 (anterpolation
in groups of 2 rows); and batched against single products on the same trees."""
import numpy as np
import pytest

from conftest import relerr
from mlfma_pmchwt_amd import api, geometry

pytestmark = pytest.mark.gpu

# radius, eps_r; the largest parent row is that of wavenumber 2 on level 2
TREES = [(0.9, 2.0), (2.5, 2.0), (6.0, 3.0), (9.0, 4.0), (9.0, 9.0)]


def _levels(op, wn):
    return range(3, op.max_level + 1), {l: 2 * op.grid(wn, l)[0] for l in range(2, op.max_level + 1)}


def _directions(op, wn, level):
    _, th, ph, _, _ = op.grid(wn, level)
    t, p = np.meshgrid(th, ph, indexing="ij")
    return np.stack([np.sin(t) * np.cos(p), np.sin(t) * np.sin(p), np.cos(t)], -1).reshape(-1, 3)


@pytest.mark.parametrize("radius,eps", TREES)
def test_rows_match_the_stencil_table(radius, eps):
    op = api.Operator(geometry.icosphere(2, radius), integral_equation=api.PMCHWT, eps_r_re=eps)
    rng = np.random.default_rng(int(10 * radius))
    op.stage(api.STAGE_AGGREGATE, rng.standard_normal(op.n) + 1j * rng.standard_normal(op.n))
    op.stage(api.STAGE_M2M)
    op.stage(api.STAGE_M2L_L2L)
    for wn in (1, 2):
        k = 2 * np.pi * (np.sqrt(eps) if wn == 2 else 1.0)
        children, samples = _levels(op, wn)
        print(f"[rows] radius {radius} wavenumber {wn}: samples per row {samples}", flush=True)
        for c in children:
            taps, w = op.interp(wn, c - 1)
            kp, cen, par = _directions(op, wn, c - 1), op.level(c)[1], op.level(c)[3]
            up_cen = op.level(c - 1)[1]
            sptr, sidx = op.level_list(c - 1, 3)
            for p in {0, len(up_cen) - 1}:   # m2m of a parent from all its children
                want = 0
                for b in sidx[sptr[p]:sptr[p + 1]]:
                    e = np.exp(-1j * k * (kp @ (up_cen[p] - cen[b])))
                    s = op.workspace(wn, 1, 0, c, int(b))
                    want = want + e[:, None] * np.einsum("qt,qtx->qx", w, s[taps])
                assert relerr(op.workspace(wn, 1, 0, c - 1, p), want) <= 1e-13, (wn, c, p)
            dptr, didx = op.level_list(c, 1)
            dvec = op.level_list(c, 2)[1]
            _, _, _, wgl, dphi = op.grid(wn, c)
            qw = np.repeat(wgl, samples[c]) * dphi
            tf = op.tf(wn, c)
            for b in {0, len(cen) // 2}:     # m2l + l2l of a box
                want = np.zeros((len(qw), 3), complex)
                for j in range(dptr[b], dptr[b + 1]):
                    want += (tf[dvec[j]] * qw)[:, None] * op.workspace(wn, 0, 0, c, int(didx[j]))
                if c > 2:
                    p = par[b]
                    e = np.exp(-1j * k * (kp @ (cen[b] - up_cen[p])))
                    v = e[:, None] * op.workspace(wn, 0, 1, c - 1, int(p))
                    for t in range(9):
                        np.add.at(want, taps[:, t], w[:, t, None] * v)
                assert relerr(op.workspace(wn, 0, 1, c, b), want) <= 1e-12, (wn, c, b)


@pytest.mark.parametrize("radius,eps", TREES)
def test_batched_products_on_the_same_trees(radius, eps):
    op = api.Operator(geometry.icosphere(2, radius), integral_equation=api.PMCHWT, eps_r_re=eps, max_rhs=8,
                      far_precision=api.FP32)
    rng = np.random.default_rng(5)
    x = rng.standard_normal((op.n, 15)) + 1j * rng.standard_normal((op.n, 15))   # passes of 8, 4, 2 and 1
    op.set_apply_precision(api.FP64)
    one = np.stack([op.apply(np.ascontiguousarray(x[:, j])) for j in range(15)], 1)
    assert relerr(op.apply(x), one) <= 1e-13
    op.set_apply_precision(api.FP32)
    assert relerr(op.apply(x), one) <= 2e-6   # FP32 far field
