"""Near-field entries from face-pair integrals against the oracle's entry-by-entry quadrature: leaves
of a handful of RWG, flat faces (K of coplanar triangles is 0), each quadrature rule's size class,
lossy media; and leaves of more than 256 RWG (several row and column groups) against smaller leaves."""
import numpy as np
import pytest

from conftest import relerr
from mlfma_pmchwt_amd import api, geometry
import pyoracle

pytestmark = pytest.mark.gpu

SHAPES = {
    "small": (lambda: geometry.icosphere(1, 0.9), 0.3, 7),
    "flat": (lambda: geometry.cube(0.8, 4), 0.3, 4),
    "one_point": (lambda: geometry.cylinder(0.4, 0.9, 12, 5, 3), 0.3, 1),
    "sixteen": (lambda: geometry.icosphere(1, 0.5), 0.3, 16),
}


@pytest.mark.parametrize("ie,eps", [(api.EFIE, (1.0, 0.0)), (api.CFIE, (1.0, 0.0)), (api.PMCHWT, (2.5, -0.1))])
@pytest.mark.parametrize("shape", list(SHAPES))
def test_near_rows_by_face_pairs(shape, ie, eps):
    make, leaf, gauss = SHAPES[shape]
    mesh = make()
    op = api.Operator(mesh, integral_equation=ie, eps_r_re=eps[0], eps_r_im=eps[1], leaf_coeff=leaf, gauss_points=gauss)
    orc = pyoracle.Oracle(mesh, ie=ie, eps=eps, leaf=leaf, gauss=gauss)
    for row in np.unique(np.linspace(0, op.n - 1, 25).astype(int)):
        ca, va = op.near_row(int(row))
        cb, vb = orc.near_row(int(row))
        assert np.array_equal(ca, cb)
        assert relerr(va, vb) <= 1e-12


@pytest.mark.parametrize("ie,eps", [(api.EFIE, (1.0, 0.0)), (api.CFIE, (1.0, 0.0)), (api.PMCHWT, (2.5, -0.1))])
def test_large_leaves_hold_the_same_entries(ie, eps):
    mesh = geometry.geodesic_sphere(11, 0.45)
    ops = [api.Operator(mesh, integral_equation=ie, eps_r_re=eps[0], eps_r_im=eps[1], leaf_coeff=leaf)
           for leaf in (0.45, 0.2)]
    large, small = (np.diff(op.level_list(op.max_level, 4)[0]).max() for op in ops)
    assert large > 256 and small <= 256, (large, small)
    for row in np.unique(np.linspace(0, ops[0].n - 1, 40).astype(int)):
        (ca, va), (cb, vb) = (op.near_row(int(row)) for op in ops)
        common, ia, ib = np.intersect1d(ca, cb, return_indices=True)
        assert len(common) > 20
        # one FP64 quadrature in both; only the order of its sums may differ
        assert relerr(va[ia], vb[ib]) <= 1e-13
