"""Batched FP64 products (all right-hand sides of a block aggregated and disaggregated at once, up to
32 at a time) against single-vector ones: blocks narrower than a pass, one and several passes, the
column padding's remainders, more than one block of 32, and max_rhs = 1 (passes of one)."""
import numpy as np
import pytest

from conftest import relerr
from mlfma_pmchwt_amd import api, geometry

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("ie,max_rhs", [(api.EFIE, 64), (api.CFIE, 5), (api.PMCHWT, 64), (api.PMCHWT, 1)])
def test_fp64_block_matches_single_vectors(ie, max_rhs):
    op = api.Operator(geometry.geodesic_sphere(8, 0.9), integral_equation=ie, eps_r_re=3.0, eps_r_im=-0.1,
                      max_rhs=max_rhs)
    rng = np.random.default_rng(max_rhs)
    for R in (2, 3, 8, 13, 32, 33, 67):
        x = rng.standard_normal((op.n, R)) + 1j * rng.standard_normal((op.n, R))
        y = op.apply(x)
        for j in sorted({0, 1, R // 2, R - 1}):
            # sums of a few hundred to a few thousand FP64 products in two orders
            assert relerr(y[:, j], op.apply(np.ascontiguousarray(x[:, j]))) <= 1e-13, (R, j)


def test_fp64_block_recorded_and_after_fp32():
    """Both precisions of one handle share the all-RHS buffers; recorded products replay them."""
    op = api.Operator(geometry.geodesic_sphere(8, 0.9), integral_equation=api.PMCHWT, eps_r_re=3.0,
                      far_precision=api.FP32, near_precision=api.BF16, max_rhs=16)
    rng = np.random.default_rng(3)
    x = rng.standard_normal((op.n, 16)) + 1j * rng.standard_normal((op.n, 16))
    want = {}
    for prec in (api.FP64, api.FP32):
        op.set_apply_precision(prec)
        want[prec] = op.apply(x)
    op.set_graphs(True)
    for prec in (api.FP32, api.FP64, api.FP64, api.FP32, api.FP64):
        op.set_apply_precision(prec)
        assert np.array_equal(op.apply(x), want[prec])
