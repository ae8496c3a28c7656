"""Cluster translation with two samples per lane: sample tiles that end inside a
workgroup's range, clusters of 1 to 4 members and every number of currents per
pass, against the per-box kernel.

A member's sum runs over the same at most 189 sources in the same order in both
kernels, so they differ only by how products and sums are contracted: at most
one rounding of the unit u per source, 189 u of the result."""
import numpy as np
import pytest

from conftest import relerr, seeded_x
from mlfma_pmchwt_amd import api, geometry

pytestmark = pytest.mark.gpu
BOUND = {api.FP64: 189 * 2.0**-53, api.FP32: 189 * 2.0**-24}
CASES = {"cfie": (api.CFIE, (1.0, 0.0)), "pmchwt_lossy": (api.PMCHWT, (2.5, -0.1))}
_op = {}


def _operator(name):
    if name not in _op:
        ie, eps = CASES[name]
        _op[name] = api.Operator(geometry.icosphere(2, 1.5), integral_equation=ie, eps_r_re=eps[0], eps_r_im=eps[1],
                                 max_rhs=16, far_precision=api.FP32, near_precision=api.FP32)
    return _op[name]


@pytest.mark.parametrize("name", list(CASES))
@pytest.mark.parametrize("nrhs", [1, 2, 4, 8, 15])
def test_translation_pairs_match_per_box(name, nrhs):
    op = _operator(name)
    X = np.stack([seeded_x(op.n, 2100 + j) for j in range(nrhs)], axis=1)
    for prec in (api.FP64, api.FP32):
        op.set_apply_precision(prec)
        out = {}
        for bits in (3, 7, 15):
            op.set_tuning(prec, 0, bits)
            out[bits] = op.apply(X)
        op.set_tuning(prec, 0, 7)
        err = max(relerr(out[7][:, j], out[3][:, j]) for j in range(nrhs))
        print(f"[pairs] {name} x{nrhs} precision {prec}: {err:.2e}")
        assert err <= BOUND[prec]
        assert np.array_equal(out[15], out[7])   # bit 3 selects nothing
    op.set_apply_precision(api.FP64)
