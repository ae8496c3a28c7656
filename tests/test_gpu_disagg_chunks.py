"""All-right-hand-side disaggregation on split BF16 pairs at its forms: one row tile per workgroup where
there are few items, chunks of 128, 64 and 32 samples otherwise, with leaves that end inside a row tile
and right-hand sides that end inside a column tile; against the per-pass FP32 kernel (tuning bit 1 off).

The split drops the product of the two low parts and what 16 bits leave of each factor, 2^-17 each, so
the far field differs by at most 3 x 2^-17 of the summed magnitudes; the near field is the same."""
import numpy as np
import pytest

from conftest import relerr, seeded_x
from mlfma_pmchwt_amd import api, geometry

pytestmark = pytest.mark.gpu
TOL = 3 * 2.0**-17
CASES = {"cfie_few": (2, 1.0, api.CFIE), "pmchwt_few": (2, 1.0, api.PMCHWT), "cfie_many": (4, 2.5, api.CFIE),
         "pmchwt_many": (4, 2.5, api.PMCHWT)}
_op = {}


def _operator(name):
    if name not in _op:
        s, r, ie = CASES[name]
        _op[name] = api.Operator(geometry.icosphere(s, r), integral_equation=ie, eps_r_re=2.0, max_rhs=64,
                                 far_precision=api.FP32, near_precision=api.BF16)
    return _op[name]


@pytest.mark.parametrize("name", list(CASES))
@pytest.mark.parametrize("nrhs", [2, 8, 9, 17, 40])
def test_disaggregation_chunks_match_per_pass(name, nrhs):
    op = _operator(name)
    X = np.stack([seeded_x(op.n, 3300 + j) for j in range(nrhs)], axis=1)
    op.set_apply_precision(api.FP32)
    out = {}
    for bits in (5, 7):
        op.set_tuning(api.FP32, 0, bits)
        out[bits] = op.apply(X)
    op.set_tuning(api.FP32, 0, 7)
    err = max(relerr(out[7][:, j], out[5][:, j]) for j in range(nrhs))
    print(f"[disagg chunks] {name} x{nrhs}: {err:.2e}", flush=True)
    assert err <= TOL
