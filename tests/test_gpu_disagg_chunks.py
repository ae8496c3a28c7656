"""All-right-hand-side disaggregation on split BF16 pairs at its forms: one row tile per workgroup where
there are few items, chunks of 128, 64 and 32 samples otherwise, with leaves of one row tile, of two to
eighteen (items of one to four) and of more than 32, and right-hand sides that end inside a column tile;
against the per-pass FP32 kernel (tuning bit 1 off).

The split drops the product of the two low parts and what 16 bits leave of each factor, 2^-17 each, so
the far field differs by at most 3 x 2^-17 of the summed magnitudes; the near field is the same."""
import numpy as np
import pytest

from conftest import relerr, seeded_x
from mlfma_pmchwt_amd import api, geometry

pytestmark = pytest.mark.gpu
TOL = 3 * 2.0**-17
CASES = {"cfie_few": (geometry.icosphere, 2, 1.0, 0.3, api.CFIE),
         "pmchwt_few": (geometry.icosphere, 2, 1.0, 0.3, api.PMCHWT),
         "cfie_many": (geometry.icosphere, 4, 2.5, 0.3, api.CFIE),
         "pmchwt_many": (geometry.icosphere, 4, 2.5, 0.3, api.PMCHWT),
         "cfie_tiles": (geometry.geodesic_sphere, 20, 0.6, 0.3, api.CFIE),
         "pmchwt_tiles": (geometry.geodesic_sphere, 20, 0.6, 0.3, api.PMCHWT),
         "cfie_large": (geometry.geodesic_sphere, 30, 0.9, 0.45, api.CFIE)}
_op = {}


def _operator(name, near=api.BF16):
    if (name, near) not in _op:
        make, s, r, leaf, ie = CASES[name]
        _op.clear()
        _op[(name, near)] = api.Operator(make(s, r), integral_equation=ie, eps_r_re=2.0, max_rhs=64, leaf_coeff=leaf,
                                         far_precision=api.FP32, near_precision=near)
    return _op[(name, near)]


def _row_tiles(op):
    """Rows of every leaf, and per leaf the row tiles of its last work item (of four)."""
    rows = np.diff(op.level_list(op.max_level, 4)[0])
    tiles = -(-rows // 16)
    return rows, (tiles - 1) % 4 + 1, int((-(-tiles // 4)).sum())


@pytest.mark.parametrize("name", list(CASES))
@pytest.mark.parametrize("nrhs", [2, 8, 9, 17, 40])
def test_disaggregation_chunks_match_per_pass(name, nrhs):
    op = _operator(name)
    rows, last, items = _row_tiles(op)
    if "tiles" in name:   # items of each length, tails inside a row tile, both launch forms
        assert set(last) == {1, 2, 3, 4} and rows.max() > 256 and (rows % 16 > 0).all()
        assert items < 256 <= 2 * items
    elif "large" in name:
        assert rows.max() > 512 and items >= 256
    X = np.stack([seeded_x(op.n, 3300 + j) for j in range(nrhs)], axis=1)
    op.set_apply_precision(api.FP32)
    out = {}
    for bits in (5, 7):
        op.set_tuning(api.FP32, 0, bits)
        out[bits] = op.apply(X)
    op.set_tuning(api.FP32, 0, 7)
    far = relerr(op.stage(api.STAGE_NEAR, X[:, 0]), out[5][:, 0])
    assert far >= 100 * TOL   # a wrong row of the far field stands out
    err = max(relerr(out[7][:, j], out[5][:, j]) for j in range(nrhs))
    print(f"[disagg chunks] {name} x{nrhs}: {err:.2e}", flush=True)
    assert err <= TOL


@pytest.mark.parametrize("name", ["cfie_tiles", "pmchwt_tiles", "cfie_large"])
def test_matrix_core_products_on_large_leaves(name):
    """Blocks on the matrix cores (near product, aggregation and disaggregation of all right-hand sides) against
    single-vector products, in FP64 and FP32, where leaves have items of one to four row tiles."""
    op = _operator(name, api.FP32)
    for R in (2, 9, 17, 33):
        X = np.stack([seeded_x(op.n, 3500 + j) for j in range(R)], axis=1)
        for prec, tol in ((api.FP64, 1e-13), (api.FP32, 2e-6)):   # two orders of FP64 sums, of FP32 sums
            op.set_apply_precision(prec)
            Y = op.apply(X)
            for j in sorted({0, R // 2, R - 1}):
                assert relerr(Y[:, j], op.apply(X[:, j])) <= tol, (R, prec, j)
