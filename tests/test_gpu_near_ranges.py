"""Single-vector near product over column ranges of large leaves: y = Z_near x against the stored
rows read back one by one (mlfma_get_near_row), in the equations' storage layouts."""
import numpy as np
import pytest

from mlfma_pmchwt_amd import api, geometry

pytestmark = pytest.mark.gpu

# leaves of 13 to 50 rows (kept whole), of about 100 (several column groups per workgroup), and of
# more than 512 (several row passes of a workgroup, one column group); one and three planes, both storages;
# the last pair has 392 leaves of up to 1.3 MB in FP64: column ranges there, whole in FP32
CASES = [("whole", 4, 0.5, 0.3, api.PMCHWT, api.FP64), ("groups", 12, 0.4, 0.3, api.EFIE, api.FP64),
         ("groups", 9, 0.4, 0.3, api.PMCHWT, api.FP64), ("rows", 17, 0.45, 0.45, api.EFIE, api.FP64),
         ("rows", 17, 0.45, 0.45, api.PMCHWT, api.FP64), ("groups", 11, 0.4, 0.3, api.CFIE, api.FP32),
         ("groups", 9, 0.4, 0.3, api.PMCHWT, api.FP32),
         ("whole", 20, 1.4, 0.3, api.PMCHWT, api.FP64), ("whole", 20, 1.4, 0.3, api.PMCHWT, api.FP32)]


@pytest.mark.parametrize("kind,freq,radius,leaf,ie,near", CASES)
def test_near_product_matches_stored_rows(kind, freq, radius, leaf, ie, near):
    op = api.Operator(geometry.geodesic_sphere(freq, radius), integral_equation=ie, eps_r_re=3.0, leaf_coeff=leaf,
                      near_precision=near)
    ptr, _ = op.level_list(op.max_level, 4)
    rows = np.diff(ptr)
    assert {"whole": rows.max() <= 64, "groups": 64 < rows.max() <= 512, "rows": rows.max() > 512}[kind], rows.max()
    rng = np.random.default_rng(freq)
    x = rng.standard_normal(op.n) + 1j * rng.standard_normal(op.n)
    if near == api.FP32:   # the FP32 copy serves FP32-mode products: the whole product against the FP64 one
        y64 = op.apply(x)
        op.set_apply_precision(api.FP32)
        y = op.apply(x)
        # entries rounded once to FP32 (2^-24 each), FP64 sums
        assert np.linalg.norm(y - y64) <= 2.0 ** -23 * np.linalg.norm(y64)
        return
    y = op.stage(api.STAGE_NEAR, x)
    for row in np.unique(np.concatenate([[0, op.n - 1], rng.integers(0, op.n, 24)])):
        cols, vals = op.near_row(int(row))
        # two orders of one FP64 sum of len(cols) products differ by at most 2 len eps sum |z x|
        bound = 2 * len(cols) * np.finfo(float).eps * np.sum(np.abs(vals) * np.abs(x[cols]))
        assert abs(y[row] - vals @ x[cols]) <= bound
