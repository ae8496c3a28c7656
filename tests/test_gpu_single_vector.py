"""Single-vector far-field kernels on few leaves (sample tiles, rows split over wavefronts) against
sums over the stored patterns (mlfma_get_pattern)."""
import numpy as np
import pytest

from mlfma_pmchwt_amd import api, geometry

pytestmark = pytest.mark.gpu

# leaves of 1 to 15 RWG, of about 100 and of more than 256 (several x chunks); both storages of x
MESHES = [(4, 0.9, 0.3), (12, 0.45, 0.3), (17, 0.45, 0.45)]


@pytest.mark.parametrize("ie", [api.EFIE, api.CFIE, api.PMCHWT])
@pytest.mark.parametrize("freq,radius,leaf", MESHES)
def test_aggregation_tiles(freq, radius, leaf, ie):
    op = api.Operator(geometry.geodesic_sphere(freq, radius), integral_equation=ie, eps_r_re=3.0, leaf_coeff=leaf)
    rng = np.random.default_rng(freq + ie)
    x = rng.standard_normal(op.n) + 1j * rng.standard_normal(op.n)
    op.stage(api.STAGE_AGGREGATE, x)
    ptr, rwg = op.level_list(op.max_level, 4)
    sizes = np.diff(ptr)
    for t in {0, len(sizes) - 1, int(sizes.argmax()), int(sizes.argmin()), len(sizes) // 2}:
        for wn in (1, 2) if ie == api.PMCHWT else (1,):
            v = np.stack([op.pattern(wn, 0, int(i)) for i in rwg[ptr[t]:ptr[t + 1]]])
            for cur in (0, 1) if ie == api.PMCHWT else (0,):
                xs = x[cur * op.n_rwg + rwg[ptr[t]:ptr[t + 1]]]
                want = np.einsum("nqc,n->qc", v, xs)
                # two orders of one FP64 sum: 2 n eps sum |v x|
                bound = 2 * len(xs) * np.finfo(float).eps * np.einsum("nqc,n->qc", np.abs(v), np.abs(xs))
                got = op.workspace(wn, cur, 0, op.max_level, t)
                assert np.all(np.abs(got - want) <= bound + 1e-300), (t, wn, cur)
