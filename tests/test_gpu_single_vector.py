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


# fewer than 2,048 rows (one row a block), up to 16,384 (four rows, samples split), above (rows by
# fours), with row counts and sample counts that are no multiple of the tiles
@pytest.mark.parametrize("ie", [api.EFIE, api.PMCHWT])
@pytest.mark.parametrize("freq,radius", [(5, 0.7), (13, 0.9), (25, 1.3)])
def test_disaggregation_rows(freq, radius, ie):
    op = api.Operator(geometry.geodesic_sphere(freq, radius), integral_equation=ie, eps_r_re=3.0, eps_r_im=-0.2)
    n = op.n_rwg
    rng = np.random.default_rng(freq + ie)
    op.stage(api.STAGE_AGGREGATE, rng.standard_normal(op.n) + 1j * rng.standard_normal(op.n))
    op.stage(api.STAGE_M2M)
    op.stage(api.STAGE_M2L_L2L)
    y = op.stage(api.STAGE_FAR)
    ptr, rwg = op.level_list(op.max_level, 4)
    box = np.empty(n, dtype=int)
    for t in range(len(ptr) - 1):
        box[rwg[ptr[t]:ptr[t + 1]]] = t
    order = np.argsort(box, kind="stable")        # internal rows are leaf by leaf
    k0, eta0 = 2 * np.pi, 119.9169832 * np.pi
    er = 3.0 - 0.2j
    for i in np.unique(np.concatenate([order[:5], order[-5:], order[ptr[1] - 3:ptr[1] + 3], rng.integers(0, n, 8)])):
        want, size = np.zeros(2, complex), np.zeros(2)
        for wn, k in enumerate([k0, k0 * np.sqrt(er)] if ie == api.PMCHWT else [k0], 1):
            v = op.pattern(wn, 1, int(i))
            b = [op.workspace(wn, c, 1, op.max_level, box[i]) for c in range(2 if ie == api.PMCHWT else 1)]
            if ie != api.PMCHWT:
                c = (k * eta0 / (4 * np.pi)) * (k / (4 * np.pi))
                want[0], size[0] = c * np.sum(v * b[0]), abs(c) * np.sum(np.abs(v * b[0]))
                continue
            _, th, ph, _, _ = op.grid(wn, op.max_level)
            T, P = np.meshgrid(th, ph, indexing="ij")
            kp = np.stack([np.sin(T) * np.cos(P), np.sin(T) * np.sin(P), np.cos(T)], -1).reshape(-1, 3)
            c, z = k * k / (16 * np.pi * np.pi), 1.0 if wn == 1 else np.sqrt(1.0 / er)
            lj, lm = (np.sum(v * b[q]) for q in (0, 1))
            kj, km = (np.sum(v * np.cross(kp, b[q])) for q in (0, 1))
            want += [c * (z * lj - km), c * (kj + lm / z)]
            size += abs(c) * 4 * np.sum(np.abs(v)) * max(np.abs(b[0]).max(), np.abs(b[1]).max())
        got = [y[i]] + ([y[n + i]] if ie == api.PMCHWT else [])
        # sums of 3K products in two orders, a few roundings per product
        bound = (6 * v.size + 64) * np.finfo(float).eps * size
        assert np.all(np.abs(np.array(got) - want[:len(got)]) <= bound[:len(got)]), i


# the three forms of the disaggregation again, in FP32
@pytest.mark.parametrize("freq,radius", [(8, 0.9), (16, 1.1), (26, 1.4)])
def test_fp32_disaggregation_keeps_its_constants(freq, radius):
    """FP32 sums of the second wavenumber meet their constants in FP64.  The constants c, c z and c / z of this
    permittivity round to FP32 by 0.98 units u = 2^-24 of either sign, which would scale the two outputs of one
    current apart by 1.96 u in every row alike.  The scales of the two outputs' errors along their exact parts
    come from one workspace, so what its own rounding adds to both cancels; the rest is 2,000 rows' independent
    errors of about 3 u, 0.07 u of each scale."""
    eps = 4.0322144
    op = api.Operator(geometry.geodesic_sphere(freq, radius), integral_equation=api.PMCHWT, eps_r_re=eps,
                      far_precision=api.FP32)
    n = op.n_rwg
    assert {8: n < 2048, 16: 2048 <= n < 16384, 26: n >= 16384}[freq]
    rng = np.random.default_rng(freq)
    ptr, rwg = op.level_list(op.max_level, 4)
    box = np.empty(n, dtype=int)
    for t in range(len(ptr) - 1):
        box[rwg[ptr[t]:ptr[t + 1]]] = t
    rows = rng.permutation(n)[:2000]
    v = np.stack([op.pattern(2, 1, int(i)) for i in rows])
    _, th, ph, _, _ = op.grid(2, op.max_level)
    T, P = np.meshgrid(th, ph, indexing="ij")
    kp = np.stack([np.sin(T) * np.cos(P), np.sin(T) * np.sin(P), np.cos(T)], -1).reshape(-1, 3)
    for cur in (0, 1):
        x = np.zeros(op.n, dtype=complex)
        x[cur * n:(cur + 1) * n] = rng.standard_normal(n) + 1j * rng.standard_normal(n)
        op.set_apply_precision(api.FP64)
        y = op.apply(x)
        far = y - op.stage(api.STAGE_NEAR, x)
        op.set_apply_precision(api.FP32)
        err = op.apply(x) - y      # the near product is the same FP64 one
        assert np.linalg.norm(err) <= 2e-6 * np.linalg.norm(far)   # FP32 sums throughout
        op.stage(api.STAGE_AGGREGATE, x)
        op.stage(api.STAGE_M2M)
        op.stage(api.STAGE_M2L_L2L)
        b = np.stack([op.workspace(2, cur, 1, op.max_level, t) for t in range(len(ptr) - 1)])[box[rows]]
        c, z = eps / 4.0, np.sqrt(1.0 / eps)
        lin, curl = c * np.einsum("nqx,nqx->n", v, b), c * np.einsum("nqx,nqx->n", v, np.cross(kp, b))
        parts = (lin * z, curl) if cur == 0 else (-curl, lin / z)
        scale = [np.vdot(p, e) / np.vdot(p, p).real for p, e in zip(parts, (err[rows], err[n + rows]))]
        print(f"[constants] {n} RWG current {cur}: {scale[0] * 2**24:.2f} {scale[1] * 2**24:.2f} u", flush=True)
        assert abs(scale[0] - scale[1]) <= 0.5 * 2.0**-24
    op.close()
