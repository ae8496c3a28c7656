"""Cluster translation with two samples per lane: sample tiles that end inside a
workgroup's range, clusters of 1 to 4 members and every number of currents per
pass, single clusters and four side by side per workgroup (from 4,096
wavefronts of a level, here with a count that four does not divide), against
the per-box kernel.

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
CASES.update({name + "_four": CASES[name] for name in list(CASES)})
_op = {}


def _mesh(name):
    if not name.endswith("_four"):
        return geometry.icosphere(2, 1.5)
    mesh = geometry.geodesic_sphere(13, 2.2)   # an egg across the octree's planes: uneven clusters
    mesh.xyz = mesh.xyz * (1.0 + 0.3 * (mesh.xyz / 2.2) @ np.array([0.36, 0.48, 0.8]))[:, None]
    return mesh


def _operator(name):
    if name not in _op:
        ie, eps = CASES[name]
        _op[name] = api.Operator(_mesh(name), integral_equation=ie, eps_r_re=eps[0], eps_r_im=eps[1],
                                 max_rhs=16, far_precision=api.FP32, near_precision=api.FP32)
    return _op[name]


def _uneven_level(op, currents, samples):
    """Whether a level has 4,096 wavefronts of 6 columns and `samples` x 64 samples, and clusters left over by fours."""
    for level in range(2, op.max_level + 1):
        siblings = np.unique(op.level(level)[3], return_counts=True)[1]
        clusters = int(((siblings + 3) // 4).sum())
        tiles = -(-2 * op.grid(1, level)[0] ** 2 // (64 * samples))
        if clusters % 4 and clusters * tiles * (currents // 2) >= 4096:
            return True
    return False


def _forms(op, currents, f64):
    """(columns, samples) per lane that the levels of one pass take, by the wavefronts they give."""
    out = set()
    for level in range(2, op.max_level + 1):
        clusters = int(((np.unique(op.level(level)[3], return_counts=True)[1] + 3) // 4).sum())
        tiles = -(-2 * op.grid(1, level)[0] ** 2 // 64)
        pairs = not f64 and currents >= 4 and clusters * (currents // 2) * (-(-tiles // 2)) >= 1024
        waves = clusters * currents / 2 * (-(-tiles // 2) if pairs else tiles)
        out.add((6 if currents >= (4 if f64 else 2) and waves >= 512 else 3, 2 if pairs else 1))
    return out


@pytest.mark.parametrize("cur,f64,forms", [(4, False, {(3, 1), (6, 1)}), (8, False, {(6, 1), (6, 2)}),
                                           (4, True, {(3, 1), (6, 1)})])
def test_forms_reached(cur, f64, forms):
    """The meshes of this file take every form of the kernel (passes of 4 and 8 vectors of one current)."""
    assert _forms(_operator("cfie"), cur, f64) | _forms(_operator("cfie_four"), cur, f64) >= forms


@pytest.mark.parametrize("name", list(CASES))
@pytest.mark.parametrize("nrhs", [1, 2, 4, 8, 15])
def test_translation_pairs_match_per_box(name, nrhs):
    op = _operator(name)
    if name.endswith("_four") and nrhs >= 8:
        cur = 2 if CASES[name][0] == api.PMCHWT else 1
        assert _uneven_level(op, 8 * cur, 2) and _uneven_level(op, 4 * cur, 1)
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
