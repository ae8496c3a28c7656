"""Excitations of several incidences per launch and far fields of several directions per thread.

Excitation columns equal single excitations: the same sums per column, so up to the contraction of a
product and a sum, one rounding for each of the 2 n quadrature terms of a function.  The far field of
many directions (four per thread) equals that of few (one per thread) up to where the projection is
taken: about eight roundings for each of T = 2 n N terms, independent, so 8 sqrt(T) u of the summed
magnitudes, which are at most some ten times the largest field of an open angle range.  The same with
a current per direction, as in a monostatic sweep."""
import numpy as np
import pytest

from conftest import seeded_x
from mlfma_pmchwt_amd import api, geometry

pytestmark = pytest.mark.gpu
U = 2.0**-53
POINTS = 16   # at most, per face
CASES = {"efie": api.EFIE, "cfie": api.CFIE, "pmchwt": api.PMCHWT}


def _operator(name):
    return api.Operator(geometry.icosphere(3, 0.8), integral_equation=CASES[name], eps_r_re=3.0)


@pytest.mark.parametrize("name", list(CASES))
@pytest.mark.parametrize("n_inc", [2, 8, 9, 17])
def test_excitation_batch_matches_single(name, n_inc):
    op = _operator(name)
    pol, th, ph = (90.0 * (np.arange(n_inc) % 2), 7.0 + 9.0 * np.arange(n_inc), 11.0 * np.arange(n_inc))
    B = op.excitation_batch(pol, th, ph)
    for j in range(n_inc):
        b = op.excitation(pol[j], th[j], ph[j])
        assert np.abs(B[:, j] - b).max() <= 2 * POINTS * U * np.abs(b).max()
    op.close()


@pytest.mark.parametrize("name", list(CASES))
@pytest.mark.parametrize("nang", [512, 513, 515])
def test_many_directions_match_few(name, nang):
    op = _operator(name)
    assert -(-op.n_rwg // 256) * nang >= 4096 > -(-op.n_rwg // 256) * 100
    current = seeded_x(op.n, 77)
    th, ph = np.linspace(0.0, 180.0, nang), np.linspace(0.0, 90.0, nang)
    many = np.asarray(op.rcs(current, th, ph))
    few = np.concatenate([np.asarray(op.rcs(current, th[a:a + 100], ph[a:a + 100])) for a in range(0, nang, 100)])
    field = lambda db: 10.0 ** (db / 20.0)
    err = np.abs(field(many) - field(few)).max() / field(few).max()
    bound = 10 * 8 * np.sqrt(2 * POINTS * op.n_rwg) * U
    print(f"[directions] {name} x{nang}: {err:.2e} bound {bound:.2e}", flush=True)
    assert err <= bound
    op.close()


@pytest.mark.parametrize("name", ["cfie", "pmchwt"])
def test_many_directions_with_a_current_each(name):
    """The monostatic sweep's far field (a current per direction, four directions per thread, a count that four
    does not divide) against one direction at a time of the same solutions."""
    op = api.Operator(geometry.icosphere(4, 0.9), integral_equation=CASES[name], eps_r_re=3.0, max_rhs=8)
    nang = 141
    assert -(-op.n_rwg // 256) * nang >= 4096
    th, ph = np.linspace(3.0, 177.0, nang), np.linspace(0.0, 90.0, nang)
    how = dict(restart=50, tol_rel=1e-12, tol_abs=0.0, itr_max=2)   # solutions of two steps
    many, _ = op.monostatic(th, ph, pol=0.0, **how)
    x, _ = op.solve_batch(op.excitation_batch(np.zeros(nang), th, ph), **how)
    few = np.concatenate([np.asarray(op.rcs(np.ascontiguousarray(x[:, a]), th[a:a + 1], ph[a:a + 1]))
                          for a in range(nang)])
    field = lambda db: 10.0 ** (db / 20.0)
    err = np.abs(field(np.asarray(many)) - field(few)).max() / field(few).max()
    bound = 10 * 8 * np.sqrt(2 * POINTS * op.n_rwg) * U
    print(f"[currents] {name}: {err:.2e} bound {bound:.2e}", flush=True)
    assert err <= bound
    op.close()
