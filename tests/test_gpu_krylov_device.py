"""Krylov steps whose Gram-Schmidt coefficients stay on the device, where a recurrence ends early.

* A zero right-hand side in a block: its column stays zero through the inner near-field solve and does
  not touch the others, which equal their single solves.
* More inner steps than unknowns: the inner recurrence breaks down, and the solution still meets the
  dense system assembled from the operator's own products.
"""
import numpy as np
import pytest

from conftest import relerr
from mlfma_pmchwt_amd import api, geometry

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("prec", [api.FP64, api.FP32])
def test_zero_column_in_an_inner_solved_block(prec):
    op = api.Operator(geometry.icosphere(2, 1.0), integral_equation=api.PMCHWT, eps_r_re=4.0,
                      far_precision=api.FP32, near_precision=api.FP32, max_rhs=4)
    op.set_apply_precision(prec)
    op.set_precond_inner(6)
    B = op.excitation_batch([0.0, 90.0, 0.0], [0.0, 45.0, 90.0], [0.0] * 3)
    B[:, 1] = 0.0
    X, st = op.solve_batch(B, restart=30, tol_rel=1e-6, itr_max=500, precond=api.PRECOND_INNER)
    print(f"[zero column] precision {prec}: {[(s['iterations'], s['rel_residual']) for s in st]}", flush=True)
    assert not X[:, 1].any()
    for j in (0, 2):
        x1, s1 = op.solve(np.ascontiguousarray(B[:, j]), restart=30, tol_rel=1e-6, itr_max=500,
                          precond=api.PRECOND_INNER)
        assert st[j]["converged"] and s1["converged"] and abs(st[j]["iterations"] - s1["iterations"]) <= 2
        assert relerr(X[:, j], x1) <= 1e-4   # 100 x the tolerance, as for the batched preconditioners
    op.close()


@pytest.mark.parametrize("nrhs", [1, 3])
def test_inner_breakdown_meets_the_dense_system(nrhs):
    op = api.Operator(geometry.icosphere(0, 0.3), integral_equation=api.CFIE, max_rhs=4)
    n = op.n
    assert n < 64
    op.set_precond_inner(64)
    A = np.stack([op.apply(np.eye(n)[:, j].astype(complex)) for j in range(n)], axis=1)
    B = op.excitation_batch([0.0, 90.0, 0.0][:nrhs], [0.0, 45.0, 90.0][:nrhs], [0.0] * nrhs)
    tol = 1e-8
    if nrhs == 1:
        x, s = op.solve(np.ascontiguousarray(B[:, 0]), restart=30, tol_rel=tol, itr_max=200, precond=api.PRECOND_INNER)
        X, st = x[:, None], [s]
    else:
        X, st = op.solve_batch(B, restart=30, tol_rel=tol, itr_max=200, precond=api.PRECOND_INNER)
    bound = np.linalg.cond(A) * tol   # error of a solution whose residual meets the tolerance
    for j in range(nrhs):
        print(f"[breakdown] x{nrhs} rhs {j}: {st[j]['iterations']} it {st[j]['rel_residual']:.2e}", flush=True)
        assert st[j]["converged"] and st[j]["rel_residual"] < tol
        assert relerr(X[:, j], np.linalg.solve(A, B[:, j])) <= bound
    op.close()
