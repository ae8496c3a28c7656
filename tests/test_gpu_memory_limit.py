"""Device memory that runs out: an allocation that fails leaves the handle usable, and the all-RHS
buffers of FP64 products, which only make them faster, give way to what a call cannot do without."""
import contextlib

import numpy as np
import pytest
import torch

from conftest import relerr
from mlfma_pmchwt_amd import api, geometry

pytestmark = pytest.mark.gpu
MIB = 1 << 20


@contextlib.contextmanager
def only_free(size):
    """All of the device's memory but about `size` bytes is taken meanwhile (never written)."""
    torch.cuda.empty_cache()
    hold = []
    for _ in range(4):   # large blocks are rounded, so what one leaves the next takes
        extra = (torch.cuda.mem_get_info()[0] - size) // (2 * MIB) * 2 * MIB
        if extra >= 20 * MIB:
            hold.append(torch.empty(extra, dtype=torch.uint8, device="cuda"))
    assert abs(torch.cuda.mem_get_info()[0] - size) <= 64 * MIB
    try:
        yield
    finally:
        del hold
        torch.cuda.empty_cache()


def test_solves_go_on_after_a_failed_allocation():
    """Bases too large for the device are refused; the buffers that the refused solve gave up are taken
    anew by the next one, which gives what it gave before."""
    op = api.Operator(geometry.geodesic_sphere(10, 0.6), integral_equation=api.CFIE, far_precision=api.FP32,
                      precond_precision=api.BF16, max_rhs=8)
    b = op.excitation_batch([0.0, 90.0, 0.0], [10.0, 50.0, 90.0], [0.0, 20.0, 40.0])
    op.set_precond_poly(np.array([1.0, 0.5, 0.25]))

    def solves(restart):
        for precond in (api.PRECOND_NONE, api.PRECOND_POLY):
            yield lambda: op.solve(np.ascontiguousarray(b[:, 0]), restart=restart, tol_rel=1e-4, itr_max=300,
                                   precond=precond)[0]
            yield lambda: op.solve_batch(b, restart=restart, tol_rel=1e-4, itr_max=300, precond=precond)[0]

    for prec in (api.FP64, api.FP32):
        op.set_apply_precision(prec)
        want = [f() for f in solves(30)]
        with only_free(512 * MIB):
            for f in solves(20_000):     # 0.96 GB a vector's basis
                with pytest.raises(api.MlfmaError, match="memory"):
                    f()
            for f, w in zip(solves(30), want):
                same = np.array_equal(f(), w)
                assert same
    op.close()


def _taken(f):
    free = torch.cuda.mem_get_info()[0]
    f()
    torch.cuda.synchronize()
    return free - torch.cuda.mem_get_info()[0]


def _large(**kw):
    return api.Operator(geometry.geodesic_sphere(14, 2.6), integral_equation=api.CFIE, max_rhs=32, **kw)


def _block(op, R):
    rng = np.random.default_rng(R)
    return rng.standard_normal((op.n, R)) + 1j * rng.standard_normal((op.n, R))


@pytest.mark.parametrize("mode", ["fp64", "fp32"])
def test_fp64_buffers_give_way_to_a_basis(mode):
    """A block solve whose bases fit only where the FP64 buffers were: it runs, and so do the products after it."""
    op = _large(**({} if mode == "fp64" else dict(far_precision=api.FP32)))
    R = 16
    x = _block(op, R)
    op.set_apply_precision(api.FP64)
    op.set_tuning(api.FP64, 0, 5)      # without the matrix-core disaggregation the buffers are not taken
    passes = op.apply(x)
    if mode == "fp32":                  # the FP32 far field needs R columns of FP32, half of them
        op.set_apply_precision(api.FP32)
        op.apply(x)
        op.set_apply_precision(api.FP64)
    op.set_tuning(api.FP64, 0, 7)
    taken = _taken(lambda: op.apply(x))
    print(f"[buffers] {mode}: {taken // MIB} MiB", flush=True)
    assert taken >= 192 * MIB      # half of it stands out against what only_free may be off
    all_rhs = op.apply(x)
    if mode == "fp32":
        op.set_apply_precision(api.FP32)
        x32 = op.apply(x)
        op.set_apply_precision(api.FP64)
    op.set_tuning(api.FP64, 0, 5)
    assert _taken(lambda: op.apply(x)) <= 32 * MIB
    op.set_tuning(api.FP64, 0, 7)
    free = 256 * MIB
    basis = op.n * R * 16
    restart = (free + taken // 2) // basis - 6      # with the six other vectors of a solve
    assert restart > 10
    with only_free(free):
        b = op.excitation_batch([0.0] * R, 10.0 * np.arange(R), [0.0] * R)
        xs, st = op.solve_batch(b, restart=int(restart), tol_rel=1e-2, itr_max=5)
        assert np.isfinite(xs).all()
        after = op.apply(x)
        # the same passes and sums as with the buffers off, or the order of the whole product's sums
        assert relerr(after, passes) <= 1e-13 and relerr(all_rhs, passes) <= 1e-13
        if mode == "fp32":
            op.set_apply_precision(api.FP32)
            same = np.array_equal(op.apply(x), x32)
            assert same
    op.close()


def test_fp64_buffers_are_left_where_little_is_free():
    """They may take an eighth of what is free: with less the product keeps to passes, in an FP32 handle to
    blocks of the columns that its own buffers hold."""
    cases = []
    for kw in ({}, dict(far_precision=api.FP32)):
        for R in (16, 32):
            op = _large(**kw)
            x = _block(op, R)
            op.set_apply_precision(api.FP64)
            op.set_tuning(api.FP64, 0, 5)
            want = op.apply(x)
            if kw:
                op.set_apply_precision(api.FP32)
                op.apply(x)
                op.set_apply_precision(api.FP64)
            op.set_tuning(api.FP64, 0, 7)
            cases.append((op, x, want))
    with only_free(400 * MIB):
        for op, x, want in cases:
            assert _taken(lambda: op.apply(x)) <= 32 * MIB
            assert relerr(op.apply(x), want) <= 1e-13
        op, x, want = cases[-1]    # FP32 products of more right-hand sides than fit, then of as many as before
        op.set_apply_precision(api.FP32)
        y = op.apply(x)
        with pytest.raises(api.MlfmaError, match="memory"):
            op.apply(_block(op, 256))
        same = np.array_equal(op.apply(x), y)
        assert same
    for op, _, _ in cases:
        op.close()
