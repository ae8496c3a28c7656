"""Device memory that runs out: an allocation that fails leaves the handle usable."""
import contextlib

import numpy as np
import pytest
import torch

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
                assert np.array_equal(f(), w)
    op.close()
