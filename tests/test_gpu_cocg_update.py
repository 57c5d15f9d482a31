"""COCG whose operator forms the next search direction: the same recursion as with the
separate update, whatever the check interval (the update is left to the operator only between
host checks)."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n,order", [((2, 5, 1), 2), ((7, 6, 5), 2), ((21, 20, 20), 2),
                                     ((3, 4, 5), 1), ((13, 9, 11), 1)])
@pytest.mark.parametrize("precision", [64, 32])
def test_check_interval_does_not_change_the_recursion(n, order, precision):
    """check_every = 1 updates p in its own kernel after every iteration; 5, 16 and 64 leave it
    to the operator in between.  After 40 iterations from the same start the residual
    histories agree: bit for bit in the update's formula, and to the rounding of the
    reductions' order (FP64 1e-9, FP32 1e-3 relative over the history, growing with the
    recursion)."""
    import torch
    from sucemfem import _hip
    from sucemfem.Utilities.Workloads import DeviceProblem
    torch.cuda.set_device(0)
    p = DeviceProblem(n, np.array(n) * 0.03, order, 7, (1.0, 2.2, 4.4), 3)
    k0 = 9.0
    c = np.array(n) * 0.015 + 1e-3
    b = p.rhs_dipoles(c[None], np.array([[0.3, 1.0, -0.2]]), k0)
    hists = []
    for ce in (1, 5, 16, 64):
        x = torch.zeros_like(b)
        h = np.zeros(40)
        # FP32 without residual replacement (a tiny ru_delta)
        p.solve(k0, b, x, precision=precision, tol=1e-300, max_iter=40, check_every=ce,
                ru_delta=1e-300, hist=h)
        hists.append((h, x.cpu().numpy()))
    h0, x0 = hists[0]
    assert np.all(h0[:20] > 0)
    tol = 1e-9 if precision == 64 else 1e-3
    for h, x in hists[1:]:
        live = h0 > (1e-12 if precision == 64 else 1e-5)
        assert np.all(np.abs(h - h0)[live] <= tol * h0[live])
        assert np.linalg.norm(x - x0) <= tol * np.linalg.norm(x0)
