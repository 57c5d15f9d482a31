"""Sums over lanes, waves and blocks behind COCG's scalars: every row once."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n", [(1, 1, 1), (2, 1, 3), (4, 3, 5)])
def test_norm_history_matches_exact_sum(n):
    """|r| of the first iterations, reduced over lanes, waves and blocks, against the residual
    recomputed in numpy: a lane left out or taken twice would show at once.  Both sum the same
    squares in FP64 (1e-12), and the recursion's own residual differs from b - A x by its
    rounding (1e-10 after three iterations)."""
    import torch
    from sucemfem.Utilities.Workloads import DeviceProblem
    torch.cuda.set_device(0)
    for order in (1, 2):
        p = DeviceProblem(n, np.array(n) * 0.05, order, 7, (1.0, 2.2), 1)
        c = np.array(n) * 0.025 + 1e-3
        b = p.rhs_dipoles(c[None], np.array([[0.3, 1.0, -0.2]]), 8.0)
        for its in (1, 2, 3):
            x, y, h = torch.zeros_like(b), torch.zeros_like(b), np.zeros(its)
            st = p.solve(8.0, b, x, precision=64, tol=1e-300, max_iter=its, check_every=its, hist=h)
            p.apply(8.0, x, y, precision=64)
            r = np.linalg.norm((b - y).cpu().numpy()) / np.linalg.norm(b.cpu().numpy())
            assert abs(h[-1] - r) <= 1e-10 * max(r, 1e-3), (order, its, h, r)
            assert abs(st["rel_residual"] - r) <= 1e-12 * max(r, 1e-3)
