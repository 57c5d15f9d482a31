"""BiCGStab and Jacobi COCG whose kernels form their own scalars: the recursion of the separate
finalising launches, whatever the check interval."""
import numpy as np
import pytest
import scipy.sparse as sp

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n", [1, 7, 64, 65, 4097, 49152, 49153, 65537, 66000])
@pytest.mark.parametrize("precision", [64, 32])
def test_check_interval_and_solution(n, precision):
    """Diagonally dominant complex systems (66,000 rows: too many partials, the separate
    launches; BiCGStab uses those from 49,153 rows on).  The histories of the first iterations are those of check_every = 1 (its
    scalars come from the finalising kernel every time): the sums are equal bit for bit, the
    two or three roundings of a scalar's formula may be contracted differently in another
    kernel (1e-16 each, 1e-12 over six iterations of a well-conditioned system).  The
    solution's residual, recomputed in scipy, is below 1e-10."""
    from sucemfem import _hip
    from sucemfem.Utilities.LinalgSolvers import BiCGStabSolver, COCGSolver
    import torch
    torch.cuda.set_device(0)
    rng = np.random.default_rng(n)
    d = 4.0 + rng.random(n) + 1j * rng.random(n)
    A = sp.diags([d], [0], format="csr", dtype=complex)
    if n > 1:
        o = rng.standard_normal(n - 1) + 0.2j
        A = (A + sp.diags([o, o], [1, -1])).tocsr()
    b = rng.standard_normal(n) + 1j * rng.standard_normal(n)
    for cls in (BiCGStabSolver, COCGSolver):
        xs, hist = [], []
        for ce in (1, 8, 64):
            s = cls(A, "diagonal", tol=1e-10, maxiter=500, precision=precision, check_every=ce)
            x = s.solve(b)
            assert s.stats["status"] == 0, (cls, ce, s.stats)
            assert np.linalg.norm(A @ x - b) <= 1.001e-10 * np.linalg.norm(b)
            hist.append(np.array([r for i, r in zip(s._logging_data["id"], s._logging_data["res"])
                                  if isinstance(i, int)]))
        if precision == 64 and n > 64:
            m = 6        # before any of them has converged and replaced its residual
            for h in hist[1:]:
                assert np.all(np.abs(h[:m] - hist[0][:m]) <= 1e-12 * hist[0][:m])
