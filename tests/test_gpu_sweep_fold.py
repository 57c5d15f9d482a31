"""Batched sweeps whose kernels form their own scalars: group widths, orders and sizes against
single solves, with a system that converges long before its group and one without a source."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n,order", [((2, 1, 1), 1), ((5, 4, 6), 1), ((13, 12, 11), 1),
                                     ((1, 2, 1), 2), ((5, 4, 3), 2)])
@pytest.mark.parametrize("width", [1, 2, 4, 8])
@pytest.mark.parametrize("precision", [64, 32])
def test_groups_match_single_solves(n, order, width, precision):
    """Both stop at 1e-10 of |b|; the systems' condition leaves 1e-6 between two such
    solutions.  The frozen system keeps its solution, the one with b = 0 stays zero."""
    import torch
    from sucemfem.Utilities.Workloads import DeviceProblem
    torch.cuda.set_device(0)
    p = DeviceProblem(n, np.array(n) * 0.03, order, 7, (1.0, 2.2, 4.4), 3)
    nb = width + 1
    k0s = np.linspace(0.5, 12.0, nb)
    rng = np.random.default_rng(0)
    B = rng.standard_normal((nb, p.ndofs)) + 1j * rng.standard_normal((nb, p.ndofs))
    if width > 2:
        B[1] = 0.0
    Bd = torch.as_tensor(B, device="cuda")
    X = torch.zeros_like(Bd)
    st = p.solve_sweep(k0s, Bd, X, precision=precision, tol=1e-10, width=width)
    for j in range(nb):
        if not np.any(B[j]):
            assert torch.count_nonzero(X[j]) == 0
            continue
        assert st[j]["status"] == 0 and st[j]["rel_residual"] <= 1e-10, (j, st[j])
        x = torch.zeros_like(Bd[j])
        p.solve(k0s[j], Bd[j].contiguous(), x, precision=64, tol=1e-10)
        assert torch.linalg.norm(X[j] - x) <= 1e-6 * torch.linalg.norm(x), j
