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


# either side of 2,048 patches, up to which the kernels form their own scalars and sum the
# shared rows themselves: 2,042 and 2,136 patches of 256 order-1 cells, 2,154 of 192 order-2 ones
@pytest.mark.parametrize("n,order,width,precision", [
    ((44, 44, 45), 1, 2, 64), ((45, 45, 45), 1, 1, 64), ((45, 45, 45), 1, 2, 64),
    ((45, 45, 45), 1, 4, 32), ((45, 45, 45), 1, 8, 64), ((45, 45, 45), 1, 8, 32),
    ((41, 41, 41), 2, 2, 64)])
def test_groups_on_meshes_of_many_patches(n, order, width, precision):
    """The recursion with and without launches of its own for the scalars and the shared rows:
    every system reaches its residual, recomputed with the assembled operator, by its own
    recursion (none is finished by the single solver); the system with b = 0 stays zero.  In FP64
    the first system takes about the iterations of a single solve, which differs in rounding
    only (a few per cent); in FP32 the two also end their cycles by different rules."""
    import torch
    from sucemfem.Utilities.Workloads import DeviceProblem
    torch.cuda.set_device(0)
    p = DeviceProblem(n, np.array(n) * 0.03, order, 7, (1.0, 2.2, 4.4), 3)
    assert (p.patch_info(192 if order == 2 else 256)["patches"] > 2048) == (n != (44, 44, 45))
    k0s = np.linspace(1.0, 8.0, width + 1)
    g = torch.Generator(device="cuda")
    g.manual_seed(0)
    B = torch.randn(width + 1, p.ndofs, dtype=torch.complex128, device="cuda", generator=g)
    if width > 2:
        B[1] = 0.0
    X = torch.zeros_like(B)
    tol = 1e-9
    st = p.solve_sweep(k0s, B, X, precision=precision, tol=tol, width=width)
    x = torch.zeros_like(B[0])
    if precision == 64:
        one = p.solve(k0s[0], B[0].contiguous(), x, precision=64, tol=tol)
        assert abs(st[0]["iterations"] - one["iterations"]) <= 0.1 * one["iterations"], (st[0], one)
    p.set_spmv(64, matrix_free=0, lanes=16, loads=4, blocks=2048)
    y = torch.zeros_like(x)
    for j in range(width + 1):
        if torch.count_nonzero(B[j]) == 0:
            assert torch.count_nonzero(X[j]) == 0
            continue
        assert st[j]["status"] == 0 and st[j]["fp64_finish"] == 0, (j, st[j])
        p.apply(k0s[j], X[j].contiguous(), y, precision=64)
        assert torch.linalg.norm(B[j] - y) <= 1.01 * tol * torch.linalg.norm(B[j]), (j, st[j])
