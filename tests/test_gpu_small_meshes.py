"""Order-2 meshes small enough for 64-cell patches (the operator's default there): partial
patches, patches of one cell, and the COCG form of the operator."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

# 6, 60, 66 (64 + 2), 126 and 1,260 cells
BOXES = [(1, 1, 1), (2, 5, 1), (11, 1, 1), (7, 3, 1), (7, 6, 5)]


def _problem(n, which=None):
    from sucemfem import _hip
    from sucemfem.Utilities.Workloads import DeviceProblem
    which = _hip.MAT_S | _hip.MAT_T | _hip.MAT_S0 if which is None else which
    return DeviceProblem(n, np.array(n) * 0.05, 2, which, (1.0, 2.2, 4.4), 3)


@pytest.mark.parametrize("n", BOXES)
@pytest.mark.parametrize("precision", [64, 32])
def test_default_operator_matches_assembled(n, precision):
    """The default (64-cell) patch operator against the assembled one, with and without the
    PEC row mask.  Both sum the same at most ~130 products per row in the working precision:
    1e-12 (FP64) and 2e-5 (FP32) of max |y| are the bounds of the other patch sizes' test."""
    import torch
    from sucemfem import _hip
    torch.cuda.set_device(0)
    p = _problem(n)
    rng = np.random.default_rng(1)
    x = rng.normal(size=(2, p.ndofs)) + 1j * rng.normal(size=(2, p.ndofs))
    dt = torch.complex128 if precision == 64 else torch.complex64
    xd = torch.as_tensor(x, dtype=dt, device="cuda")
    k0 = 20.0
    out = []
    for assembled in (False, True):
        if assembled:
            p.set_spmv(precision, matrix_free=0, lanes=8, loads=4, blocks=64)
        for pec in (0, 1):
            y = torch.zeros_like(xd)
            _hip.call("sucem_system_apply", p.ctx.handle, p.system.handle.h, k0, precision, pec,
                      2, _hip.ptr(xd), _hip.ptr(y))
            out.append(y.cpu().numpy().astype(np.complex128))
    tol = 1e-12 if precision == 64 else 2e-5
    for a, b in ((0, 2), (1, 3)):
        assert np.abs(out[a] - out[b]).max() <= tol * np.abs(out[b]).max(), (n, precision, a)


@pytest.mark.parametrize("n", BOXES[1:])
@pytest.mark.parametrize("precision", [64, 32])
def test_solve_on_small_patches(n, precision):
    """COCG on 64-cell patches reaches the residual, judged with the assembled operator, and
    agrees with the 192-cell operator's solution (both stop at 1e-10 of |b|)."""
    import torch
    torch.cuda.set_device(0)
    p = _problem(n)
    k0 = 8.0
    c = np.array(n) * 0.025 + 1e-3
    b = p.rhs_dipoles(c[None], np.array([[0.3, 1.0, -0.2]]), k0)
    x, y = torch.zeros_like(b), torch.zeros_like(b)
    st = p.solve(k0, b, x, precision=precision, tol=1e-10)
    assert st["status"] == 0 and st["rel_residual"] <= 1e-10, st
    for q in (32, 64):
        p.set_spmv(q, matrix_free=2, loads=192, blocks=64)
    p.solve(k0, b, y, precision=64, tol=1e-10)
    assert torch.linalg.norm(x - y) <= 1e-6 * torch.linalg.norm(y)
    p.set_spmv(64, matrix_free=0, lanes=8, loads=4, blocks=64)
    p.apply(k0, x, y, precision=64)
    assert torch.linalg.norm(b - y) <= 1.01e-10 * torch.linalg.norm(b)


def test_paired_solve_on_small_patches():
    """Two real systems in one solve on 64-cell patches: each part solves its own."""
    import torch
    from sucemfem import _hip
    torch.cuda.set_device(0)
    p = _problem((5, 4, 4), _hip.MAT_S | _hip.MAT_T)
    rng = np.random.default_rng(4)
    b = rng.normal(size=p.ndofs) + 1e3j * rng.normal(size=p.ndofs)
    b[p.space.pec_mask()] = 0
    bd = torch.as_tensor(b, device="cuda")
    x = torch.zeros_like(bd)
    st = p.solve_coef(1.0, -30.0, 0.0, bd, x, precision=64, tol=1e-11, eliminate_pec=True,
                      paired=True)
    assert st["status"] == 0, st
    y = torch.zeros_like(bd)
    p.set_spmv(64, matrix_free=0, lanes=8, loads=4, blocks=64)
    _hip.call("sucem_system_apply_coef", p.ctx.handle, p.system.handle.h, 1.0, -30.0, 0.0, 64, 1,
              1, _hip.ptr(x), _hip.ptr(y))
    r, bb = (bd - y).cpu().numpy(), b
    assert np.linalg.norm(r.real) <= 1.1e-11 * np.linalg.norm(bb.real)
    assert np.linalg.norm(r.imag) <= 1.1e-11 * np.linalg.norm(bb.imag)


@pytest.mark.parametrize("n,order", [((7, 3, 1), 2), ((7, 6, 5), 2), ((9, 9, 8), 1)])
@pytest.mark.parametrize("precision", [64, 32])
@pytest.mark.parametrize("nvec", [2, 65, 70])
def test_vectors_of_one_call_equal_single_calls(n, order, precision, nvec):
    """Vectors that share a launch (up to 64) give the results of one call each, bit for bit."""
    import torch
    from sucemfem.Utilities.Workloads import DeviceProblem
    torch.cuda.set_device(0)
    p = DeviceProblem(n, np.array(n) * 0.05, order, 7, (1.0, 2.2, 4.4), 3)
    dt = torch.complex128 if precision == 64 else torch.complex64
    g = torch.Generator(device="cuda")
    g.manual_seed(1)
    x = torch.randn(nvec, p.ndofs, dtype=dt, device="cuda", generator=g)
    y, one = torch.zeros_like(x), torch.zeros_like(x)
    p.apply(15.0, x, y, precision=precision, nvec=nvec)
    for v in range(nvec):
        p.apply(15.0, x[v], one[v], precision=precision)
    assert torch.equal(y, one)
