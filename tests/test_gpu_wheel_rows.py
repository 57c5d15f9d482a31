"""Preconditioner rows that take their edges and faces in batches, on wheels of m cells around
an axis edge: the axis has m faces and its ends m + 1 edges and 2 m faces, so that m runs
through the remainders and the rows longer than a batch."""
import numpy as np
import pytest

import oracle as O

pytestmark = pytest.mark.gpu


def _wheel(m):
    t = 2 * np.pi * np.arange(m) / m
    co = np.vstack([[[0, 0, -0.02], [0, 0, 0.03]],
                    np.c_[0.04 * np.cos(t), 0.05 * np.sin(t), 0.01 * np.cos(3 * t)]])
    ce = np.array([[0, 1, 2 + i, 2 + (i + 1) % m] for i in range(m)])
    return co, np.sort(ce, axis=1)


@pytest.mark.parametrize("order", [1, 2])
@pytest.mark.parametrize("m", [3, 4, 6, 7, 15, 16, 17, 20, 21, 32, 33, 41])
def test_rows_of_wheels_match_the_oracle(m, order):
    """z = M^-1 r against the oracle's: the same sums in another order, at most 2 m + 1 = 83
    terms a row (FP64 1e-12, FP32 1e-5 as for the box meshes).  One step of the batched sweep
    from zero is a multiple of M^-1 b, in the same bounds (its FP64 steps)."""
    import torch
    from sucemfem import _hip
    from sucemfem.Mesh import FunctionSpace, Mesh
    from sucemfem.SystemMatrices import AssembledSystem
    from sucemfem.Utilities.Workloads import DeviceProblem
    torch.cuda.set_device(0)
    co, ce = _wheel(m)
    p = DeviceProblem.__new__(DeviceProblem)
    p.mesh = Mesh(co, ce)
    one = np.ones(1)
    _hip.call("sucem_mesh_set_materials", p.mesh.device_handle().h, None, 1,
              _hip.ptr(np.zeros(1, np.int64)), _hip.ptr(one), _hip.ptr(one))
    p.space = FunctionSpace(p.mesh, "Nedelec 1st kind H(curl)", order)
    p.ctx = p.space.ctx
    p.system = AssembledSystem(p.space, 7)
    osp = O.Space(co, ce, order)
    p.ndofs = osp.ndofs
    mats = O.assemble_fast(osp, abc=True)
    k0, shift = 20.0, 0.25
    P = (mats["S"] - (1 - 1j * shift) * k0 ** 2 * mats["M"] + 1j * k0 * mats["S_0"]).tocsr()
    G = O.discrete_gradient(osp).tocsr().astype(np.complex128)
    Pi = O.nodal_interpolation(osp).tocsr().astype(np.complex128)

    def inv(d):
        return np.where(d != 0, 1.0 / np.where(d != 0, d, 1), 0)
    W = (3.0 if order == 2 else 2.0) * inv(O.gradient_diag(P, G))
    V = 2.0 * inv(O.gradient_diag(P, Pi))
    rng = np.random.default_rng(m)
    r = rng.standard_normal(osp.ndofs) + 1j * rng.standard_normal(osp.ndofs)
    zo = r / P.diagonal() + G @ (W * (G.T @ r)) + Pi @ (V * (Pi.T @ r))
    for precision, dt, tol in ((64, torch.complex128, 1e-12), (32, torch.complex64, 1e-5)):
        rd = torch.as_tensor(r, device="cuda").to(dt)
        zd = torch.zeros_like(rd)
        _hip.call("sucem_system_precond_apply", p.ctx.handle, p.system.handle.h, 1.0, -k0 * k0,
                  k0, shift, precision, 0, _hip.ptr(rd), _hip.ptr(zd))
        z = zd.cpu().numpy().astype(np.complex128)
        assert np.linalg.norm(z - zo) <= tol * np.linalg.norm(zo), precision
    for width in (1, 2, 4, 8):
        B = torch.as_tensor(np.tile(r, (width, 1)), device="cuda")
        X = torch.zeros_like(B)
        p.solve_sweep([k0] * width, B, X, precision=64, tol=1e-300, max_iter=1, check_every=1,
                      width=width, precond_shift=shift)
        for x in X.cpu().numpy():
            s = np.vdot(zo, x) / np.vdot(zo, zo)
            assert abs(s) > 0
            assert np.linalg.norm(x - s * zo) <= 1e-12 * np.linalg.norm(x), width
