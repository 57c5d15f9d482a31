"""The default operator of small order-2 meshes (64-cell patches) can be set, described and
found by tuning like every other form."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def _problem(n, order):
    from sucemfem.Utilities.Workloads import DeviceProblem
    return DeviceProblem(n, np.array(n) * 0.05, order, 7, (1.0, 2.2, 4.4), 3)


@pytest.mark.parametrize("n", [(2, 5, 1), (7, 6, 5), (21, 20, 21)])
@pytest.mark.parametrize("precision", [64, 32])
def test_64_cell_patches_can_be_set(n, precision):
    """Set explicitly after another form, 64-cell patches are the default's result bit for bit
    on meshes whose default they are, and the assembled operator's to rounding on any (1e-12 and
    2e-5 of max |y| as for the other patch sizes); their maps' sizes are reported."""
    import torch
    torch.cuda.set_device(0)
    p = _problem(n, 2)
    dt = torch.complex128 if precision == 64 else torch.complex64
    g = torch.Generator(device="cuda")
    g.manual_seed(2)
    x = torch.randn(p.ndofs, dtype=dt, device="cuda", generator=g)
    first, asm, y = torch.zeros_like(x), torch.zeros_like(x), torch.zeros_like(x)
    p.apply(9.0, x, first, precision=precision)
    p.set_spmv(precision, matrix_free=0, lanes=8, loads=4, blocks=64)
    p.apply(9.0, x, asm, precision=precision)
    p.set_spmv(precision, matrix_free=2, loads=64, blocks=64)
    p.apply(9.0, x, y, precision=precision)
    nc = 6 * int(np.prod(n))
    if nc <= 50000:
        assert torch.equal(y, first)
    tol = 1e-12 if precision == 64 else 2e-5
    assert (y - asm).abs().max() <= tol * asm.abs().max()
    info = p.patch_info(64)
    assert info["patches"] == -(-nc // 64)
    assert 0 < info["shared_dofs"] * 2 <= info["partial_sums"] or info["patches"] == 1
    assert p.operator_bytes(precision, 2, cb=64) > 0


def test_order_1_has_no_64_cell_patches():
    import torch
    torch.cuda.set_device(0)
    p = _problem((3, 4, 2), 1)
    with pytest.raises(ValueError, match="64"):
        p.set_spmv(64, matrix_free=2, loads=64, blocks=64)
    with pytest.raises(ValueError, match="64"):
        p.patch_info(64)


@pytest.mark.parametrize("precision", [64, 32])
def test_tuning_a_small_mesh_finds_64_cell_patches(precision):
    """17 x 22 x 13 boxes: 64-cell patches are a third faster than any other form there."""
    import torch
    torch.cuda.set_device(0)
    p = _problem((17, 22, 13), 2)
    cfg, ms = p.tune(precision, reps=10)
    assert (cfg["matrix_free"], cfg["loads"]) == (2, 64), (cfg, ms)
