"""Far-field sums over few and many directions: the two kernels share their summation order, so
a direction's result does not depend on how many are asked for."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n,order", [((1, 1, 1), 1), ((1, 1, 1), 2), ((3, 4, 2), 2),
                                     ((9, 7, 8), 1)])
def test_directions_do_not_depend_on_their_number(n, order):
    """1, 16 (the few-directions kernel), 17, 64, 65 and 130 directions: equal bit for bit to
    the same directions one at a time, for the surface and the variational form."""
    import torch
    from sucemfem.PostProcessing import surface_ntff, variational_ntff
    from sucemfem.Utilities.Workloads import DeviceProblem
    torch.cuda.set_device(0)
    p = DeviceProblem(n, np.array(n) * 0.1, order, 7)
    rng = np.random.default_rng(2)
    x = rng.standard_normal(p.ndofs) + 1j * rng.standard_normal(p.ndofs)
    th, ph = rng.uniform(0, 180, 130), rng.uniform(0, 360, 130)
    for cls in (surface_ntff.NTFF, variational_ntff.NTFF):
        t = cls(p.space)
        t.set_dofs(x)
        t.set_frequency(5e8)
        one = np.array([t.calc_pt(a, b) for a, b in zip(th, ph)])
        assert np.all(np.isfinite(one)) and np.abs(one).min() > 0
        for m in (1, 16, 17, 64, 65, 130):
            assert np.array_equal(t.calc_pts(th[:m], ph[:m]), one[:m]), (cls, m)
