"""Point location, basis values at points and point-source right-hand sides at the sizes where
their kernels' tiles end: 64 points per box test, 64 sources per tile."""
import numpy as np
import pytest
import oracle as O

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module", params=[1, 2])
def prob(request):
    import torch
    from sucemfem import _hip
    from sucemfem.Utilities.Workloads import DeviceProblem
    torch.cuda.set_device(0)
    order = request.param
    p = DeviceProblem((4, 3, 5), (0.8, 0.7, 0.9), order, _hip.MAT_S | _hip.MAT_T)
    co, ce = O.box_mesh((0.8, 0.7, 0.9), (4, 3, 5))
    return p, O.Space(co, ce, order)


@pytest.mark.parametrize("n", [1, 63, 64, 65, 200])
def test_basis_at_points_matches_oracle(prob, n):
    """Cells and DOFs equal, values to 1e-13: both evaluate the same order-2 polynomials in
    FP64 on unit-sized cells.  Vertices of the mesh (points of many cells: the lowest-index
    one counts) are among the points."""
    from sucemfem.Sources.point_source import basis_at_points
    p, sp = prob
    rng = np.random.default_rng(n)
    pts = rng.uniform(0.0, 1.0, (n, 3)) * (0.8, 0.7, 0.9)
    pts[::7] = sp.coords[rng.integers(0, len(sp.coords), len(pts[::7]))]
    vals, dofs = basis_at_points(p.space, pts)
    for k in range(n):
        c = O.locate_cell(sp.coords, sp.cells, pts[k])
        assert np.array_equal(dofs[k], sp.cell_dofs[c]), (k, pts[k])
        v, _ = O.eval_basis(sp.order, sp.coords[sp.cells[c]], pts[k][None])
        assert np.abs(vals[k] - v[0]).max() <= 1e-13 * max(1.0, np.abs(v).max())


def test_point_outside_is_refused(prob):
    from sucemfem.Sources.point_source import basis_at_points
    p, _ = prob
    pts = np.full((70, 3), 0.3)
    pts[66] = (0.3, 0.3, 0.9001)
    with pytest.raises(AssertionError):
        basis_at_points(p.space, pts)


@pytest.mark.parametrize("nsrc,nrhs", [(1, 1), (63, 1), (64, 2), (65, 1), (129, 3), (300, 40)])
def test_sources_summed_in_input_order(prob, nsrc, nrhs):
    """Every DOF's sources are added one after another in input order, onto what b held: the
    same sums in numpy, where only the basis values' rounding differs (1e-13 of max |b|).
    Sources crowd into a few cells, so that DOFs recur within and across tiles."""
    import torch
    from sucemfem import _hip
    p, sp = prob
    rng = np.random.default_rng(nsrc)
    pos = np.ascontiguousarray(0.31 + 0.2 * rng.uniform(0.0, 1.0, (nsrc, 3)))
    val = np.ascontiguousarray(rng.standard_normal((nsrc, 3)) + 1j * rng.standard_normal((nsrc, 3)))
    idx = np.ascontiguousarray(rng.integers(0, nrhs, nsrc), np.int64)
    b0 = rng.standard_normal((nrhs, p.ndofs)) + 1j * rng.standard_normal((nrhs, p.ndofs))
    b = torch.as_tensor(b0, device="cuda")
    for entry in ("sucem_rhs_point_sources", "sucem_rhs_point_sources_noalloc"):
        got = b.clone()
        _hip.call(entry, p.ctx.handle, p.space.handle.h, nsrc, _hip.ptr(pos), _hip.ptr(val),
                  _hip.ptr(idx), nrhs, 0.0, -3.0, _hip.ptr(got))
        want = b0.copy()
        for s in range(nsrc):
            dn, v = O.point_source_contrib(sp, pos[s], val[s])
            want[idx[s], dn] += -3j * v
        assert np.abs(got.cpu().numpy() - want).max() <= 1e-13 * np.abs(want).max()
