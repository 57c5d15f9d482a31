"""Operator products in captured graphs: what a graph refers to stays where it is, whatever the
system is asked to do between capture and replay."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

K0 = 12.0


def _problem(n, order, stream):
    from sucemfem.Utilities.Workloads import DeviceProblem
    from sucemfem.runtime import Context
    return DeviceProblem(n, np.array(n) * 0.05, order, 7, (1.0, 2.2, 4.4), 3,
                         ctx=Context(stream=stream))


def _vectors(p, nvec, precision, seed=1):
    import torch
    dt = torch.complex128 if precision == 64 else torch.complex64
    g = torch.Generator(device="cuda")
    g.manual_seed(seed)
    return torch.randn(nvec, p.ndofs, dtype=dt, device="cuda", generator=g)


# 64-cell patches, 192 / 256-cell patches (128-cell ones need more partial sums), order 1
@pytest.mark.parametrize("n,order", [((7, 6, 5), 2), ((21, 20, 21), 2), ((9, 9, 8), 1)])
@pytest.mark.parametrize("precision", [64, 32])
@pytest.mark.parametrize("nvec", [1, 3])
def test_replay_after_other_products_and_meshes(n, order, precision, nvec):
    """A captured product, replayed after products of several vectors, after another patch size
    has been prepared and after another mesh has taken the memory that was free by then: its
    result, and the other system's, are those of eager calls bit for bit."""
    import torch
    torch.cuda.set_device(0)
    s = torch.cuda.Stream()
    with torch.cuda.stream(s):
        p = _problem(n, order, s)
        x = _vectors(p, 8, precision)
        ref, y = torch.zeros_like(x), torch.zeros_like(x)
        for v in range(nvec):
            p.apply(K0, x[v], ref[v], precision=precision)
    s.synchronize()
    g = torch.cuda.CUDAGraph()
    with torch.cuda.graph(g, stream=s):
        p.apply(K0, x, y, precision=precision, nvec=nvec)
    with torch.cuda.stream(s):
        z = torch.zeros_like(x)
        p.apply(K0, x, z, precision=precision, nvec=8)
        if order == 2:
            for cb in (128, 192, 256):
                p.patch_info(cb)
        q = _problem((6, 5, 7), 3 - order, s)
        qx = _vectors(q, 1, 64)
        qref, qy = torch.zeros_like(qx), torch.zeros_like(qx)
        q.apply(K0, qx, qref, precision=64)
        for _ in range(3):
            y.zero_()
            g.replay()
            q.apply(K0, qx, qy, precision=64)
            s.synchronize()
            assert torch.equal(y[:nvec], ref[:nvec])
            assert torch.equal(qy, qref)
        assert torch.equal(z[:nvec], ref[:nvec])


def test_products_while_another_stream_is_captured():
    """Products of several vectors on the context's stream while another stream is captured
    (in the mode that refuses allocations): the results of eager calls, and the capture ends
    well, also when these products are the first ones."""
    import torch
    torch.cuda.set_device(0)
    s, other = torch.cuda.Stream(), torch.cuda.Stream()
    with torch.cuda.stream(s):
        p = _problem((7, 6, 5), 2, s)
        x = _vectors(p, 5, 64)
        y, ref = torch.zeros_like(x), torch.zeros_like(x)
    w = torch.ones(16, device="cuda")
    torch.cuda.synchronize()
    g = torch.cuda.CUDAGraph()
    with torch.cuda.graph(g, stream=other, capture_error_mode="global"):
        w.add_(1.0)
        p.apply(K0, x, y, precision=64, nvec=5)
    with torch.cuda.stream(s):
        for v in range(5):
            p.apply(K0, x[v], ref[v], precision=64)
    g.replay()
    torch.cuda.synchronize()
    assert torch.equal(y, ref)
    assert torch.all(w == 2.0)
