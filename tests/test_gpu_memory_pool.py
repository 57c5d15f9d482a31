"""Buffers of finished objects are used again by the context's next ones: bounded, given back
with the workspace, and never before the work that uses them is done."""
import ctypes
import threading

import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def _free(ctx):
    from sucemfem import _hip
    f, t = ctypes.c_int64(), ctypes.c_int64()
    _hip.call("sucem_ctx_mem_info", ctx.handle, ctypes.byref(f), ctypes.byref(t))
    return f.value


def _solve(ctx, n, order, seed):
    import torch
    from sucemfem.Utilities.Workloads import DeviceProblem
    p = DeviceProblem(n, np.array(n) * 0.03, order, 7, (1.0, 2.2, 4.4), seed, ctx=ctx)
    c = np.array(n) * 0.015 + 1e-3
    b = p.rhs_dipoles(c[None], np.array([[0.3, 1.0, -0.2]]), 9.0)
    x = torch.zeros_like(b)
    st = p.solve(9.0, b, x, precision=64, tol=1e-10)
    ctx.synchronize()
    assert st["status"] == 0
    return x.cpu().numpy()


def _raw():
    """Free device memory as the device reports it: idle blocks of a pool are not in it."""
    import gc
    import torch
    gc.collect()
    torch.cuda.synchronize()
    torch.cuda.empty_cache()
    return torch.cuda.mem_get_info()[0]


SLACK = 64 << 20     # granularity of the device's allocations


def test_repeated_meshes_do_not_grow_and_release_gives_back():
    import torch
    from sucemfem import _hip
    from sucemfem.runtime import Context
    torch.cuda.set_device(0)
    ctx = Context()
    ref = _solve(ctx, (9, 8, 7), 2, 0)
    sizes = ((9, 8, 7), 2, 0), ((8, 8, 8), 2, 1), ((12, 9, 10), 1, 2)
    start = None
    for k in range(5):
        for n, order, seed in sizes:
            x = _solve(ctx, n, order, seed)
            if (n, order, seed) == ((9, 8, 7), 2, 0):
                assert np.array_equal(x, ref)       # reused memory changes nothing
        if k == 0:
            start = _raw()
    # once every size has been seen, repetitions take nothing more
    assert start - _raw() <= SLACK
    ws = ctypes.c_int64()
    _hip.call("sucem_ctx_workspace_bytes", ctx.handle, ctypes.byref(ws))
    held = _raw()
    _hip.call("sucem_ctx_release_workspace", ctx.handle)
    assert _raw() - held >= ws.value
    _hip.call("sucem_ctx_workspace_bytes", ctx.handle, ctypes.byref(ws))
    assert ws.value == 0


def test_idle_blocks_are_bounded_and_go_back():
    """What a 20^3 order-2 problem leaves in the pool (several hundred MB, at most 4 GB), in
    free memory as the device reports it: no more after repetitions, nothing after the release
    and nothing after the context."""
    import torch
    from sucemfem import _hip
    from sucemfem.Utilities.Workloads import DeviceProblem
    from sucemfem.runtime import Context
    torch.cuda.set_device(0)

    def build(ctx):
        p = DeviceProblem((20, 20, 20), 0.6, 2, 7, (1.0, 2.2, 4.4), 0, ctx=ctx)
        ctx.synchronize()
        del p

    ctx = Context()
    build(ctx)                                    # code and tables of the library
    _hip.call("sucem_ctx_release_workspace", ctx.handle)
    before = _raw()
    build(ctx)
    ws = ctypes.c_int64()
    _hip.call("sucem_ctx_workspace_bytes", ctx.handle, ctypes.byref(ws))
    idle = before - _raw() - ws.value
    assert (128 << 20) < idle <= (4 << 30) + SLACK
    for _ in range(3):
        build(ctx)
    assert before - _raw() - ws.value <= idle + SLACK
    _hip.call("sucem_ctx_release_workspace", ctx.handle)
    assert abs(before - _raw()) <= SLACK
    build(ctx)
    assert before - _raw() > (128 << 20)
    del ctx
    assert before - _raw() <= SLACK


def test_threads_with_contexts_of_their_own():
    """Four threads build, solve and drop problems at once, each on its own stream and context,
    and drop each other's objects: results equal the ones computed alone."""
    import torch
    from sucemfem.runtime import Context
    torch.cuda.set_device(0)
    sizes = [((6, 5, 4), 2), ((9, 8, 7), 1), ((5, 6, 7), 2), ((7, 7, 7), 1)]
    alone = [_solve(Context(), n, o, 5) for n, o in sizes]
    got, errs = [[] for _ in sizes], []

    def work(i):
        try:
            torch.cuda.set_device(0)
            s = torch.cuda.Stream()
            with torch.cuda.stream(s):
                ctx = Context(stream=s)
                for _ in range(4):
                    got[i].append(_solve(ctx, sizes[i][0], sizes[i][1], 5))
        except Exception as e:  # noqa: BLE001 - reported below
            errs.append(e)

    ths = [threading.Thread(target=work, args=(i,)) for i in range(len(sizes))]
    for t in ths:
        t.start()
    for t in ths:
        t.join()
    assert not errs, errs
    for a, g in zip(alone, got):
        for x in g:
            assert np.array_equal(x, a)


def test_unused_blocks_count_as_free_memory():
    """Dropped buffers that the pool keeps stay available to admission by free memory: what a
    20^3 order-2 set-up (several hundred MB) leaves behind changes the reported free bytes by
    less than 64 MB (allocation granularity), and releasing the pool adds no more than that."""
    import gc
    import torch
    from sucemfem import _hip
    from sucemfem.Utilities.Workloads import DeviceProblem
    from sucemfem.runtime import Context
    torch.cuda.set_device(0)
    ctx = Context()
    ctx.synchronize()
    before = _free(ctx)
    p = DeviceProblem((20, 20, 20), 0.6, 2, 7, (1.0, 2.2, 4.4), 0, ctx=ctx)
    ctx.synchronize()
    assert before - _free(ctx) > (128 << 20)
    del p
    gc.collect()
    ws = ctypes.c_int64()
    _hip.call("sucem_ctx_workspace_bytes", ctx.handle, ctypes.byref(ws))
    after = _free(ctx) + ws.value        # the workspace is reported on its own
    _hip.call("sucem_ctx_release_workspace", ctx.handle)
    print("free bytes:", before, after, _free(ctx), ws.value, flush=True)
    assert abs(_free(ctx) - after) < (64 << 20)
    assert abs(before - after) < (64 << 20)


def test_free_memory_is_what_any_allocation_can_have():
    """The free memory reported to admission holds for torch too: the pools of every context
    have given their idle blocks back by then."""
    import torch
    from sucemfem.Serving import device_free_bytes
    from sucemfem.Utilities.Workloads import DeviceProblem
    from sucemfem.runtime import Context
    torch.cuda.set_device(0)
    ctx = Context()
    DeviceProblem((20, 20, 20), 0.6, 2, 7, (1.0, 2.2, 4.4), 0, ctx=ctx)
    low = _raw()
    told = device_free_bytes()
    assert told - low > (128 << 20)
    assert abs(_raw() - told) <= SLACK


def test_request_survives_torch_running_out_of_memory(monkeypatch):
    """A request whose vectors torch cannot allocate runs again once the pools' idle blocks are
    free."""
    import torch
    from sucemfem.Serving import Request, Server, device_executor
    from sucemfem.Utilities import Workloads
    from sucemfem.runtime import Context
    torch.cuda.set_device(0)
    other = Context()
    seen = []
    rhs = Workloads.DeviceProblem.rhs_dipoles

    def short_of_memory(self, *a, **kw):
        if not seen:       # what another slot's request leaves behind
            Workloads.DeviceProblem((20, 20, 20), 0.6, 2, 7, (1.0, 2.2, 4.4), 0, ctx=other)
        seen.append(torch.cuda.mem_get_info()[0])
        if len(seen) == 1:
            raise torch.cuda.OutOfMemoryError("no memory for b")
        return rhs(self, *a, **kw)

    monkeypatch.setattr(Workloads.DeviceProblem, "rhs_dipoles", short_of_memory)
    req = Request(0, "driven", (0.3, 0.2, 0.25), 4, 1, 0.0, freq=4e8)
    (r,), _ = Server(device_executor(), slots=1).run([req], realtime=False)
    assert r.status == "done", r.error
    assert len(seen) == 2 and seen[1] - seen[0] > (128 << 20)


@pytest.mark.parametrize("mode", ["relaxed", "global"])
def test_objects_dropped_by_another_thread_during_a_capture(mode):
    """A thread that drops a mesh, its space and its system leaves a capture of another thread
    alone (the batched sweep captures its iterations), and the next launch reports nothing.
    Free memory can be asked for as well."""
    import torch
    from sucemfem.Utilities.Workloads import DeviceProblem
    from sucemfem.runtime import Context
    torch.cuda.set_device(0)
    s = torch.cuda.Stream()
    with torch.cuda.stream(s):
        ctx = Context(stream=s)
        ps = [DeviceProblem((3, 4, 2), 0.1, 2, 7, (1.0, 2.2, 4.4), 0, ctx=ctx),
              DeviceProblem((2, 2, 2), 0.1, 1, 7, (1.0, 2.2, 4.4), 0, ctx=ctx)]
        x = torch.ones(ps[1].ndofs, dtype=torch.complex128, device="cuda")
        y, ref = torch.zeros_like(x), torch.zeros_like(x)
        ps[1].apply(3.0, x, ref, precision=64)
    errs = []

    def drop():
        try:
            torch.cuda.set_device(0)
            del ps[0]
            ps[0].apply(3.0, x, y, precision=64)
            assert _free(ctx) > 0
            if mode == "relaxed":
                with torch.cuda.stream(s):
                    DeviceProblem((2, 3, 2), 0.1, 2, 7, (1.0, 2.2, 4.4), 0, ctx=ctx)
            del ps[0]
        except Exception as e:  # noqa: BLE001 - reported below
            errs.append(e)

    w = torch.ones(16, device="cuda")
    torch.cuda.synchronize()
    g = torch.cuda.CUDAGraph()
    with torch.cuda.graph(g, stream=torch.cuda.Stream(), capture_error_mode=mode):
        t = threading.Thread(target=drop)
        t.start()
        t.join()
        w.add_(1.0)
    g.replay()
    torch.cuda.synchronize()
    assert not errs, errs
    assert torch.all(w == 2.0)
    assert torch.equal(y, ref)


def test_sweeps_beside_a_thread_that_drops_problems():
    """Batched sweeps (whose iterations are captured) on one thread while another one builds
    and drops problems: the sweeps' solutions are those of a sweep alone."""
    import torch
    from sucemfem.Utilities.Workloads import DeviceProblem
    from sucemfem.runtime import Context
    torch.cuda.set_device(0)
    k0s = np.linspace(0.5, 12.0, 4)

    def problem(ctx, n, order):
        return DeviceProblem(n, np.array(n) * 0.03, order, 7, (1.0, 2.2, 4.4), 3, ctx=ctx)

    s1 = torch.cuda.Stream()
    with torch.cuda.stream(s1):
        p = problem(Context(stream=s1), (6, 5, 4), 1)
        g = torch.Generator(device="cuda")
        g.manual_seed(0)
        B = torch.randn(4, p.ndofs, dtype=torch.complex128, device="cuda", generator=g)
        ref, X = torch.zeros_like(B), torch.zeros_like(B)
        p.solve_sweep(k0s, B, ref, precision=64, tol=1e-10, width=2, use_graph=True)
    s1.synchronize()
    stop, errs = threading.Event(), []

    def churn():
        try:
            torch.cuda.set_device(0)
            s2 = torch.cuda.Stream()
            with torch.cuda.stream(s2):
                ctx = Context(stream=s2)
                while not stop.is_set():
                    q = problem(ctx, (3, 4, 2), 2)
                    del q
        except Exception as e:  # noqa: BLE001 - reported below
            errs.append(e)

    t = threading.Thread(target=churn)
    t.start()
    try:
        with torch.cuda.stream(s1):
            for _ in range(20):
                X.zero_()
                st = p.solve_sweep(k0s, B, X, precision=64, tol=1e-10, width=2, use_graph=True)
                s1.synchronize()
                assert all(q["status"] == 0 for q in st)
                assert torch.equal(X, ref)
    finally:
        stop.set()
        t.join()
    assert not errs, errs


@pytest.mark.parametrize("mb,extra", [(9, 4), (1000, 12345)])
def test_what_a_buffer_takes_from_the_device(mb, extra):
    """An allocation takes at most an eighth more than its size from the device (whose own
    granularity, 2 MB, comes on top)."""
    import torch
    from sucemfem import _hip
    from sucemfem.runtime import Context
    torch.cuda.set_device(0)
    ctx = Context()
    # a matrix of nnz values keeps nnz (4 + 16 + 8) bytes and 8 (n + 1) of row pointers and
    # diagonals: one row holds them all
    nnz = ((mb << 20) + extra) // 16
    ptr = np.array([0, nnz], np.int64)
    col = np.zeros(nnz, np.int32)
    val = np.ones(nnz, np.complex128)
    h = _hip.out_handle()
    before = _raw()
    _hip.call("sucem_csr_create", ctx.handle, 1, nnz, _hip.ptr(ptr), _hip.ptr(col), _hip.ptr(val),
              ctypes.byref(h))
    took = before - _raw()
    _hip.call("sucem_csr_destroy", h)
    assert 28 * nnz - (2 << 20) <= took <= 28 * nnz * 9 // 8 + (8 << 20), (took, 28 * nnz)
