"""Positions set on one stream and products on another: setPositions does not
wait for its kernels where the positions are in the solver's own buffer, so the
change of the stream does, also while the other stream is being captured."""
import ctypes

import numpy as np
import pytest

import oracle

pytestmark = pytest.mark.gpu

ETA, A, N = 0.9, 1.1, 900


def _solver(wall):
    from libmobility_amd import NBody
    s = NBody("open", "open", "single_wall" if wall else "open")
    s.setParameters(**({"wallHeight": 0.0} if wall else {}))
    s.initialize(viscosity=ETA, hydrodynamicRadius=A)
    return s


def _positions(step):
    rng = np.random.default_rng(step)
    pos = rng.uniform(0, 3.0 * A * N ** (1 / 3), (N, 3))
    pos[:, 2] += A
    return pos


@pytest.mark.parametrize("wall", [False, True])
@pytest.mark.parametrize("host", [True, False])
def test_product_on_another_stream(wall, host):
    import torch
    s = _solver(wall)
    F = torch.randn((N, 3), dtype=torch.float64, device="cuda")
    other = torch.cuda.Stream()
    torch.cuda.synchronize()
    for step in range(4):
        pos = _positions(step)
        s.setPositions(pos if host else torch.as_tensor(pos, device="cuda"))
        with torch.cuda.stream(other):
            U, _ = s.Mdot(F)
        ref, _ = oracle.mdot(pos, ETA, A, F=F.cpu().numpy(), wall=wall)
        assert np.linalg.norm(U.cpu().numpy().ravel() - ref) <= 1e-12 * np.linalg.norm(ref)


@pytest.mark.parametrize("wall", [False, True])
def test_captured_product_after_host_positions(wall):
    """The allocation-free product on a stream that is being captured, right after
    positions from the host; the graph is replayed with other forces and positions."""
    import torch
    s = _solver(wall)
    F = torch.randn((N, 3), dtype=torch.float64, device="cuda")
    U = torch.empty((N, 3), dtype=torch.float64, device="cuda")
    lib, h = s._lib, s._h

    def product():
        rc = lib.lm_nbody_mdot_noalloc(h, ctypes.c_void_p(F.data_ptr()), None,
                                       ctypes.c_void_p(U.data_ptr()), None)
        assert rc == 0, lib.lm_last_error()

    s.setPositions(_positions(0))
    product()  # warm: kernels loaded
    torch.cuda.synchronize()
    stream = torch.cuda.Stream()
    graph = torch.cuda.CUDAGraph()
    s.setPositions(_positions(1))
    with torch.cuda.graph(graph, stream=stream):
        assert lib.lm_nbody_set_stream(h, ctypes.c_void_p(stream.cuda_stream)) == 0
        product()
    for step in range(1, 4):
        pos = _positions(step)
        s.setPositions(pos)
        torch.cuda.synchronize()
        F.copy_(torch.randn((N, 3), dtype=torch.float64, device="cuda"))
        U.zero_()
        torch.cuda.synchronize()
        graph.replay()
        torch.cuda.synchronize()
        ref, _ = oracle.mdot(pos, ETA, A, F=F.cpu().numpy(), wall=wall)
        assert np.linalg.norm(U.cpu().numpy().ravel() - ref) <= 1e-12 * np.linalg.norm(ref)


@pytest.mark.parametrize("n", [1, 255, 257, 4097, 16384, 16385])
def test_positions_overwritten_on_another_stream(n):
    """Above a wall setPositions has read the caller's tensor when it returns."""
    import torch
    s = _solver(True)
    rng = np.random.default_rng(n)
    pos = rng.uniform(0, 3.0 * A * n ** (1 / 3), (n, 3))
    pos[:, 2] += A
    F = rng.standard_normal((n, 3))
    ref, _ = oracle.mdot(pos, ETA, A, F=F, wall=True)
    other = torch.cuda.Stream()
    for _ in range(3):
        tensor = torch.as_tensor(pos, device="cuda")
        torch.cuda.synchronize()
        s.setPositions(tensor)
        with torch.cuda.stream(other):
            tensor.fill_(float("nan"))
        U, _ = s.Mdot(torch.as_tensor(F, device="cuda"))
        torch.cuda.synchronize()
        assert np.linalg.norm(U.cpu().numpy().ravel() - ref) <= 1e-12 * np.linalg.norm(ref)


def _occupy_default_stream():
    """Some tens of milliseconds of work queued on the default stream."""
    import torch
    x = torch.full((8192, 8192), 1e-4, dtype=torch.float64, device="cuda")
    torch.cuda.synchronize()
    for _ in range(3):
        x = x @ x
    return x


@pytest.mark.parametrize("wall", [False, True])
@pytest.mark.parametrize("host", [True, False])
@pytest.mark.parametrize("valid", [True, False])
def test_product_on_another_stream_behind_other_work(wall, host, valid):
    """The records of a busy default stream: a product on another stream has those
    of the last positions, also where setPositions refused the batch parameters
    (which leaves one system of all particles)."""
    import torch
    from libmobility_amd import NBody
    s = NBody("open", "open", "single_wall" if wall else "open")
    s.setParameters(**({"wallHeight": 0.0} if wall else {}))
    s.initialize(viscosity=ETA, hydrodynamicRadius=A)
    F = torch.randn((N, 3), dtype=torch.float64, device="cuda")
    s.setPositions(_positions(0))
    if not valid:
        s.setParameters(Nbatch=2, NperBatch=N, **({"wallHeight": 0.0} if wall else {}))
    # several streams: some may share the default stream's hardware queue
    for step, other in enumerate([torch.cuda.Stream() for _ in range(4)], 1):
        s.Mdot(F)  # back on the default stream, where host arrays then stay
        pos = _positions(step)
        given = pos if host else torch.as_tensor(pos, device="cuda")
        _occupy_default_stream()
        if valid:
            s.setPositions(given)
        else:
            with pytest.raises(RuntimeError, match="Invalid batch parameters"):
                s.setPositions(given)
        with torch.cuda.stream(other):
            U, _ = s.Mdot(F)
        ref, _ = oracle.mdot(pos, ETA, A, F=F.cpu().numpy(), wall=wall)
        assert np.linalg.norm(U.cpu().numpy().ravel() - ref) <= 1e-12 * np.linalg.norm(ref)
