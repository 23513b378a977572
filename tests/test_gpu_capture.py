"""Calls on a stream that is being captured, where nothing that is launched runs:
what they prepare for later calls is not taken as prepared."""
import contextlib
import ctypes

import numpy as np
import pytest

import oracle

pytestmark = pytest.mark.gpu

ETA, A = 0.9, 1.1


def _hip():
    import torch
    torch.zeros(1, device="cuda")
    with open("/proc/self/maps") as f:
        return ctypes.CDLL(next(line.split()[-1] for line in f if "libamdhip64" in line))


@contextlib.contextmanager
def _captured(s, stream):
    """The body on `stream`, captured (relaxed) into a graph that is thrown away."""
    hip, raw = _hip(), ctypes.c_void_p(stream.cuda_stream)
    assert s._lib.lm_nbody_set_stream(s._h, raw) == 0
    assert hip.hipStreamBeginCapture(raw, 2) == 0
    yield
    graph = ctypes.c_void_p()
    assert hip.hipStreamEndCapture(raw, ctypes.byref(graph)) == 0
    assert hip.hipGraphDestroy(graph) == 0
    assert s._lib.lm_nbody_set_stream(s._h, None) == 0


def _solver(wall, **kw):
    from libmobility_amd import NBody
    s = NBody("open", "open", "single_wall" if wall else "open")
    s.setParameters(**({"wallHeight": 0.0} if wall else {}))
    s.initialize(viscosity=ETA, hydrodynamicRadius=A, **kw)
    return s


def _inputs(N, seed):
    import torch
    rng = np.random.default_rng(seed)
    pos = rng.uniform(0, 4.0 * A * N ** (1 / 3), (N, 3))
    pos[:, 2] += A
    F = rng.normal(size=(N, 3))
    dev = torch.as_tensor(pos, device="cuda"), torch.as_tensor(F, device="cuda")
    torch.cuda.synchronize()
    return pos, F, dev


def _right(s, pos, F, dF, wall):
    U, _ = s.Mdot(dF)
    ref, _ = oracle.mdot(pos, ETA, A, F=F, wall=wall)
    return np.linalg.norm(U.cpu().numpy().ravel() - ref) <= 1e-12 * np.linalg.norm(ref)


def test_work_list_of_a_captured_product():
    """The symmetric work list is written by a kernel: a captured product may not be
    the one that makes it."""
    import torch
    N = 4500
    s = _solver(True)
    pos, F, (dp, dF) = _inputs(N, 1)
    U = torch.empty_like(dF)
    stream = torch.cuda.Stream()

    def captured_mdot():
        with _captured(s, stream):
            rc = s._lib.lm_nbody_mdot(s._h, ctypes.c_void_p(dF.data_ptr()), 3 * N, None, 0,
                                      ctypes.c_void_p(U.data_ptr()), None, 1)
            assert rc != 0 and b"cannot be captured" in s._lib.lm_last_error()

    s.setPositions(dp)
    captured_mdot()
    assert _right(s, pos, F, dF, True)
    assert s.lastPairSymmetric()
    s.setPairTiling(2, 0)
    captured_mdot()
    assert _right(s, pos, F, dF, True)
    s.setPairTiling(0, 0)
    captured_mdot()
    assert _right(s, pos, F, dF, True)


def test_offsets_of_captured_positions():
    """An upload that was only recorded does not count as made."""
    import torch
    s = _solver(False)
    stream = torch.cuda.Stream()
    pos, F, (dp, dF) = _inputs(200, 2)
    small = dp[:100].contiguous()
    s.setPositions(dp)
    assert _right(s, pos, F, dF, False)
    s.setPositions(small)
    assert _right(s, pos[:100], F[:100], dF[:100].contiguous(), False)
    torch.cuda.synchronize()
    with _captured(s, stream):
        assert s._lib.lm_nbody_set_positions(s._h, ctypes.c_void_p(dp.data_ptr()), 600, 1) == 0
    pos, F, (dp, dF) = _inputs(200, 3)
    s.setPositions(dp)
    assert _right(s, pos, F, dF, False)


@pytest.mark.parametrize("wall", [False, True])
def test_square_root_is_not_captured(wall):
    """It waits for its convergence; what its first call clears and fills is not
    left to a graph: the next one has the bits of a solver that was never captured."""
    import torch
    N = 300
    s = _solver(wall, tolerance=1e-6)
    _, _, (dp, _) = _inputs(N, 4)
    dW = torch.as_tensor(np.random.default_rng(5).normal(size=3 * N), device="cuda")
    U = torch.empty_like(dW)
    stream = torch.cuda.Stream()
    s.setPositions(dp)
    torch.cuda.synchronize()
    with _captured(s, stream):
        rc = s._lib.lm_nbody_sqrt_mdot_w_noise(s._h, ctypes.c_void_p(dW.data_ptr()),
                                               ctypes.c_void_p(U.data_ptr()), None, 1.0, 1)
        assert rc != 0
    other = _solver(wall, tolerance=1e-6)
    other.setPositions(dp)
    u, v = s.sqrtMdotW_with_noise(dW)[0], other.sqrtMdotW_with_noise(dW)[0]
    assert s.lastLanczosIterations() == other.lastLanczosIterations()
    assert np.array_equal(u.cpu().numpy(), v.cpu().numpy())
