"""Host and device arrays through setPositions and Mdot: the paths of small
calls (mapped host buffers up to 16384 particles, one launch placing systems
of up to 1024) give what the others give, call after call."""
import numpy as np
import pytest

import oracle

pytestmark = pytest.mark.gpu

ETA, A = 0.9, 1.1


def _solver(wall, angular, **params):
    from libmobility_amd import NBody
    s = NBody("open", "open", "single_wall" if wall else "open")
    if wall:
        params["wallHeight"] = 0.0
    s.setParameters(**params)
    s.initialize(viscosity=ETA, hydrodynamicRadius=A, includeAngular=angular)
    return s


def _inputs(N, wall, seed):
    rng = np.random.default_rng(seed)
    pos = rng.uniform(0, 3.0 * A * max(1.0, N ** (1 / 3)), (N, 3))
    if wall:
        pos[:, 2] = rng.uniform(0.3 * A, 9 * A, N)
    return pos, rng.normal(size=(N, 3)), rng.normal(size=(N, 3))


@pytest.mark.parametrize("N,nbatch", [(1, 1), (255, 1), (256, 1), (257, 1), (1024, 1), (1025, 1),
                                      (16384, 1), (16385, 1), (2048, 2), (2050, 2), (3000, 300)])
@pytest.mark.parametrize("wall,angular", [(False, False), (False, True), (True, True)])
def test_host_and_device_arrays_agree(N, nbatch, wall, angular):
    import torch
    kw = dict(Nbatch=nbatch, NperBatch=N // nbatch) if nbatch > 1 else {}
    host, dev = _solver(wall, angular, **kw), _solver(wall, angular, **kw)
    for step in range(3):  # the same buffers again, with other values
        pos, F, T = _inputs(N, wall, 10 * N + step)
        t = T if angular else None
        host.setPositions(pos)
        given = [F.copy(), None if t is None else t.copy()]
        pos[:] = -1.0  # the caller's array may change once the call has returned
        U, W = host.Mdot(*given)
        pos, _, _ = _inputs(N, wall, 10 * N + step)
        dev.setPositions(torch.as_tensor(pos, device="cuda"))
        Ud, Wd = dev.Mdot(torch.as_tensor(F, device="cuda"),
                          None if t is None else torch.as_tensor(t, device="cuda"))
        assert np.array_equal(U, Ud.cpu().numpy())
        assert W is None or np.array_equal(W, Wd.cpu().numpy())
    if N <= 4096:
        sizes = [N // nbatch] * nbatch
        Uo, Wo = oracle.mdot(pos, ETA, A, F=F, T=t, angular=angular, wall=wall, sys_sizes=sizes)
        # a few hundred FP64 roundings in sums that hardly cancel
        assert np.linalg.norm(U.ravel() - Uo) <= 1e-12 * np.linalg.norm(Uo)
        if angular:
            assert np.linalg.norm(W.ravel() - Wo) <= 1e-12 * max(np.linalg.norm(Wo), 1e-300)


@pytest.mark.parametrize("angular", [False, True])
def test_systems_of_another_size_between_calls(angular):
    """The offsets on the device follow the systems, also back to earlier ones."""
    s = _solver(False, angular)
    for sizes in ([700], [300, 400], [699, 1], [300, 400], [1500, 20]):
        N = sum(sizes)
        pos, F, T = _inputs(N, False, N + len(sizes))
        s.setSystems(sizes)
        s.setPositions(pos)
        U, W = s.Mdot(F, T if angular else None)
        Uo, Wo = oracle.mdot(pos, ETA, A, F=F, T=T if angular else None, angular=angular,
                             wall=False, sys_sizes=sizes)
        assert np.linalg.norm(U.ravel() - Uo) <= 1e-12 * np.linalg.norm(Uo)
        if angular:
            assert np.linalg.norm(W.ravel() - Wo) <= 1e-12 * np.linalg.norm(Wo)
