"""The autotuner: the first product of a combination times the candidates, also where
the default is the kernel of small systems, and later ones take the fastest."""
import time

import numpy as np
import pytest

import oracle

pytestmark = pytest.mark.gpu

ETA, A = 0.9, 1.1


def _solver(wall, angular, precision, tune):
    from libmobility_amd import NBody
    s = NBody("open", "open", "single_wall" if wall else "open")
    s.setParameters(**({"wallHeight": 0.0} if wall else {}))
    s.setPairPrecision(precision)
    assert s._lib.lm_nbody_set_autotune(s._h, int(tune)) == 0
    s.initialize(viscosity=ETA, hydrodynamicRadius=A, includeAngular=angular, tolerance=1e-4, seed=7)
    return s


def _inputs(N):
    rng = np.random.default_rng(N)
    pos = rng.uniform(0, 3.0 * A * N ** (1 / 3), (N, 3))
    pos[:, 2] += A
    return pos, rng.normal(size=(N, 3)), rng.normal(size=(N, 3))


def _first(call, solvers):
    """The shortest first call of several new solvers, in seconds."""
    import torch
    times = []
    for s in solvers:
        torch.cuda.synchronize()
        t = time.perf_counter()
        call(s)
        torch.cuda.synchronize()
        times.append(time.perf_counter() - t)
    return min(times)


@pytest.mark.parametrize("precision", ["fp64", "fp32"])
@pytest.mark.parametrize("wall,angular", [(False, False), (True, True)])
def test_first_product_times_the_candidates(wall, angular, precision):
    import torch
    N = 3000
    pos, F, T = _inputs(N)
    dev = [torch.as_tensor(x, device="cuda") for x in (pos, F, T)]

    def make(tune):
        s = _solver(wall, angular, precision, tune)
        s.setPositions(dev[0])
        return s

    def call(s):
        return s.Mdot(dev[1], dev[2] if angular else None)

    for tune in (True, False):  # kernels loaded
        call(make(tune))
    tuned = [make(True) for _ in range(3)]
    # ten candidates and more, three launches each, against one launch
    assert _first(call, tuned) > 4 * _first(call, [make(False) for _ in range(5)])
    U, W = call(tuned[0])
    Uo, Wo = oracle.mdot(pos, ETA, A, F=F, T=T if angular else None, angular=angular, wall=wall)
    tol = 1e-12 if precision == "fp64" else 1e-5
    assert np.linalg.norm(U.cpu().numpy().ravel() - Uo) <= tol * np.linalg.norm(Uo)
    if angular:
        assert np.linalg.norm(W.cpu().numpy().ravel() - Wo) <= tol * np.linalg.norm(Wo)


@pytest.mark.parametrize("wall,angular", [(False, False), (True, False), (True, True)])
@pytest.mark.parametrize("sizes", [None, (300, 0, 17, 1, 1000)])
@pytest.mark.parametrize("per_system", [False, True])
def test_square_root_with_the_autotuner(wall, angular, sizes, per_system):
    """Recurrences over tuned products, before and after a product has been tuned on
    its own, applied twice, against M."""
    N = 1318
    pos, F, T = _inputs(N)
    rng = np.random.default_rng(3)
    s = _solver(wall, angular, "fp64", True)
    if sizes:
        s.setSystems(sizes)
    s.setLanczosPerSystem(per_system)
    s.setPositions(pos)
    z = rng.normal(size=(6 if angular else 3) * N)

    def root(x):
        return np.concatenate([v.ravel() for v in s.sqrtMdotW_with_noise(x) if v is not None])

    for _ in range(2):
        y = root(root(z))
        ref = np.concatenate([v for v in oracle.mdot(
            pos, ETA, A, F=z[:3 * N], T=z[3 * N:] if angular else None, angular=angular, wall=wall,
            sys_sizes=sizes) if v is not None])
        # two square roots that stop near a relative 1e-4 (their estimate is no bound)
        assert np.linalg.norm(y - ref) <= 2e-3 * np.linalg.norm(ref)
        s.Mdot(F, T if angular else None)


@pytest.mark.parametrize("root_first", [True, False])
def test_symmetric_choices_of_roots_and_products_are_apart(root_first):
    """Plain Lanczos products over open systems run other symmetric kernels than Mdot
    at the same size: each is timed at its own first use."""
    import torch
    N = 17000
    pos, F, _ = _inputs(N)
    dpos, dF = (torch.as_tensor(x, device="cuda") for x in (pos, F))
    z = torch.as_tensor(np.random.default_rng(1).normal(size=3 * N), device="cuda")

    def make():
        s = _solver(False, False, "fp64", True)
        s.setPositions(dpos)
        return s

    def product(s):
        return s.Mdot(dF)

    def root(s):
        return s.sqrtMdotW_with_noise(z)

    first, then = (root, product) if root_first else (product, root)
    s = make()  # kernels loaded, both tuned
    for call in (product, root, product, root):
        call(s)
    again = min(_first(then, [s]) for _ in range(5))
    new = [make() for _ in range(3)]
    for t in new:
        first(t)
    # ten candidates and more, three products each: thirty products besides
    one = min(_first(product, [s]) for _ in range(5))
    assert _first(then, new) > again + 10 * one
    U, _ = product(new[0])
    Uo, _ = product(s)
    assert float((U - Uo).norm()) <= 1e-12 * float(Uo.norm())
