"""The Lanczos recurrence at the vector lengths where its step changes its
launches (lanczos_kernels.hip: one workgroup up to 4096 entries, two launches
up to 16384, three beyond), against the oracle's restatement of the algorithm."""
import numpy as np
import pytest

import oracle
from tests.test_gpu_mdot import _solver

pytestmark = pytest.mark.gpu

TOL = 1e-6


@pytest.mark.parametrize("angular,N", [
    (False, 1), (False, 342), (False, 1365), (False, 1366), (False, 5461), (False, 5462),
    (True, 682), (True, 683), (True, 2730), (True, 2731)])
def test_step_lengths_vs_oracle(angular, N):
    rng = np.random.default_rng(N)
    eta, a = 1 / (6 * np.pi), 1.0
    # dilute, above a wall: the solve converges before orthogonality is lost,
    # so both sides follow the same iterates
    side = 6.0 * max(1.0, (N / 2) ** 0.5)
    pos = rng.uniform(0, side, (N, 3))
    pos[:, 2] = rng.uniform(1.5, 12.0, N)
    s = _solver(True, a, eta)
    s.initialize(viscosity=eta, hydrodynamicRadius=a, includeAngular=angular, tolerance=TOL)
    s.setPositions(pos)

    def product(v):
        F, T = (v[:3 * N], v[3 * N:]) if angular else (v, None)
        U, W = oracle.mdot(pos, eta, a, F=F, T=T, angular=angular, wall=True)
        return np.concatenate([U, W]) if angular else U

    lz = oracle.LanczosOracle()
    for _ in range(2):  # the second call keeps the first one's schedule and estimate
        W = rng.normal(size=(6 if angular else 3) * N)
        u, w = s.sqrtMdotW_with_noise(W)
        got = np.concatenate([u.ravel(), w.ravel()]) if angular else u.ravel()
        ref, it = lz.run(product, W, TOL)
        # an estimate at the tolerance may fall on either side of it: one
        # iteration apart, and then the two differ by about the tolerance
        assert abs(s.lastLanczosIterations() - it) <= 1
        assert np.linalg.norm(got - ref) <= 2 * TOL * np.linalg.norm(ref)


@pytest.mark.parametrize("sizes", [(2,) * 2730, (40,) * 30, (300, 0, 17, 1, 1000)])
@pytest.mark.parametrize("precision", ["fp64", "fp32"])
def test_one_recurrence_over_systems_vs_oracle(sizes, precision):
    """A recurrence over bottom-wall systems: one wave and four per unit of the
    product (many tiny systems and few), equal systems and a list."""
    rng = np.random.default_rng(len(sizes))
    eta, a, N = 1 / (6 * np.pi), 1.0, sum(sizes)
    pos = np.concatenate([rng.uniform(0, 6.0 * max(1.0, (n / 2) ** 0.5), (n, 3)) for n in sizes])
    pos[:, 2] = rng.uniform(1.5, 12.0, N)
    s = _solver(True, a, eta, precision=precision)
    s.initialize(viscosity=eta, hydrodynamicRadius=a, tolerance=TOL)
    s.setSystems(sizes)
    s.setPositions(pos)
    lz = oracle.LanczosOracle()
    W = rng.normal(size=3 * N)
    u, _ = s.sqrtMdotW_with_noise(W)
    ref, it = lz.run(lambda v: oracle.mdot(pos, eta, a, F=v, wall=True, sys_sizes=sizes)[0], W, TOL)
    assert abs(s.lastLanczosIterations() - it) <= 1
    # FP32 pair terms (6e-8 each) add to the tolerance
    assert np.linalg.norm(u.ravel() - ref) <= (2 * TOL if precision == "fp64" else 4 * TOL) * np.linalg.norm(ref)


@pytest.mark.parametrize("angular,N", [(False, 65), (False, 1365), (False, 1366),
                                       (True, 65), (True, 682), (True, 683)])
@pytest.mark.parametrize("precision", ["fp64", "fp32"])
@pytest.mark.parametrize("params,tiling", [
    ({}, (0, 0)), ({"algorithm": "block"}, (0, 0)), ({"algorithm": "block"}, (1, 1)),
    ({"algorithm": "block"}, (0, 1)), ({"algorithm": "naive"}, (1, 0)), ({}, (1, 1)), ({}, (1, 3))])
def test_open_step_lengths_vs_oracle(angular, N, precision, params, tiling):
    """Open systems, where the product finishes the step before it up to 4096
    entries: not with one source chunk, whichever of the tiling and the
    algorithm asks for it."""
    from libmobility_amd import NBody
    rng = np.random.default_rng(N)
    eta, a = 1 / (6 * np.pi), 1.0
    # dilute: the solve converges before orthogonality is lost (as above; a product
    # perturbed by 1e-7 moves the oracle's own result by 3e-7 at most)
    pos = rng.uniform(0, 25.0 * N ** (1 / 3), (N, 3))
    s = NBody("open", "open", "open")
    s.setParameters(**params)
    s.setPairPrecision(precision)
    s.setPairTiling(*tiling)
    s.initialize(viscosity=eta, hydrodynamicRadius=a, includeAngular=angular, tolerance=TOL)
    s.setPositions(pos)

    def product(v):
        F, T = (v[:3 * N], v[3 * N:]) if angular else (v, None)
        U, W = oracle.mdot(pos, eta, a, F=F, T=T, angular=angular)
        return np.concatenate([U, W]) if angular else U

    W = rng.normal(size=(6 if angular else 3) * N)
    u, w = s.sqrtMdotW_with_noise(W)
    got = np.concatenate([u.ravel(), w.ravel()]) if angular else u.ravel()
    ref, it = oracle.LanczosOracle().run(product, W, TOL)
    assert abs(s.lastLanczosIterations() - it) <= 1
    assert np.linalg.norm(got - ref) <= (2 * TOL if precision == "fp64" else 4 * TOL) * np.linalg.norm(ref)


@pytest.mark.parametrize("N", [399, 400])
@pytest.mark.parametrize("precision", ["fp64", "fp32"])
def test_open_steps_with_torques_vs_oracle(N, precision):
    """With torques the product finishes the step before it from 400 particles."""
    test_open_step_lengths_vs_oracle(True, N, precision, {}, (0, 0))
