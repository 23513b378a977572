"""setSystems applies to the next setPositions: until then every call works on the
systems that the current positions came with."""
import numpy as np
import pytest

import oracle

pytestmark = pytest.mark.gpu

ETA, A = 0.9, 1.1
OLD, OLD_WALL = (400, 130, 129), [True, False, True]
NEW, NEW_WALL = (1, 64, 65, 0, 200, 29, 300), [False, True, True, False, False, True, False]


def _inputs(N):
    rng = np.random.default_rng(N)
    pos = rng.uniform(0, 3.0 * A * N ** (1 / 3), (N, 3))
    pos[:, 2] = rng.uniform(0.3 * A, 8 * A, N)
    return pos, rng.normal(size=(N, 3)), rng.normal(size=(N, 3))


def _solver(precision, symmetric):
    from libmobility_amd import NBody
    s = NBody("open", "open", "single_wall")
    s.setParameters(wallHeight=0.0)
    s.setPairPrecision(precision)
    s.setPairSymmetric(symmetric)
    s.initialize(viscosity=ETA, hydrodynamicRadius=A, includeAngular=True)
    return s


def _kinds(wall):
    return ["single_wall" if w else "open" for w in wall]


def _right(s, pos, F, T, sizes, wall, precision):
    tol = 1e-12 if precision == "fp64" else 1e-5
    U, W = s.Mdot(F, T)
    Uo, Wo = oracle.mdot(pos, ETA, A, F=F, T=T, angular=True, wall=wall, sys_sizes=sizes)
    return (np.linalg.norm(U.ravel() - Uo) <= tol * np.linalg.norm(Uo)
            and np.linalg.norm(W.ravel() - Wo) <= tol * np.linalg.norm(Wo))


@pytest.mark.parametrize("precision", ["fp64", "fp32"])
@pytest.mark.parametrize("symmetric", [0, 1])
@pytest.mark.parametrize("warm", [False, True])
def test_products_before_the_next_positions(precision, symmetric, warm):
    s = _solver(precision, symmetric)
    pos, F, T = _inputs(sum(OLD))
    s.setSystems(OLD, _kinds(OLD_WALL))
    s.setPositions(pos)
    if warm:
        assert _right(s, pos, F, T, OLD, OLD_WALL, precision)
    s.setSystems(NEW, _kinds(NEW_WALL))
    assert s._lib.lm_nbody_num_systems(s._h) == len(OLD)
    assert _right(s, pos, F, T, OLD, OLD_WALL, precision)
    s.setPositions(pos)
    assert s._lib.lm_nbody_num_systems(s._h) == len(NEW)
    assert _right(s, pos, F, T, NEW, NEW_WALL, precision)


@pytest.mark.parametrize("sizes", [(100, 50), (1000, 2000)])
@pytest.mark.parametrize("symmetric", [0, 1])
def test_systems_of_another_total(sizes, symmetric):
    s = _solver("fp64", symmetric)
    pos, F, T = _inputs(sum(OLD))
    s.setSystems(OLD, _kinds(OLD_WALL))
    s.setPositions(pos)
    s.setSystems(sizes)
    assert _right(s, pos, F, T, OLD, OLD_WALL, "fp64")
    with pytest.raises(RuntimeError, match="do not cover"):
        s.setPositions(pos)
    assert _right(s, pos, F, T, OLD, OLD_WALL, "fp64")
    pos, F, T = _inputs(sum(sizes))
    s.setPositions(pos)
    assert _right(s, pos, F, T, sizes, True, "fp64")
