"""The product of small systems with sources across the lanes (wide_kernels.hip)
against the CPU oracle, at the sizes where its units of 4 targets and groups of
64 sources have remainders, and in every form it accepts."""
import numpy as np
import pytest

import oracle

pytestmark = pytest.mark.gpu

ETA, A = 0.9, 1.1


def _solver(wall, angular, precision, **params):
    from libmobility_amd import NBody
    s = NBody("open", "open", "single_wall" if wall else "open")
    if wall:
        params["wallHeight"] = 0.0
    s.setParameters(**params)
    s.setPairPrecision(precision)
    s.initialize(viscosity=ETA, hydrodynamicRadius=A, includeAngular=angular)
    return s


def _cloud(N, wall, seed):
    rng = np.random.default_rng(seed)
    # dense enough for overlaps, with heights down to below one radius
    pos = rng.uniform(0, 2.2 * A * max(1.0, N ** (1 / 3)), (N, 3))
    if wall:
        pos[:, 2] = rng.uniform(0.3 * A, 8 * A, N)
    if N >= 4:
        pos[N - 1] = pos[0]  # coincident
    return pos, rng.normal(size=(N, 3)), rng.normal(size=(N, 3))


def _rel(x, y):
    return np.linalg.norm(np.asarray(x).ravel() - y) / np.linalg.norm(y)


# FP64: a few hundred roundings of 1.1e-16 in sums that hardly cancel.  FP32
# pair terms: tens of roundings of 6e-8, and wall cross blocks that cancel.
TOL = {"fp64": 1e-12, "fp32": 1e-5}


@pytest.mark.parametrize("N", [1, 2, 3, 4, 5, 63, 64, 65, 127, 255, 256, 257, 1001, 2050])
@pytest.mark.parametrize("wall,angular", [(False, False), (False, True), (True, False), (True, True)])
@pytest.mark.parametrize("precision", ["fp64", "fp32"])
def test_single_system_vs_oracle(N, wall, angular, precision):
    pos, F, T = _cloud(N, wall, N)
    s = _solver(wall, angular, precision)
    s.setPositions(pos)
    for f, t in ((F, None), (F, T), (None, T)) if angular else ((F, None),):
        U, W = s.Mdot(f, t)
        assert s.lastPairTiling() == (4, 1) and not s.lastPairSymmetric()
        Uo, Wo = oracle.mdot(pos, ETA, A, F=f, T=t, angular=angular, wall=wall)
        for got, ref in ((U, Uo), (W, Wo)) if angular else ((U, Uo),):
            # one free particle has no cross terms: both sides are zero there
            assert np.linalg.norm(got.ravel() - ref) <= TOL[precision] * max(np.linalg.norm(ref), 1e-300)


@pytest.mark.parametrize("nbatch,per", [(7, 1), (3, 66), (200, 50), (90, 131), (2, 3001)])
@pytest.mark.parametrize("wall,angular", [(False, False), (True, True)])
@pytest.mark.parametrize("precision", ["fp64", "fp32"])
def test_equal_batches_vs_oracle(nbatch, per, wall, angular, precision):
    """Few and many units: four waves per unit and one."""
    parts = [_cloud(per, wall, 100 + b) for b in range(nbatch)]
    pos, F, T = (np.concatenate([p[k] for p in parts]) for k in range(3))
    s = _solver(wall, angular, precision, Nbatch=nbatch, NperBatch=per)
    s.setPositions(pos)
    U, W = s.Mdot(F, T if angular else None)
    assert s.lastPairTiling() == (4, 1)
    Uo, Wo = oracle.mdot(pos, ETA, A, F=F, T=T if angular else None, angular=angular, wall=wall,
                         sys_sizes=[per] * nbatch)
    assert _rel(U, Uo) <= TOL[precision]
    if angular:
        assert _rel(W, Wo) <= TOL[precision]


@pytest.mark.parametrize("sizes", [(1, 70, 0, 300, 5), (64,) * 40 + (1, 2, 1500), (300, 17) * 60])
@pytest.mark.parametrize("angular", [False, True])
@pytest.mark.parametrize("precision", ["fp64", "fp32"])
def test_ragged_mixed_systems_vs_oracle_and_the_general_kernel(sizes, angular, precision):
    from libmobility_amd import NBody
    kinds = [k % 2 for k in range(len(sizes))]
    parts = [_cloud(n, k, 7 + i) for i, (n, k) in enumerate(zip(sizes, kinds)) if n]
    pos, F, T = (np.concatenate([p[k] for p in parts]) for k in range(3))
    out = []
    for tiling in (0, 1):
        s = NBody("open", "open", "single_wall")
        s.setParameters(wallHeight=0.0)
        s.setSystems(sizes, kinds=kinds)
        s.setPairPrecision(precision)
        s.setPairTiling(tiling, 0)
        s.initialize(viscosity=ETA, hydrodynamicRadius=A, includeAngular=angular)
        s.setPositions(pos)
        out.append(s.Mdot(F, T if angular else None))
        assert (s.lastPairTiling() == (4, 1)) == (tiling == 0)
    Uo, Wo = oracle.mdot(pos, ETA, A, F=F, T=T if angular else None, angular=angular, wall=kinds,
                         sys_sizes=sizes)
    for k, ref in enumerate((Uo, Wo) if angular else (Uo,)):
        assert _rel(out[0][k], ref) <= TOL[precision]
        assert _rel(out[0][k], np.asarray(out[1][k]).ravel()) <= 2 * TOL[precision]


def test_infinite_and_nan_forces_stay_with_their_system():
    parts = [_cloud(70, False, k) for k in range(3)]
    pos, F = (np.concatenate([p[k] for p in parts]) for k in range(2))
    pos[[69, 139, 209]] += 0.5  # no coincident pair: 0 * inf only there
    F[75] = np.inf
    F[150] = np.nan
    s = _solver(False, False, "fp64", Nbatch=3, NperBatch=70)
    s.setPositions(pos)
    U, _ = s.Mdot(F)
    assert np.isfinite(U[:70]).all()
    assert not np.isfinite(U[70:140]).any() and np.isnan(U[140:]).all()


@pytest.mark.parametrize("wall", [False, True])
def test_fp32_sums_of_a_large_system_among_small_ones(wall):
    """A system of 60000 in an ensemble whose mean size selects one wave per four
    targets: a lane's 938 terms are not one FP32 sum.  The worst case of such a sum
    is equal terms: one target, and all other particles at one place."""
    import torch
    from libmobility_amd import NBody
    big, small, count = 60000, 64, 39700
    sizes = [big] + [small] * count
    N = sum(sizes)
    g = torch.Generator(device="cuda")
    g.manual_seed(1)
    pos = torch.rand((N, 3), generator=g, device="cuda", dtype=torch.float64) * 40.0 + 1.0
    pos[:big] = torch.tensor([128.0, 0.0, 64.0], dtype=torch.float64)
    pos[0] = torch.tensor([0.0, 0.0, 64.0], dtype=torch.float64)
    got = {}
    for precision in ("fp64", "fp32"):
        s = NBody("open", "open", "single_wall" if wall else "open")
        s.setParameters(**({"wallHeight": 0.0} if wall else {}))
        s.setPairPrecision(precision)
        s.initialize(viscosity=1 / (6 * np.pi), hydrodynamicRadius=1.0)
        s.setSystems(sizes)
        s.setPositions(pos)
        u = []
        for f in np.geomspace(1.0, 2.0, 24, endpoint=False):
            F = torch.zeros((N, 3), dtype=torch.float64, device="cuda")
            F[1:big, 1] = float(f)
            u.append(float(s.Mdot(F)[0][0, 1]))
            assert s.lastPairTiling() == (4, 1)
        got[precision] = np.array(u)
    error = np.abs(got["fp32"] / got["fp64"] - 1).max()
    # 256 equal terms: each addition rounds by half an ulp of the sum so far, at most
    # 2^-24 (1 + 2 + ... + 256) / 256 of the sum; the terms themselves some 1e-6 (a
    # dozen roundings of 6e-8, with the wall's differences of open and image terms)
    assert error <= 129 * 2.0 ** -24 + 1.5e-6
