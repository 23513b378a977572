"""The symmetric evaluation with its default shapes, forced on at sizes around
its tiles (64 particles per wave, one wave per item below 16384 particles):
one tile, odd and even tile counts, nearly empty last tiles, several passes
over the ring, one system and ensembles, against the CPU oracle."""
import numpy as np
import pytest

import oracle

pytestmark = pytest.mark.gpu

ETA, A = 0.9, 1.1
TOL = {"fp64": 1e-12, "fp32": 1e-5}


def _cloud(N, wall, seed):
    rng = np.random.default_rng(seed)
    pos = rng.uniform(0, 2.2 * A * max(1.0, N ** (1 / 3)), (N, 3))
    if wall:
        pos[:, 2] = rng.uniform(0.3 * A, 8 * A, N)
    return pos, rng.normal(size=(N, 3)), rng.normal(size=(N, 3))


def _check(s, pos, F, T, angular, wall, sizes, tol):
    for f, t in ((F, None), (F, T), (None, T)) if angular else ((F, None),):
        U, W = s.Mdot(f, t)
        assert s.lastPairSymmetric()
        Uo, Wo = oracle.mdot(pos, ETA, A, F=f, T=t, angular=angular, wall=wall, sys_sizes=sizes)
        for got, ref in ((U, Uo), (W, Wo)) if angular else ((U, Uo),):
            assert np.linalg.norm(got.ravel() - ref) <= tol * max(np.linalg.norm(ref), 1e-300)


@pytest.mark.parametrize("N,slabs", [(1, 0), (64, 0), (65, 0), (128, 0), (129, 0), (255, 0),
                                     (257, 0), (513, 0), (1000, 0), (1000, 6), (2111, 9)])
@pytest.mark.parametrize("wall,angular", [(False, False), (False, True), (True, False), (True, True)])
@pytest.mark.parametrize("precision", ["fp64", "fp32"])
def test_one_system_vs_oracle(N, slabs, wall, angular, precision):
    """slabs: room for that many partial sums, so the ring takes several passes."""
    from libmobility_amd import NBody
    pos, F, T = _cloud(N, wall, N)
    s = NBody("open", "open", "single_wall" if wall else "open")
    s.setParameters(**({"wallHeight": 0.0} if wall else {}))
    s.setPairPrecision(precision)
    s.setPairSymmetric(1, memoryBytes=slabs * 24 * N * (2 if angular else 1))
    s.initialize(viscosity=ETA, hydrodynamicRadius=A, includeAngular=angular)
    s.setPositions(pos)
    _check(s, pos, F, T, angular, wall, None, TOL[precision])


@pytest.mark.parametrize("sizes", [(64, 65, 0, 1, 300), (1500, 130, 129), (200,) * 7])
@pytest.mark.parametrize("kinds", ["open", "wall", "mixed"])
@pytest.mark.parametrize("angular", [False, True])
@pytest.mark.parametrize("precision", ["fp64", "fp32"])
def test_ensembles_vs_oracle(sizes, kinds, angular, precision):
    from libmobility_amd import NBody
    walls = [kinds == "wall" or (kinds == "mixed" and k % 2 == 0) for k in range(len(sizes))]
    parts = [_cloud(n, w, 7 + k) for k, (n, w) in enumerate(zip(sizes, walls))]
    pos, F, T = (np.concatenate([p[k] for p in parts]) for k in range(3))
    s = NBody("open", "open", "single_wall")
    s.setParameters(wallHeight=0.0)
    s.setPairPrecision(precision)
    s.setPairSymmetric(1)
    s.initialize(viscosity=ETA, hydrodynamicRadius=A, includeAngular=angular)
    s.setSystems(sizes, ["single_wall" if w else "open" for w in walls])
    s.setPositions(pos)
    for f, t in ((F, None), (F, T)) if angular else ((F, None),):
        U, W = s.Mdot(f, t)
        assert s.lastPairSymmetric()
        Uo, Wo = oracle.mdot(pos, ETA, A, F=f, T=t, angular=angular, wall=walls, sys_sizes=sizes)
        assert np.linalg.norm(U.ravel() - Uo) <= TOL[precision] * np.linalg.norm(Uo)
        if angular:
            assert np.linalg.norm(W.ravel() - Wo) <= TOL[precision] * np.linalg.norm(Wo)


@pytest.mark.parametrize("slabs", [70, 20])
@pytest.mark.parametrize("angular", [False, True])
def test_partial_sums_of_a_mixed_ensemble_fit_their_memory(slabs, angular):
    """Open systems have the longest rings and the longest items, the walls' items
    are shorter: the memory limit holds for what both need."""
    import torch
    from libmobility_amd import NBody
    sizes, walls = [6000] * 11 + [1000] * 8, [False] * 11 + [True] * 8
    parts = [_cloud(n, w, 7 + k) for k, (n, w) in enumerate(zip(sizes, walls))]
    pos, F, T = (torch.as_tensor(np.concatenate([p[k] for p in parts]), device="cuda") for k in range(3))
    if not angular:
        T = None
    N = sum(sizes)
    limit = slabs * 24 * N * (2 if angular else 1)
    results = []
    for memory in (limit, 0):
        s = NBody("open", "open", "single_wall")
        s.setParameters(wallHeight=0.0)
        s.setPairSymmetric(1, memoryBytes=memory)
        s.initialize(viscosity=ETA, hydrodynamicRadius=A, includeAngular=angular)
        s.setSystems(sizes, ["single_wall" if w else "open" for w in walls])
        s.setPositions(pos)
        torch.cuda.synchronize()
        out = [torch.empty_like(pos) for _ in range(3)]  # the allocator has what Mdot returns
        del out
        free = torch.cuda.mem_get_info()[0]
        results.append(s.Mdot(F, T))
        taken = free - torch.cuda.mem_get_info()[0]
        if memory:
            # besides: 20 bytes per item, at most some 10^5 of them, and page granularity
            assert taken <= limit + (8 << 20)
    for got, ref in zip(*results):
        if ref is not None:
            assert float((got - ref).norm()) <= 1e-12 * float(ref.norm())


@pytest.mark.parametrize("tiling", [(0, 0), (1, 0), (1, 3), (2, 0), (2, 5), (0, 7)])
@pytest.mark.parametrize("slabs", [0, 9])
@pytest.mark.parametrize("kinds", ["open", "mixed"])
def test_work_lists_of_ensembles(tiling, slabs, kinds):
    """Rings whose items have two lengths, shared evenly or with a rest, in one pass
    and in several: every pair is met once."""
    from libmobility_amd import NBody
    sizes = (1500, 64, 0, 1, 2111, 700, 129)
    walls = [kinds == "mixed" and k % 2 == 0 for k in range(len(sizes))]
    parts = [_cloud(n, w, 7 + k) for k, (n, w) in enumerate(zip(sizes, walls))]
    pos, F, _ = (np.concatenate([p[k] for p in parts]) for k in range(3))
    s = NBody("open", "open", "single_wall")
    s.setParameters(wallHeight=0.0)
    s.setPairSymmetric(1, memoryBytes=slabs * 24 * sum(sizes))
    s.setPairTiling(*tiling)
    s.initialize(viscosity=ETA, hydrodynamicRadius=A)
    s.setSystems(sizes, ["single_wall" if w else "open" for w in walls])
    s.setPositions(pos)
    U, _ = s.Mdot(F)
    assert s.lastPairSymmetric()
    Uo, _ = oracle.mdot(pos, ETA, A, F=F, wall=walls, sys_sizes=sizes)
    assert np.linalg.norm(U.ravel() - Uo) <= TOL["fp64"] * np.linalg.norm(Uo)


@pytest.mark.parametrize("angular", [False, True])
@pytest.mark.parametrize("precision", ["fp64", "fp32"])
@pytest.mark.parametrize("per_system", [False, True])
def test_order_keeping_products_of_mixed_ensembles(angular, precision, per_system):
    """Square roots over open and wall systems around the tiles of 256 and their
    blocks of 64, applied twice, against the product."""
    from libmobility_amd import NBody
    sizes = (1, 63, 64, 65, 100, 0, 128, 129, 255, 256, 257, 330, 513)
    walls = [k % 2 == 0 for k in range(len(sizes))]
    parts = [_cloud(n, w, 7 + k) for k, (n, w) in enumerate(zip(sizes, walls))]
    pos, F, T = (np.concatenate([p[k] for p in parts]) for k in range(3))
    pos *= 3.0  # dilute: few iterations
    s = NBody("open", "open", "single_wall")
    s.setParameters(wallHeight=0.0)
    s.setPairPrecision(precision)
    s.setPairSymmetric(1)
    s.initialize(viscosity=ETA, hydrodynamicRadius=A, includeAngular=angular, tolerance=1e-6)
    s.setSystems(sizes, ["single_wall" if w else "open" for w in walls])
    s.setLanczosPerSystem(per_system)
    s.setPositions(pos)

    def root(x):
        out = s.sqrtMdotW_with_noise(x)
        assert s.lastPairSymmetric()
        return np.concatenate([v.ravel() for v in out if v is not None])

    z = np.concatenate([F.ravel(), T.ravel()]) if angular else F.ravel()
    got = root(root(z))
    ref = np.concatenate([v for v in oracle.mdot(pos, ETA, A, F=F, T=T if angular else None,
                                                 angular=angular, wall=walls, sys_sizes=sizes)
                          if v is not None])
    off = np.concatenate([[0], np.cumsum(sizes)])
    for a, b in zip(off, off[1:]):
        g, r = (x.reshape(-1, len(pos), 3)[:, a:b] for x in (got, ref))
        # two roots that end some 1e-6 from theirs; a block left out is far off in its system
        assert np.linalg.norm(g - r) <= 1e-4 * max(np.linalg.norm(r), 1e-300)


@pytest.mark.parametrize("sizes", [(300,) * 70, (300,) * 130, (2111,) * 8, (2111,) * 20])
def test_open_fp32_ensembles_with_few_and_many_items(sizes):
    """Up to two workgroups per CU the open translational kernel runs without its
    scheduling fences: 280 and 520 items, some 400 and 1000."""
    from libmobility_amd import NBody
    parts = [_cloud(n, False, 7 + k) for k, n in enumerate(sizes)]
    pos, F = (np.concatenate([p[k] for p in parts]) for k in range(2))
    results = {}
    for precision in ("fp64", "fp32"):
        s = NBody("open", "open", "open")
        s.setParameters()
        s.setPairPrecision(precision)
        s.setPairSymmetric(1)
        s.initialize(viscosity=ETA, hydrodynamicRadius=A)
        s.setSystems(sizes)
        s.setPositions(pos)
        results[precision], _ = s.Mdot(F)
        assert s.lastPairSymmetric()
    Uo, _ = oracle.mdot(pos[:sizes[0]], ETA, A, F=F[:sizes[0]], wall=False)
    assert np.linalg.norm(results["fp64"][:sizes[0]].ravel() - Uo) <= TOL["fp64"] * np.linalg.norm(Uo)
    error = np.linalg.norm(results["fp32"] - results["fp64"])
    assert error <= TOL["fp32"] * np.linalg.norm(results["fp64"])
