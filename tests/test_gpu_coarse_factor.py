"""The factors of the coarse level over the counts of 64-row tiles where their
kernels change course: one tile, a block of 4 tile columns, one more, and
several blocks; one matrix at a time, and one workgroup per system."""
import numpy as np
import pytest

import oracle
from oracle import coarse
from libmobility_amd.workloads import rsa_cube

pytestmark = pytest.mark.gpu

ETA = 1.0 / (6 * np.pi)


@pytest.mark.parametrize("nsys,N,ppc,tiles", [
    (1, 600, 400, 1), (1, 600, 20, 2), (1, 600, 8, 3), (1, 95, 1, 4), (1, 100, 1, 5),
    (1, 200, 1, 8), (1, 600, 4, 6), (1, 600, 2, 15),
    (12, 60, 20, 1), (12, 60, 2, 2), (12, 60, 1, 3), (12, 95, 1, 4), (12, 100, 1, 5)])
def test_factors_vs_oracle(nsys, N, ppc, tiles):
    from libmobility_amd import NBody
    parts = [rsa_cube(N, 0.2, seed=5 + q)[0] for q in range(nsys)]
    s = NBody("open", "open", "open")
    s.setParameters(Nbatch=nsys, NperBatch=N)
    s.initialize(viscosity=ETA, hydrodynamicRadius=1.0, tolerance=1e-6)
    s.setPositions(np.concatenate(parts))
    s.setCoarseLevel(ppc)
    s.sqrtMdotW_with_noise(np.random.default_rng(0).normal(size=3 * N * nsys))
    for q in {0, nsys - 1}:
        M = oracle.dense_matrix(parts[q], ETA, 1.0)
        cell_of, _, C = coarse.coarse_cells(parts[q], ppc)
        assert q > 0 or -(-3 * C // 64) == tiles
        L, X = s.coarseFactors(q)
        Mc = coarse.coarse_matrix(M, cell_of, C)
        assert np.allclose(L, np.tril(L))
        # FP32 pair terms in the matrix; the inverse to FP64 rounding (entries of
        # L up to some units, conditioning of tens)
        assert np.linalg.norm(L @ L.T - Mc) <= 1e-5 * np.linalg.norm(Mc)
        assert np.abs(X @ L - np.eye(3 * C)).max() <= 1e-11
