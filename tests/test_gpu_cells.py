"""Cells of the coarse level found on the device (one system) against the
oracle's rule: few particles, one cell, more particles in a cell than the
device ranks (4096), a cap on the cells, planes, lines and a far outlier."""
import numpy as np
import pytest

from oracle import coarse

pytestmark = pytest.mark.gpu


def _positions(shape, N):
    rng = np.random.default_rng(N)
    x = rng.uniform(0, 4.0 * max(1.0, N ** (1 / 3)), (N, 3))
    if shape == "plane":
        x[:, 1] = 2.5
    elif shape == "line":
        x[:, :2] = 1.0
    elif shape == "outlier":
        x[-1] = 400.0
    return x


@pytest.mark.parametrize("shape,N,ppc,cap", [
    ("cube", 1, 8, 0), ("cube", 2, 1, 0), ("cube", 255, 8, 0), ("cube", 257, 1, 0),
    ("cube", 3000, 16, 0), ("cube", 3000, 16, 150), ("cube", 4200, 5000, 0), ("cube", 4096, 5000, 0),
    ("plane", 700, 8, 0), ("line", 300, 8, 0), ("outlier", 1500, 8, 0)])
def test_cells_vs_oracle(shape, N, ppc, cap):
    from libmobility_amd import NBody
    pos = _positions(shape, N)
    s = NBody("open", "open", "open")
    s.setParameters()
    s.initialize(viscosity=1 / (6 * np.pi), hydrodynamicRadius=1.0, tolerance=1e-3)
    s.setPositions(pos)
    s.setCoarseLevel(ppc)
    if cap:
        s.setCoarseMaxDim(cap)
    for _ in range(2):  # the second build reuses the buffers
        s.setPositions(pos)
        s.sqrtMdotW_with_noise(np.ones(3 * N))
        cell_of, grid, C = s.coarseCells()
        ref, g, Cr = coarse.coarse_cells(pos, ppc, cap) if cap else coarse.coarse_cells(pos, ppc)
        assert C == Cr and list(grid) == list(g)
        assert np.array_equal(cell_of, ref)
