"""FP32 sums of the ordered wall kernel: U and W are one accumulator each over the
blocks of forces and torques."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("tiling", [(1, 8), (2, 0)])
def test_error_of_forces_and_torques_together(tiling):
    """The roundings of the two blocks are independent, so the error of a product with
    forces and torques is no larger than those of the two alone, squares added."""
    import torch
    from libmobility_amd import NBody
    N = 17000
    rng = np.random.default_rng(5)
    pos = rng.uniform(0, 70.0, (N, 3))
    pos[:, 2] = rng.uniform(1.0, 15.0, N)
    pos, F, T = (torch.as_tensor(x, device="cuda")
                 for x in (pos, rng.normal(size=(N, 3)), rng.normal(size=(N, 3))))
    errors = []
    for f, t in ((F, None), (None, T), (F, T)):
        got = []
        for precision in ("fp64", "fp32"):
            s = NBody("open", "open", "single_wall")
            s.setParameters(wallHeight=0.0)
            s.setPairPrecision(precision)
            s.setPairSymmetric(0)
            s.setPairTiling(*tiling)
            s.initialize(viscosity=1 / (6 * np.pi), hydrodynamicRadius=1.0, includeAngular=True)
            s.setPositions(pos)
            got.append(s.Mdot(f, t))
            assert not s.lastPairSymmetric()
        errors.append([float((a - b).norm()) for a, b in zip(*got)])
    for forces, torques, both in zip(*errors):
        # 51000 components: the measured norms are within 1 % of their expectation
        assert both <= 1.02 * np.hypot(forces, torques)
