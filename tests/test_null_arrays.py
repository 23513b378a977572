"""Null arrays through the C ABI come back as errors, on both sides of the size
up to which host arrays go through the solver's mapped buffer (16384 particles)."""
import ctypes

import numpy as np
import pytest

def _solver():
    from libmobility_amd import NBody
    s = NBody("open", "open", "open")
    s.setParameters()
    s.initialize(viscosity=1.0, hydrodynamicRadius=1.0)
    return s


@pytest.mark.parametrize("mem", [0, 1])
@pytest.mark.parametrize("n", [1, 16384, 16385])
def test_null_positions(n, mem):
    s = _solver()
    lib, h = s._lib, s._h
    assert lib.lm_nbody_set_positions(h, None, 3 * n, mem) != 0
    assert b"positions array" in lib.lm_last_error()
    assert lib.lm_nbody_num_particles(h) <= 0


@pytest.mark.gpu
@pytest.mark.parametrize("mem", [0, 1])
@pytest.mark.parametrize("n", [1, 16384, 16385])
def test_null_output(n, mem):
    import torch
    s = _solver()
    lib, h = s._lib, s._h
    x = np.random.default_rng(n).uniform(0, 3 * n ** (1 / 3), (n, 3))
    d = torch.as_tensor(x, device="cuda")
    torch.cuda.synchronize()
    p = ctypes.c_void_p(d.data_ptr() if mem else x.ctypes.data)
    assert lib.lm_nbody_set_positions(h, p, 3 * n, mem) == 0
    for forces in (p, None):
        assert lib.lm_nbody_mdot(h, forces, 3 * n, None, 0, None, None, mem) != 0
        assert b"linear output array" in lib.lm_last_error()
