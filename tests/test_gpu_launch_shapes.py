"""The launch shapes' tuning of the step kernels."""
import ctypes as C

import pytest

from test_gpu_step_ends import FUSED64, MIXED, lattice


def settled(sim, kernel):
    s = C.c_int(-1)
    assert sim.abi.launch_config(sim.handle, kernel, None, None, C.byref(s)) == 1
    return s.value


@pytest.mark.gpu
def test_each_precision_tunes_its_own_step():
    """140,000 voxels: the mixed step splits link directions and has nothing to tune, the FP64 fused step
    has a voxel per lane; the first does not settle the second's launch shape"""
    sim = lattice(0, 140000)
    sim.setPrecision(MIXED)
    sim.step(1e-5, 3)
    assert settled(sim, 0) == 1
    sim.setPrecision(FUSED64)
    sim.step(1e-5, 3)
    assert settled(sim, 0) == 0
    sim.step(1e-5, 30)
    assert settled(sim, 0) == 1
    sim.setPrecision(MIXED)
    sim.step(1e-5, 3)
    assert settled(sim, 0) == 1
