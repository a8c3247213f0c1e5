"""A reset of the fused steps' state on the device against the reset through the host mirror, bit
for bit, over what may come before and after it.  Two simulations go through the same calls; in one
of them a material's setter, called with the value it has, sends every reset through the mirror."""
import numpy as np
import pytest

import backends as B
from voxelyze_amd import workloads as W


def build(precision, act):
    sim = B.maker(B.product_abi())(0.005)
    mats = [sim.addMaterial(1e6, 1000.0), sim.addMaterial(5e6, 1500.0)]
    mats[1].setCte(0.01)
    mats[1].setExternalScaleFactor([1.0, 0.9, 1.1])
    sim.setGravity(1.0)
    sim.enableFloor(True)
    for r, (nx, ny, nz) in enumerate([(9, 5, 6), (1, 1, 1), (13, 3, 5)]):
        if r:
            sim.addRobot()
        s = np.arange(nx * ny * nz)
        s = s[(W.uniform(3 + r, s.astype(np.uint64)) < 0.8) | (s == 0)]
        sim.setVoxels((s % 3 == 0).astype(np.int32), np.stack([s % nx, (s // nx) % ny, s // (nx * ny)], 1))
    sim.setPrecision(precision)
    if act:
        n = sim.voxelCount()
        sim.setActuation(True, 1.0, 20.0, 50.0)
        sim.setPhases(W.uniform(9, np.arange(n, dtype=np.uint64)).astype(np.float32))
    return sim, mats


def run(sim):
    return sim.robotStep(17, 1e-4)


def moduli(sim):
    n = sim.voxelCount()
    sim.setModuli((1e6 * (0.5 + W.uniform(2, np.arange(n, dtype=np.uint64)))).astype(np.float32))


def hot(sim):
    sim.voxel(3).setTemperature(12.5)
    sim.voxel(11).setTemperature(-7.25)


BEFORE = {
    "steps": lambda s, m: run(s),
    "a read": lambda s, m: (run(s), s.state()),
    "temperatures": lambda s, m: (hot(s), run(s)),
    "moduli and a force": lambda s, m: (moduli(s), run(s), s.voxel(5).external().setForce(0.0, 0.01, 0.02)),
    "a checkpoint": lambda s, m: (run(s), s.checkpointSave(1), run(s), s.checkpointRestore(1)),
}
AFTER = {
    "steps": lambda s, m: run(s),
    "a read, steps": lambda s, m: (s.state(), run(s)),
    "temperatures": lambda s, m: (hot(s), run(s)),
    "moduli": lambda s, m: (moduli(s), run(s)),
    "a material": lambda s, m: (m[1].setModelLinear(2e6), m[1].setExternalScaleFactor([1.0, 1.0, 0.95]), run(s)),
    "the split FP64 step": lambda s, m: (s.clearModuli(), s.setPrecision(0), run(s)),
    "another reset": lambda s, m: (s.resetTime(), run(s)),
    "no actuation": lambda s, m: (s.setActuation(False), run(s)),
}


def everything(sim):
    t = [sim.voxel(i).temperature() for i in range(0, sim.voxelCount(), 7)]
    info = [sim.stateInfo(i, 1) for i in (0, 1, 2, 4, 5, 6)]
    r = {"temperature": np.array(t), "info": np.array(info)}
    for k, v in list(sim.state().items()) + list(sim.link_state().items()):
        r[k] = v
    r["temperature after"] = np.array([sim.voxel(i).temperature() for i in range(0, sim.voxelCount(), 7)])
    return r


@pytest.mark.gpu
@pytest.mark.parametrize("precision", [1, 2])
@pytest.mark.parametrize("act", [False, True])
@pytest.mark.parametrize("before", list(BEFORE))
def test_reset_on_the_device_equals_the_mirrors(before, act, precision):
    for after in AFTER:
        got = []
        for mirror in (False, True):
            sim, mats = build(precision, act)
            sim.resetTime()
            BEFORE[before](sim, mats)
            if mirror:
                mats[0].setStaticFriction(mats[0].staticFriction())
            sim.resetTime()
            first = [sim.voxel(3).temperature(), sim.currentTime()]
            AFTER[after](sim, mats)
            got.append((first, everything(sim)))
        assert got[0][0] == got[1][0], after
        bad = [k for k, v in got[0][1].items() if v.tobytes() != got[1][1][k].tobytes()]
        assert not bad, (after, bad)
