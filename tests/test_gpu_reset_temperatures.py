"""Temperatures the host sets after a reset on the device are kept until the device sets its own: a
read, or the end of actuation, brings the state back without them.  Two simulations go through the same
calls; in one of them a material's setter, called with the value it has, sends the reset through the
host mirror."""
import numpy as np
import pytest

from test_gpu_reset_on_device import build, hot, run


def one(sim):
    sim.setAmbientTemperature(7.5, True)
    hot(sim)


@pytest.mark.gpu
@pytest.mark.parametrize("precision", [1, 2])
@pytest.mark.parametrize("between", ["state", "link_state", "no actuation", "moduli"])
def test_temperatures_set_after_a_reset(between, precision):
    got = []
    for mirror in (False, True):
        sim, mats = build(precision, True)
        sim.resetTime()
        run(sim)
        if mirror:
            mats[0].setStaticFriction(mats[0].staticFriction())
        sim.resetTime()
        one(sim)
        if between == "moduli":
            sim.setModuli(np.full(sim.voxelCount(), 1.5e6, np.float32))
        elif between == "no actuation":
            sim.setActuation(False)
        else:
            getattr(sim, between)()
        r = {"temperature": np.array([sim.voxel(i).temperature() for i in range(sim.voxelCount())])}
        r["rest"] = sim.link_state()["restLength"]
        dt = np.full(sim.robotCount(), 1e-4, np.float32)
        dt[0] = 0.0   # under actuation the robots that step take the device's
        sim.robotStep(9, dt)
        r.update(sim.state())
        r["temperature after"] = np.array([sim.voxel(i).temperature() for i in range(sim.voxelCount())])
        got.append(r)
    assert got[0]["temperature"][3] == 12.5 and got[0]["temperature"][5] == 7.5
    bad = [k for k in got[0] if got[0][k].tobytes() != got[1][k].tobytes()]
    assert not bad, bad
