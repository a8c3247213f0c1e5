"""A reset on the device leaves vxg_robot_com_noalloc refusing as one through the mirror does: until a
step, or vxg_robot_com, has made the reset state the resident one."""
import pytest

from test_gpu_reset_on_device import build, run


@pytest.mark.gpu
@pytest.mark.parametrize("act", [False, True])
def test_no_allocation_read_after_a_reset(act):
    sim, _ = build(1, act)
    for _ in range(2):
        sim.resetTime()  # the first through the mirror, the second on the device
        with pytest.raises(RuntimeError, match="pending edits"):
            sim.robotComNoAlloc()
        want = sim.robotCom()
        assert sim.robotComNoAlloc().tobytes() == want.tobytes()
        run(sim)
        assert sim.robotComNoAlloc().tobytes() == sim.robotCom().tobytes()
