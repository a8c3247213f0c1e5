"""A checkpoint saved before a material has a Poisson's ratio, restored after: the links' transverse info is
what it was then, on the fused FP64 step as on the split one, bit for bit."""
import numpy as np
import pytest

import backends as B


@pytest.mark.gpu
@pytest.mark.parametrize("before", [1, 2, 5])
@pytest.mark.parametrize("grown", [False, True])
def test_checkpoint_from_before_a_poissons_ratio(before, grown):
    sims = []
    for path in (0, 1):
        sim = B.maker(B.product_abi(), path)(0.005)
        mats = [sim.addMaterial(1e6, 1000.0), sim.addMaterial(5e6, 1500.0)]
        sim.setGravity(1.0)
        sim.enableFloor(True)
        i = np.arange(240)
        sim.setVoxels((i % 3 == 0).astype(np.int32), np.stack([i % 5, (i // 5) % 6, i // 30], 1))
        if grown:   # the halves of the state are enlarged between two launches
            sim.step(1e-5, 1)
            sim.setVoxels(np.zeros(60, np.int32), np.stack([i[:60] % 5, (i[:60] // 5) % 6, 8 + i[:60] // 30], 1))
        sim.step(1e-5, before)
        sim.checkpointSave(0)
        mats[0].setPoissonsRatio(0.3)   # links of the other material keep what they have
        sim.step(1e-5, 4)
        sim.checkpointRestore(0)
        first = sim.link_transverse()
        sim.step(1e-5, 7)
        sims.append((sim.state(), sim.link_state(), first, sim.link_transverse()))
    for x, y in zip(*sims):
        bad = [k for k in x if x[k].tobytes() != y[k].tobytes()]
        assert not bad, bad
    assert (sims[0][2]["area"] > 0).all()
