"""The self-collision watch list where one voxel's partners fill, and pass, the list that the device
sorts beside the search, and where voxels share one cell, against the oracle, bit for bit: a cloud of
fixed voxels drawn together around a free one (its forces are summed in partner order, so the order
shows in its bits), and a falling block of many surface voxels."""
import numpy as np
import pytest

import backends as B
from voxelyze_amd import workloads as W


def cloud(abi, n):
    sim = B.maker(abi)(0.01)
    m = sim.addMaterial(1e5, 1000.0)
    u = W.uniform(21, np.arange(3 * n, dtype=np.uint64)).reshape(n, 3)
    side = int(np.ceil(n ** (1 / 3)))
    at = np.array([[2 * (k % side), 2 * (k // side % side), 2 * (k // side ** 2)] for k in range(n)])
    free = n // 2
    for k in range(n):
        v = sim.setVoxel(m, *map(int, at[k]))
        if k != free:  # drawn to within half a pitch of the free one
            v.external().setDisplacementAll(0.01 * (at[free] + u[k] - 0.5 - at[k]))
    sim.enableCollisions(True)
    return sim


def block(abi, n):
    sim = B.maker(abi)(0.01)
    m = sim.addMaterial(1e5, 1000.0)
    s = np.arange(n ** 3)
    s = s[W.uniform(5, s.astype(np.uint64)) < 0.6]
    for k in map(int, s):
        sim.setVoxel(m, k % n, k // n % n, k // n ** 2 + 2)
    sim.setGravity(60.0)
    sim.enableFloor(True)
    sim.enableCollisions(True)
    return sim


@pytest.mark.gpu
@pytest.mark.parametrize("model,n", [(cloud, n) for n in (1, 2, 33, 64, 65, 66, 150)] + [(block, n) for n in (3, 7)])
def test_watch_list_equals_the_oracles(model, n):
    a, b = model(B.product_abi(), n), model(B.oracle_cr_abi(), n)
    for steps in (1, 1, 3, 25):
        for sim in (a, b):
            sim.step(2e-5, steps)
        assert a.collisionCount() == b.collisionCount()
        sa, sb = a.state(), b.state()
        for k in ("pos", "orient", "linMom", "angMom"):
            assert sa[k].tobytes() == sb[k].tobytes(), (steps, k)
    print(f"[watch list] {model.__name__} {n}: {a.collisionCount()} pairs", flush=True)
