"""The linear solve where the rule that picks its kernels (one launch fewer up to 262,144 voxels)
and their block sizes change: a block on one side of each line and the same block with one fully
held voxel beside it, on the other side, have the same solution.  Both are solved to 1e-12 of the
load; the stiffness of these blocks has a condition number below 1e6, so the two may differ by
1e-6 of the largest displacement.  A solve repeated has to give the same bits."""
import numpy as np
import pytest

import backends as B


def solve(nv, beside):
    side = round(nv ** (1 / 3) + 0.5)
    s = np.arange(nv)
    ijk = np.stack([s % side, (s // side) % side, s // side ** 2], 1)
    if beside:
        ijk = np.concatenate([ijk, [[-5, 0, 0]]])
    sim = B.maker(B.product_abi())(0.005)
    m = sim.addMaterial(1e6, 1000.0)
    sim.setVoxels(np.full(len(ijk), m.index, np.int32), ijk)
    for i in np.nonzero(ijk[:, 2] == 0)[0]:
        sim.voxel(int(i)).external().setFixedAll()
    top = np.nonzero(ijk[:, 2] == ijk[:, 2].max())[0]
    for i in top:
        sim.voxel(int(i)).external().setForce(1e-2 / len(top), 1e-3 / len(top), -2e-3 / len(top))
    out = []
    for _ in range(2):
        assert sim.doLinearSolve(1e-12), sim.lastError()
        st = sim.state()
        out.append(np.concatenate([st["pos"][:nv] - ijk[:nv] * 0.005, st["orient"][:nv]], 1))
    assert out[0].tobytes() == out[1].tobytes()
    return out[0]


@pytest.mark.gpu
@pytest.mark.parametrize("nv", [64, 16384, 32768, 131072, 262144])
def test_both_sides_of_a_line_agree(nv):
    print(f"[linear] {nv} and {nv + 1} voxels", flush=True)
    a, b = solve(nv, False), solve(nv, True)
    d = np.abs(a[:, :3]).max()
    assert 1e-9 < d < 1e-2
    assert np.abs(a[:, :3] - b[:, :3]).max() < 1e-6 * d
    assert np.abs(a[:, 3:] - b[:, 3:]).max() < 1e-6
