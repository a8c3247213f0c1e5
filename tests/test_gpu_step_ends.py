"""The FP64 step with a voxel's link directions split over the waves of a workgroup
(k_step_fp64_ends) against the split FP64 step, bit for bit: every size at which its tiling or the
rule that picks it changes, and its own machinery (divergence, idle robots, contacts, ramps, the
volumetric terms) in both of its forms."""
import numpy as np
import pytest

import backends as B
from voxelyze_amd import workloads as W

TILE, WIDE, LARGEST = 64, 16384, 294912   # voxels of a tile; of the widest form; of the kernel at all


def lattice(path, nv, nu=0.0, bilinear=False):
    """the first nv sites of a two-material lattice with holes, lying on the floor"""
    sim = B.maker(B.product_abi(), path)(0.005)
    mats = [sim.addMaterial(1e6, 1000.0), sim.addMaterial(1e7, 1500.0)]
    for m in mats:
        m.setStaticFriction(1.0)
        m.setKineticFriction(0.5)
        m.setPoissonsRatio(nu)
    if bilinear:
        mats[0].setModelBilinear(1e6, 1e5, 5e3)
    sim.setGravity(1.0)
    sim.enableFloor(True)
    side = 1
    while 0.85 * side ** 3 < nv:
        side += 1
    s = np.arange(side ** 3, dtype=np.uint64)
    s = s[W.uniform(4, 2 * s) < 0.9][:nv].astype(np.int64)
    assert len(s) == nv
    mat = (W.uniform(4, 2 * s.astype(np.uint64) + np.uint64(1)) < 0.3).astype(np.int32)
    sim.setVoxels(mat, np.stack([s % side, (s // side) % side, s // side ** 2], 1))
    return sim


def assert_same(a, b, what):
    for x, y in ((a.state(), b.state()), (a.link_state(), b.link_state())):
        bad = [k for k in x if x[k].tobytes() != y[k].tobytes()]
        assert not bad, f"{what}: differs in {bad}"


@pytest.mark.gpu
@pytest.mark.parametrize("nv", [1, TILE - 1, TILE, TILE + 1, WIDE, WIDE + 1, LARGEST, LARGEST + 1])
def test_sizes_at_the_edges(nv):
    print(f"[ends] {nv} voxels", flush=True)
    a, b = lattice(0, nv), lattice(1, nv)
    dt = a.recommendedTimeStep()
    for n in (1, 5, 4):
        assert a.step(dt, n) == b.step(dt, n)
    assert_same(a, b, f"{nv} voxels")


@pytest.mark.gpu
@pytest.mark.parametrize("nv", [1000, WIDE + 500])
@pytest.mark.parametrize("model", ["poisson", "bilinear", "contacts and ramps", "many materials"])
def test_options_in_both_forms(model, nv):
    print(f"[ends] {model}, {nv} voxels", flush=True)
    sims = []
    for path in (0, 1):
        sim = lattice(path, nv, nu=0.3 if model == "poisson" else 0.0, bilinear=model == "bilinear")
        v = [sim.voxel(i).external() for i in (0, 5, 9, nv - 1)]
        v[0].setFixedAll()
        v[1].setFixed(1 | 16)
        v[2].setForce(0.0, 0.02, 0.5)
        v[2].setMoment(1e-4, 0.0, 0.0)
        if model == "contacts and ramps":
            sim.enableCollisions(True)
            v[3].setDisplacementRamp((0.0, 0.0, 0.0), (0.0, 0.0, -3.0))
        if model == "many materials":   # more than the tables in LDS hold
            for k in range(40):
                sim.setVoxel(sim.addMaterial(1e6 + 1e4 * k, 1000.0), 100 + k, 0, 0)
        sims.append(sim)
    a, b = sims
    dt = 0.3 * a.recommendedTimeStep()
    assert dt == 0.3 * b.recommendedTimeStep()
    for n in (1, 90, 40):
        assert a.step(dt, n) == b.step(dt, n)
    assert_same(a, b, model)


@pytest.mark.gpu
@pytest.mark.parametrize("side", [6, 26])
@pytest.mark.parametrize("actuated", [False, True])
def test_diverging_and_idle_robots(side, actuated):
    print(f"[ends] robots beside a {side}^3 block, actuated {actuated}", flush=True)
    sims = []
    for path in (0, 1):
        sim = B.maker(B.product_abi(), path)(0.005)
        mats = W.robot_materials(sim)
        sim.setGravity(1.0)
        sim.enableFloor(True)
        for r, (n, mat) in enumerate(((3, 2), (side, 3), (4, 0), (3, 1))):
            if r:
                sim.addRobot()
            g = np.arange(n ** 3)
            sim.setVoxels(np.full(n ** 3, mats[mat].index, np.int32),
                          np.stack([g % n, (g // n) % n, g // n ** 2], 1))
        if actuated:
            sim.setActuation(True, 0.0, 20.0, 2.0)
            sim.setPhases(np.linspace(0.0, 6.0, sim.voxelCount()))
        f, _ = sim.robotVoxels(2)
        sim.voxel(f).external().setForce(1e4, 0.0, 0.0)   # blows up inside the launch
        sims.append(sim)
    a, b = sims
    dt = np.array([a.robotRecommendedTimeStep(r) for r in range(4)], np.float32)
    dt[3] = 0.0
    for n in (7, 60, 1):
        da, db = a.robotStep(n, dt), b.robotStep(n, dt)
        assert np.array_equal(da, db)
    assert da[2] < 1 or a.robotTime(2) < 60 * dt[2]
    assert [a.robotTime(r) for r in range(4)] == [b.robotTime(r) for r in range(4)]
    assert_same(a, b, "robots")
    assert [a.voxel(i).temperature() for i in (0, 30, f, f + 9)] == [b.voxel(i).temperature() for i in (0, 30, f, f + 9)]
