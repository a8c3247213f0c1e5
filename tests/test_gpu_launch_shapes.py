"""The kernels with a voxel per lane (k_step_fp64, k_step_mixed), which models small enough for the form
that splits link directions over waves only run with a pinned launch shape: every shape and option against
a step that does not share their code, bit for bit.  And the shapes' tuning, above the sizes of that form."""
import ctypes as C

import numpy as np
import pytest

import backends as B
from test_gpu_step_ends import FUSED64, MIXED, assert_same, lattice
from voxelyze_amd import workloads as W

SHAPES = [(block, xcd) for xcd in (0, 1) for block in (256, 128, 64)]


def pin(sim, kernel, block, xcd):
    assert sim.abi.set_launch_config(sim.handle, kernel, block, xcd) == 1


def settled(sim, kernel):
    s = C.c_int(-1)
    assert sim.abi.launch_config(sim.handle, kernel, None, None, C.byref(s)) == 1
    return s.value


@pytest.mark.gpu
@pytest.mark.parametrize("precision", [0, MIXED, FUSED64])
def test_every_shape_gives_the_same_bits(precision):
    """FP64 against the split step, the others against the form with split link directions"""
    ref = lattice(1, 4601)
    ref.setPrecision(precision)
    dt = ref.recommendedTimeStep()
    ref.step(dt, 30)
    for block, xcd in SHAPES:
        sim = lattice(0, 4601)
        sim.setPrecision(precision)
        pin(sim, 0 if precision else 3, block, xcd)
        sim.step(dt, 30)
        assert_same(ref, sim, f"precision {precision}, block {block}, mapping {xcd}")


@pytest.mark.gpu
@pytest.mark.parametrize("shape", [(64, 0), (256, 1)])
@pytest.mark.parametrize("model", ["poisson", "bilinear", "contacts and ramps", "many materials"])
def test_options_of_the_voxel_per_lane_step(model, shape):
    sims = []
    for path in (0, 1):
        sim = lattice(path, 1000, nu=0.3 if model == "poisson" else 0.0, bilinear=model == "bilinear")
        v = [sim.voxel(i).external() for i in (0, 5, 9, 999)]
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
        if path == 0:
            pin(sim, 3, *shape)
        sims.append(sim)
    a, b = sims
    dt = 0.3 * a.recommendedTimeStep()
    for n in (1, 90, 40):
        assert a.step(dt, n) == b.step(dt, n)
    assert_same(a, b, model)


def population(path, nu, actuated, contacts):
    sim = B.maker(B.product_abi(), path)(0.005)
    mats = W.robot_materials(sim)
    for m in mats:
        m.setPoissonsRatio(nu)
    sim.setGravity(1.0)
    sim.enableFloor(True)
    for r, (n, mat) in enumerate(((3, 2), (6, 3), (4, 0), (3, 1))):
        if r:
            sim.addRobot()
        g = np.arange(n ** 3)
        sim.setVoxels(np.full(n ** 3, mats[mat].index, np.int32), np.stack([g % n, (g // n) % n, g // n ** 2], 1))
    if actuated:
        sim.setActuation(True, 0.0, 20.0, 2.0)
        sim.setPhases(np.linspace(0.0, 6.0, sim.voxelCount()))
    sim.enableCollisions(contacts)
    f, _ = sim.robotVoxels(2)
    sim.voxel(f).external().setForce(1e4, 0.0, 0.0)   # blows up inside the launch
    return sim, f


@pytest.mark.gpu
@pytest.mark.parametrize("pinned", [False, True])
@pytest.mark.parametrize("contacts", [False, True])
@pytest.mark.parametrize("actuated", [False, True])
@pytest.mark.parametrize("nu", [0.0, 0.3])
def test_diverging_and_idle_robots_in_both_forms(nu, actuated, contacts, pinned):
    (a, f), (b, _) = population(0, nu, actuated, contacts), population(1, nu, actuated, contacts)
    if pinned:
        pin(a, 3, 64, 0)
    dt = np.array([a.robotRecommendedTimeStep(r) for r in range(4)], np.float32)
    dt[3] = 0.0
    done = np.zeros(4, int)
    for n in (7, 60, 60, 1):
        da, db = a.robotStep(n, dt), b.robotStep(n, dt)
        assert np.array_equal(da, db)
        done += da
    assert done[2] < 128 and done[1] == 128
    assert [a.robotTime(r) for r in range(4)] == [b.robotTime(r) for r in range(4)]
    assert_same(a, b, "robots")
    at = (0, 30, f, f + 9, a.voxelCount() - 1)
    assert [a.voxel(i).temperature() for i in at] == [b.voxel(i).temperature() for i in at]


@pytest.mark.gpu
@pytest.mark.parametrize("pinned", [False, True])
@pytest.mark.parametrize("nu,actuated,precision", [(0.3, False, 0), (0.0, True, 0), (0.3, True, 0), (0.0, True, 1),
                                                   (0.0, True, 2)])
def test_halted_batches_take_back_temperatures_and_poisson_strains(nu, actuated, precision, pinned):
    """a cube falls several pitches onto a plate: its watch list goes stale inside the batches of one
    launch, whose skipped steps' swaps are taken back.  Against launches of one step each."""
    sims = []
    for _ in range(2):
        sim = B.maker(B.product_abi())(0.001)
        soft = sim.addMaterial(2e4, 1000.0)
        soft.setCollisionDamping(0.2)
        soft.setPoissonsRatio(nu)
        soft.setCte(0.001)
        for x in range(4):
            for y in range(4):
                sim.setVoxel(soft, x, y, 0).external().setFixedAll()
        for x in range(1, 3):
            for y in range(1, 3):
                for z in range(5, 8):
                    sim.setVoxel(soft, x, y, z)
        sim.setGravity(1.0)
        sim.enableCollisions(True)
        if actuated:
            sim.setActuation(True, 1.0, 20.0, 40.0)
            sim.setPhases(np.linspace(0.0, 6.0, sim.voxelCount()))
        sim.setPrecision(precision)
        sims.append(sim)
    a, b = sims
    if pinned:
        pin(a, 0 if precision else 3, 64, 0)
    dt = 0.4 * a.recommendedTimeStep()
    n = 3400
    z0 = a.state()["pos"][:, 2].max()
    assert a.step(dt, n) == (n, -1)
    fall = 0.0
    for k in range(n):
        b.step(dt, 1)
        if k % 50 == 0:
            fall = max(fall, z0 - b.positions()[:, 2].max())
    print(f"[halts] nu {nu}, actuated {actuated}, precision {precision}: top fell {fall / 0.001:.2f} pitch, "
          f"{a.collisionCount()} pairs")
    assert fall > 3.0 * 0.001 and a.collisionCount() == b.collisionCount()
    assert_same(a, b, "halted batches")
    assert [a.voxel(i).temperature() for i in range(20)] == [b.voxel(i).temperature() for i in range(20)]


@pytest.mark.gpu
@pytest.mark.parametrize("precision,nv", [(0, 294913), (MIXED, 262145), (MIXED, 524288), (FUSED64, 131073)])
def test_tuned_steps_above_the_split_forms_size(precision, nv):
    """the launch shapes' tuning, and k_step_mixed on either side of its cached sizes: a body stepped among
    the others as it is alone (in the form with split link directions)"""
    small = 300
    kernel = 0 if precision else 3
    both, alone = lattice(0, nv - small), lattice(0, small)
    s = np.arange(small)
    ijk = np.stack([s % 7, (s // 7) % 7, s // 49], 1)
    states = []
    for sim in (both, alone):
        sim.addRobot()
        sim.setVoxels((s % 3 == 0).astype(np.int32), ijk)
        sim.setPrecision(precision)
        sim.robotStep(3, np.full(2, 1e-5, np.float32))
        if sim is both:
            assert sim.voxelCount() == nv and settled(sim, kernel) == 0
        sim.robotStep(30, np.full(2, 1e-5, np.float32))
        assert settled(sim, kernel) == 1
        sim.robotStep(4, np.full(2, 1e-5, np.float32))
        states.append(sim.state(sim.voxelCount() - small, small))
    for k, v in states[0].items():
        assert v.tobytes() == states[1][k].tobytes(), k


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
