"""The steps with a voxel's link directions split over the waves of a workgroup, bit for bit:
k_step_fp64_ends against the split FP64 step, k_step_mixed_ends (mixed and FP64 fused) against
k_step_mixed, which a pinned launch configuration selects: every size at which its tiling or the
rule that picks it changes, and its own machinery (divergence, idle robots, contacts, ramps, the
volumetric terms) in both of its forms."""
import numpy as np
import pytest

import backends as B
from voxelyze_amd import workloads as W

TILE, WIDE = 64, 16384   # voxels of a tile; of the widest form


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
@pytest.mark.parametrize("nv", [1, TILE - 1, TILE, TILE + 1, WIDE, WIDE + 1, 294912, 294913])
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
@pytest.mark.parametrize("nu", [0.0, 0.3])
def test_diverging_and_idle_robots(side, actuated, nu):
    print(f"[ends] robots beside a {side}^3 block, actuated {actuated}, Poisson's ratio {nu}", flush=True)
    sims = []
    for path in (0, 1):
        sim = B.maker(B.product_abi(), path)(0.005)
        mats = W.robot_materials(sim)
        for m in mats:
            m.setPoissonsRatio(nu)
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
    assert [b.robotRecommendedTimeStep(r) for r in range(4)] == list(dt)
    dt[3] = 0.0
    for n in (7, 60, 60, 1):
        da, db = a.robotStep(n, dt), b.robotStep(n, dt)
        assert np.array_equal(da, db)
    assert da[2] < 1 or a.robotTime(2) < 60 * dt[2]
    assert [a.robotTime(r) for r in range(4)] == [b.robotTime(r) for r in range(4)]
    assert_same(a, b, "robots")
    assert [a.voxel(i).temperature() for i in (0, 30, f, f + 9)] == [b.voxel(i).temperature() for i in (0, 30, f, f + 9)]


MIXED, FUSED64 = 1, 2


def same_bits_pinned(build, precision, run, what):
    """the form the size picks, and the per-voxel kernel by a pinned launch configuration"""
    a, b = build(), build()
    for sim in (a, b):
        sim.setPrecision(precision)
    assert b.abi.set_launch_config(b.handle, 0, 64, 0) == 1
    ra, rb = run(a), run(b)
    assert np.array_equal(ra, rb), what
    assert_same(a, b, what)


@pytest.mark.gpu
@pytest.mark.parametrize("precision,nv", [(MIXED, n) for n in (1, TILE + 1, WIDE, WIDE + 1, 368640, 368641)] +
                         [(FUSED64, n) for n in (TILE - 1, WIDE, WIDE + 1, 131072, 131073)])
def test_mixed_sizes_at_the_edges(precision, nv):
    print(f"[ends] precision {precision}, {nv} voxels", flush=True)
    build = lambda: lattice(0, nv)  # noqa: E731

    def run(sim):
        dt = sim.recommendedTimeStep()
        return [sim.step(dt, n) for n in (1, 5, 4)]
    same_bits_pinned(build, precision, run, f"{nv} voxels")


@pytest.mark.gpu
@pytest.mark.parametrize("precision", [MIXED, FUSED64])
@pytest.mark.parametrize("nv", [1000, WIDE + 500])
@pytest.mark.parametrize("model", ["bilinear", "contacts and ramps", "moduli"])
def test_mixed_options_in_both_forms(model, nv, precision):
    print(f"[ends] {model}, {nv} voxels, precision {precision}", flush=True)

    def build():
        sim = lattice(0, nv, bilinear=model == "bilinear")
        v = [sim.voxel(i).external() for i in (0, 5, 9, nv - 1)]
        v[0].setFixedAll()
        v[1].setFixed(1 | 16)
        v[2].setForce(0.0, 0.02, 0.5)
        if model == "contacts and ramps":
            sim.enableCollisions(True)
            v[3].setDisplacementRamp((0.0, 0.0, 0.0), (0.0, 0.0, -3.0))
        if model == "moduli":
            sim.setModuli(np.linspace(5e5, 2e6, nv))
        return sim

    def run(sim):
        dt = 0.3 * sim.recommendedTimeStep()
        return [sim.step(dt, n) for n in (1, 90, 40)]
    same_bits_pinned(build, precision, run, model)


@pytest.mark.gpu
@pytest.mark.parametrize("precision", [MIXED, FUSED64])
@pytest.mark.parametrize("side", [6, 26])
def test_mixed_diverging_and_idle_robots(side, precision):
    print(f"[ends] robots beside a {side}^3 block, precision {precision}", flush=True)

    def build():
        sim = B.maker(B.product_abi(), 0)(0.005)
        mats = W.robot_materials(sim)
        sim.setGravity(1.0)
        sim.enableFloor(True)
        for r, (n, mat) in enumerate(((3, 2), (side, 3), (4, 0), (3, 1))):
            if r:
                sim.addRobot()
            g = np.arange(n ** 3)
            sim.setVoxels(np.full(n ** 3, mats[mat].index, np.int32), np.stack([g % n, (g // n) % n, g // n ** 2], 1))
        sim.setActuation(True, 0.0, 20.0, 2.0)
        sim.setPhases(np.linspace(0.0, 6.0, sim.voxelCount()))
        f, _ = sim.robotVoxels(2)
        sim.voxel(f).external().setForce(1e4, 0.0, 0.0)
        return sim

    def run(sim):
        dt = np.array([sim.robotRecommendedTimeStep(r) for r in range(4)], np.float32)
        dt[3] = 0.0
        done = [sim.robotStep(n, dt) for n in (7, 60, 1)]
        return np.array(done + [[sim.robotTime(r) for r in range(4)], [sim.voxel(i).temperature() for i in (0, 30, 40, 60)]])
    same_bits_pinned(build, precision, run, "robots")


@pytest.mark.gpu
@pytest.mark.parametrize("nv", [262144, 262145, 524288])
def test_mixed_sizes_where_the_cached_kernel_starts_and_ends(nv):
    test_mixed_sizes_at_the_edges(MIXED, nv)


@pytest.mark.gpu
@pytest.mark.parametrize("moduli", [False, True])
def test_mixed_step_past_the_caches(moduli):
    """one voxel more than the cached kernel takes: a body stepped among them as it is alone"""
    small, big = 300, 524289 - 300
    both, alone = lattice(0, big), lattice(0, small)
    both.addRobot()
    n = 7
    s = np.arange(small)
    ijk = np.stack([s % n, (s // n) % n, s // n ** 2], 1)
    mat = (s % 3 == 0).astype(np.int32)
    both.setVoxels(mat, ijk)
    alone.addRobot()
    alone.setVoxels(mat, ijk)
    states = []
    for sim in (both, alone):
        sim.setPrecision(MIXED)
        if moduli:
            E = np.full(sim.voxelCount(), 1e6, np.float32)
            E[-small:] = 1e6 * (0.5 + W.uniform(7, np.arange(small, dtype=np.uint64)))
            sim.setModuli(E)
        sim.robotStep(9, np.full(2, 1e-5, np.float32))
        states.append(sim.state(sim.voxelCount() - small, small))
    for k, v in states[0].items():
        assert v.tobytes() == states[1][k].tobytes(), k
