"""Reads of the voxels' state after steps.  A read of all of it is held for the reads after it: they give
the same bits as reads from the device, cost no round trip, and never outlive the state they were of."""
import ctypes as C
import time

import numpy as np
import pytest

import backends as B
from test_gpu_step_ends import lattice

CHUNK = 19200   # voxels packed at a time when every field is read
KEYS = ("pos", "orient", "linMom", "angMom", "flags")


def build(nv, precision=0):
    sim = lattice(0, nv)
    sim.setPrecision(precision)
    sim.step(1e-5, 3)
    return sim


def fields(sim, first, n, names):
    out = {k: np.zeros((n, w), np.uint32 if k == "flags" else np.float64) for k, w in zip(KEYS, (3, 4, 3, 3, 1)) if k in names}
    p = [C.cast(out[k].ctypes.data, C.POINTER(C.c_uint32 if k == "flags" else C.c_double)) if k in out else None for k in KEYS]
    sim.abi.voxel_get_state(sim.handle, first, n, *p)
    return out


@pytest.mark.gpu
@pytest.mark.parametrize("nv", [1, 300, CHUNK, CHUNK + 1, 2 * CHUNK + 700])
def test_ranges_of_a_held_read(nv):
    print(f"[reads] {nv} voxels", flush=True)
    a, b = build(nv), build(nv)
    quarter = (nv + 3) // 4
    first = (nv - quarter) // 2
    part = fields(a, first, quarter, KEYS[:4])   # enough of the population to be held
    check(a, b, nv)
    for k in part:
        assert part[k].tobytes() == fields(b, first, quarter, (k,))[k].tobytes(), k
    whole = a.state()   # takes its place
    check(a, b, nv)
    for k in KEYS:
        assert whole[k].tobytes() == fields(b, 0, nv, (k,))[k].tobytes(), k


def check(a, b, nv):
    at = sorted({0, nv // 2, max(0, min(nv, CHUNK) - 1), min(nv - 1, CHUNK), nv - 1})
    for f in at:
        for n in sorted({1, min(2, nv - f), max(1, (nv - f) // 2), nv - f}):
            for names in (KEYS[:1], KEYS[1:2], KEYS[2:], KEYS):
                x = fields(a, f, n, names)
                for k in names:   # single fields, and never a quarter of everything: from the device
                    y = fields(b, f, n, (k,))
                    assert x[k].tobytes() == y[k].tobytes(), (f, n, k)


MOVES = {
    "steps": lambda s: s.step(1e-5, 4),
    "robot steps": lambda s: s.robotStep(2, np.full(1, 1e-5, np.float32)),
    "a reset": lambda s: s.resetTime(),
    "a checkpoint": lambda s: s.checkpointRestore(2),
    "a static solve": lambda s: ([s.voxel(i).external().setFixedAll() for i in range(121)], s.doLinearSolve(1e-6)),
    "the floor": lambda s: s.enableFloor(False),
    "a voxel": lambda s: (s.setVoxel(s.addMaterial(1e6, 1000.0), 40, 40, 40), s.step(1e-5, 1)),
    "a rollout": lambda s: s.adjointRun(4, 2, np.full(1, 1e-5, np.float32)),
    "the precision": lambda s: (s.setPrecision(0), s.step(1e-5, 2)),
}


def block(precision):
    sim = B.maker(B.product_abi())(0.005)
    sim.addMaterial(1e6, 1000.0)
    sim.setGravity(1.0)
    sim.enableFloor(True)
    i = np.arange(11 * 11 * 12)
    sim.setVoxels(np.zeros(len(i), np.int32), np.stack([i % 11, (i // 11) % 11, i // 121], 1))
    sim.setPrecision(precision)
    sim.voxel(len(i) - 1).external().setForce(0.0, 0.01, 0.02)
    sim.step(1e-5, 3)
    return sim


@pytest.mark.gpu
@pytest.mark.parametrize("precision", [0, 1])
def test_a_held_read_does_not_outlive_its_state(precision):
    a, b = block(precision), block(precision)
    for sim in (a, b):
        sim.resetTime()
        sim.step(1e-5, 2)
        sim.checkpointSave(2)
        sim.step(1e-5, 2)
    for what, move in MOVES.items():
        if what == "a rollout" and precision == 0:   # refused
            continue
        before = a.state()
        move(a)
        move(b)
        n = a.voxelCount()
        for k in KEYS:
            y = fields(b, 0, n, (k,))[k]
            assert fields(a, 0, n, (k,))[k].tobytes() == y.tobytes(), (what, k)
        after = a.state()
        assert any(after[k].tobytes() != before[k].tobytes() for k in KEYS), what
        assert after["pos"].tobytes() == fields(b, 0, n, ("pos",))["pos"].tobytes(), what


@pytest.mark.gpu
def test_reads_after_a_whole_read_cost_no_round_trip():
    """one voxel's position: a launch and a wait (20 us) where nothing is held, a few bytes copied where
    something is; the bound is half"""
    sim = build(50000)
    out = np.zeros(3)
    p = C.cast(out.ctypes.data, C.POINTER(C.c_double))
    read = sim.abi.voxel_get_state

    def best():
        t = []
        for _ in range(20):
            x = time.perf_counter()
            for i in range(50):
                read(sim.handle, 900 * i, 1, p, None, None, None, None)
            t.append(time.perf_counter() - x)
        return min(t) / 50 * 1e6
    device = best()
    sim.state()
    held = best()
    print(f"[reads] one voxel's position: {device:.1f} us from the device, {held:.1f} us held")
    assert held < 0.5 * device
