"""The reverse pass lists the links of each axis once and gives its lanes the listed ones only.
Its shares are compared over the shapes at which a list's length meets a workgroup's (no link at
all, links along one axis only, one link less or more than a workgroup holds, axes of unequal
length, holes): a link's derivatives do not depend on which lane forms them, so every robot's
gradient in a batch has the bits it has alone, and so has a second pass over the same lists."""
import numpy as np
import pytest

from test_gpu_adjoint import build, weighted_loss
from voxelyze_amd import workloads as W


def line(axis, n):
    ijk = np.zeros((n, 3), np.int32)
    ijk[:, axis] = np.arange(n)
    return ijk


def holed(nx, ny, nz, keep, seed):
    s = np.arange(nx * ny * nz)
    s = s[W.uniform(seed, s.astype(np.uint64)) < keep]
    return np.stack([s % nx, (s // nx) % ny, s // (nx * ny)], 1).astype(np.int32)


BATCHES = {
    "no link": [line(0, 1), line(0, 1)],
    "one axis": [line(2, 257), line(2, 1)],
    "a workgroup's edges": [line(0, 256), line(0, 257), line(0, 258), line(1, 513), line(2, 2)],
    "unequal axes and holes": [holed(31, 7, 2, 0.6, 5), line(1, 300), holed(9, 9, 9, 0.3, 6), line(0, 1)],
}


@pytest.mark.gpu
@pytest.mark.parametrize("precision", [1, 2])
@pytest.mark.parametrize("name", list(BATCHES))
def test_gradient_of_a_robot_alone_and_in_a_batch(name, precision):
    shapes = [(ijk, np.arange(len(ijk)) % 3) for ijk in BATCHES[name]]
    batch = build(shapes, precision)
    n = batch.voxelCount()
    u = W.uniform(8, np.arange(5 * n, dtype=np.uint64))
    theta, phi, w = np.log(1e6) + 0.3 * (u[:n] - 0.5), 6.28 * u[n:2 * n], (u[2 * n:] - 0.5).reshape(n, 3)
    _, ge, gp = weighted_loss(batch, theta, phi, w, 12)
    again = batch.adjointBackward(w)
    assert np.array_equal(again[0], ge) and np.array_equal(again[1], gp)
    assert np.isfinite(ge).all() and np.isfinite(gp).all() and (n == 2 or np.any(gp != 0))
    for r, shape in enumerate(shapes):
        f, c = batch.robotVoxels(r)
        alone = build([shape], precision)
        _, e1, p1 = weighted_loss(alone, theta[f:f + c], phi[f:f + c], w[f:f + c], 12)
        assert np.array_equal(e1, ge[f:f + c]) and np.array_equal(p1, gp[f:f + c]), r
