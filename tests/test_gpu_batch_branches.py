"""Batches whose degree groups are parallel branches of the step graphs against the same runs
advanced alone: the same bits over several replays, with calls of long and of short graphs
(branches and in turn) between each other and with other work on the device in between."""
import numpy as np
import pytest

import self_amd

pytestmark = pytest.mark.gpu


def _model(kind, N, nx, ny, seed):
    mesh = self_amd.Mesh2D.structured(nx, ny, bcid=self_amd.BC_NONORMALFLOW)
    geom = self_amd.SEMQuad(self_amd.Lagrange(N, self_amd.GAUSS, N, self_amd.GAUSS), mesh)
    m = {"euler": self_amd.CompressibleIdealGas2D, "sw": self_amd.ShallowWater,
         "lsw": self_amd.LinearShallowWater}[kind](mesh, geom)
    s = 0.01 * np.random.default_rng(seed).standard_normal(m.shape)
    s[:, 2] += 1.0
    if kind == "euler":
        s[:, 3] += 2.5
    if kind == "lsw":
        m.SetBathymetry(1.0)
    m.SetSolution(s)
    return m


@pytest.mark.parametrize("kind,meshes,calls", [
    ("sw", [(3, 5, 4), (5, 3, 3), (7, 2, 3), (3, 1, 1)], (8, 8, 3, 16, 25)),  # by step count
    ("lsw", [(N, N, 2) for N in range(1, 8)], (9, 8, 1)),  # a branch per degree
    ("euler", [(4, 3, 3), (6, 70, 80), (4, 5, 1)], (2, 1, 3, 2)),  # two groups, by nodes x steps
    ("sw", [(5, 9, 9), (7, 130, 80)], (1, 1, 2)),  # from one step on
    ("sw", [(3, 2, 2), (7, 2, 2)], (8, 2)),  # two small groups: in turn
])
def test_branches_equal_separate_runs(kind, meshes, calls):
    dts = [1e-5 * (1 + k) for k in range(len(meshes))]
    batched = [_model(kind, *mesh, seed=k) for k, mesh in enumerate(meshes)]
    alone = [_model(kind, *mesh, seed=k) for k, mesh in enumerate(meshes)]
    batch = self_amd.Batch(batched, dts)
    for n in calls:
        batch.ForwardStep(n)
        for m, dt in zip(alone, dts):
            m.ForwardStep(n, dt)
        batch.scatter()
        for a, b in zip(alone, batched):
            np.testing.assert_array_equal(b.solution, a.solution)
            assert np.isfinite(a.solution).all()
