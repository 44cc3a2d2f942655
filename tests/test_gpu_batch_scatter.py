"""Batch.scatter copies many arrays per launch: more arrays than one launch takes, with and
without lagged velocities, down to single elements, bit for bit against separate runs."""
import numpy as np
import pytest

import self_amd

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("kind,runs", [("euler", 60), ("sw", 45), ("lsw", 2)])
def test_scatter_many_small_runs(kind, runs):
    def model(k):
        N, nx, ny = 1 + k % 3, 1 + k % 4, 1 + k % 2
        mesh = self_amd.Mesh2D.structured(nx, ny, bcid=self_amd.BC_NONORMALFLOW)
        geom = self_amd.SEMQuad(self_amd.Lagrange(N, self_amd.GAUSS, N, self_amd.GAUSS), mesh)
        m = {"euler": self_amd.CompressibleIdealGas2D, "sw": self_amd.ShallowWater,
             "lsw": self_amd.LinearShallowWater}[kind](mesh, geom)
        s = 0.01 * np.random.default_rng(k).standard_normal(m.shape)
        s[:, 2] += 1.0
        if kind == "euler":
            s[:, 3] += 2.5
        if kind == "lsw":
            m.SetBathymetry(1.0)
        m.SetSolution(s)
        return m

    dts = [1e-3 / (1 + k % 5) for k in range(runs)]
    models = [model(k) for k in range(runs)]
    batch = self_amd.Batch(models, dts)
    batch.ForwardStep(3)
    batch.scatter()
    for k, m in enumerate(models):
        alone = model(k)
        alone.ForwardStep(3, dts[k])
        np.testing.assert_array_equal(m.solution, alone.solution)
        # the run continues from the copied traces and lagged velocities
        m.ForwardStep(2, dts[k])
        alone.ForwardStep(2, dts[k])
        np.testing.assert_array_equal(m.solution, alone.solution)
