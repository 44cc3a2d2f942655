"""Resident stepping of meshes that fill the device, with each of the instances that hold more
blocks, against the same steps taken by stage launches: the same bits, on both sides of what the
device holds and of the call length from which instances that spill are taken."""
import numpy as np
import pytest

import self_amd

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("kind,N,nx,ny,nodal", [
    ("sw", 7, 64, 64, False), ("sw", 7, 80, 64, True), ("sw", 7, 81, 64, False), ("sw", 3, 128, 128, True),
    ("sw", 3, 160, 128, False), ("sw", 5, 96, 80, True), ("sw", 6, 70, 73, False), ("lsw", 2, 160, 160, False),
    ("lsw", 4, 101, 101, True), ("lsw", 7, 73, 70, False), ("lsw", 1, 181, 181, False), ("euler", 7, 64, 48, False),
    ("euler", 7, 60, 59, True), ("euler", 2, 120, 120, False), ("euler", 4, 77, 79, False),
])
def test_full_device_equals_stages(kind, N, nx, ny, nodal):
    mesh = self_amd.Mesh2D.structured(nx, ny, bcid=self_amd.BC_NONORMALFLOW)
    geom = self_amd.SEMQuad(self_amd.Lagrange(N, self_amd.GAUSS, N, self_amd.GAUSS), mesh)
    m = {"euler": self_amd.CompressibleIdealGas2D, "sw": self_amd.ShallowWater,
         "lsw": self_amd.LinearShallowWater}[kind](mesh, geom)
    if nodal:
        m.SetNodalMetrics(True)
    rng = np.random.default_rng(N)
    s = 0.01 * rng.standard_normal(m.shape)
    s[:, 2] += 1.0
    if kind == "euler":
        s[:, 3] += 2.5
    if kind == "lsw":
        m.SetBathymetry(1.0)
    if kind == "sw":
        m.SetTopography(0.05 * rng.random((mesh.nElem, N + 1, N + 1)))
    dt, calls = 1e-5, (5, 1, 4, 6)
    m.SetSolution(s)
    want = []
    for n in calls:
        for _ in range(n):
            for st in range(3):
                m.Stage(st, dt)
        want.append(m.solution)
    m.SetSolution(s)
    for n, w in zip(calls, want):
        m.ForwardStep(n, dt)
        np.testing.assert_array_equal(m.solution, w)
    assert np.isfinite(want[-1]).all()
