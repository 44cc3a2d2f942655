"""Resident stepping (all stages of a ForwardStep call in one cooperative launch, meshes that fit
the device) against the same steps taken stage by stage by the stage kernel: the same bits, for
every degree and physics, both metric modes, partly filled last tiles, flipped and unpaired
connectivity, a call after a call, and the state it leaves for the stage kernel."""
import numpy as np
import pytest

import self_amd
from tests.cases import Case

pytestmark = pytest.mark.gpu

CASES = [
    ("lsw", 7, 10, 10, "wall", "affine"), ("lsw", 6, 5, 3, "open", "affine"), ("lsw", 2, 7, 5, "wall", "nodal"),
    ("lsw", 3, 33, 31, "wall", "affine"), ("sw", 1, 9, 7, "periodic", "affine"), ("sw", 2, 4, 3, "wall", "nodal"),
    ("sw", 3, 64, 64, "periodic", "affine"), ("sw", 4, 7, 7, "wall", "affine"), ("sw", 5, 11, 13, "periodic", "nodal"),
    ("sw", 6, 3, 2, "periodic", "nodal"), ("sw", 7, 1, 1, "wall", "affine"), ("sw", 7, 54, 55, "periodic", "affine"),
    ("euler", 1, 60, 60, "wall", "affine"), ("euler", 3, 5, 5, "open", "nodal"), ("euler", 4, 73, 61, "wall", "affine"),
    ("euler", 5, 4, 4, "periodic", "affine"), ("euler", 6, 2, 9, "open", "affine"), ("euler", 7, 6, 5, "wall", "nodal"),
]


def stages(m, n, dt):
    for _ in range(n):
        for st in range(3):
            m.Stage(st, dt)


def check(m, sol, dt):
    """Runs of 5, 1 and 4 steps from the same state, by calls and by stages."""
    m.SetSolution(sol)
    want = []
    for n in (5, 1, 4):
        stages(m, n, dt)
        want.append(m.solution)
    stages(m, 2, dt)
    after = m.solution
    m.SetSolution(sol)
    for n, w in zip((5, 1, 4), want):
        m.ForwardStep(n, dt)
        np.testing.assert_array_equal(m.solution, w)
    stages(m, 2, dt)  # the traces and lagged velocities left behind serve the stage kernel
    np.testing.assert_array_equal(m.solution, after)
    assert np.isfinite(after).all()


@pytest.mark.parametrize("kind,N,nx,ny,bc,metrics", CASES)
def test_resident_equals_stages(kind, N, nx, ny, bc, metrics):
    bcid = self_amd.BC_NONORMALFLOW if bc == "wall" else self_amd.BC_RADIATION
    c = Case(kind, N, nx, ny, periodic=bc == "periodic", bcid=bcid, metrics=metrics)
    m, _ = c.gpu_model()
    check(m, c.sol, c.dt(0.05))


def _model(mesh, N, nodal=False):
    geom = self_amd.SEMQuad(self_amd.Lagrange(N, self_amd.GAUSS, N, self_amd.GAUSS), mesh)
    m = self_amd.ShallowWater(mesh, geom)
    if nodal:
        m.SetNodalMetrics(True)
    m.SetTopography(0.05 * np.random.default_rng(1).random((mesh.nElem, N + 1, N + 1)))
    s = 0.01 * np.random.default_rng(2).standard_normal(m.shape)
    s[:, 2] += 1.0
    return m, s


@pytest.mark.parametrize("N", [3, 5, 7])
def test_flipped_sides(N):
    """The reference's Circle mesh: curved elements whose neighbours' faces run the other way."""
    import json
    import os
    with open(os.path.join(os.path.dirname(__file__), "golden", "hopr_circle.json")) as f:
        fx = json.load(f)
    mesh = self_amd.Mesh2D.from_hopr(
        fx["Ngeo"], np.array(fx["SideInfo"]["data"], np.int32).reshape(fx["SideInfo"]["shape"]),
        np.array(fx["NodeCoords"]["data"]).reshape(fx["NodeCoords"]["shape"]),
        np.array(fx["GlobalNodeIDs"]["data"], np.int32))
    mesh.ResetBoundaryConditionType(self_amd.BC_NONORMALFLOW)
    m, s = _model(mesh, N)
    check(m, s, 1e-5)


def test_unpaired_connectivity_runs_by_stages():
    """A side whose neighbour does not name it back cannot exchange traces inside a launch: such a
    mesh runs as before."""
    mesh = self_amd.Mesh2D.structured(6, 6, periodic=(True, True))
    mesh.sideInfo[0, 1, 2] = 9  # element 1 reads element 9's west side, which does not read it
    m, s = _model(mesh, 4)
    check(m, s, 1e-5)
