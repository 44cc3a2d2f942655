"""Resident launches that need every place on the device while other streams' launches hold some: a
mesh of 4,096 blocks (SW N = 7, four wavefronts of 128 registers on each SIMD) beside a mesh that is
stepped one stage per launch, whose wavefronts of 96 registers leave gaps that a fourth does not fit.
Whether the launch goes in or is given up, every call ends and gives the bits of the stage kernel."""
import numpy as np
import pytest

import self_amd
from self_amd import call

pytestmark = pytest.mark.gpu


def model(nx, ny, seed):
    mesh = self_amd.Mesh2D.structured(nx, ny, periodic=(True, True))
    m = self_amd.ShallowWater(mesh, self_amd.SEMQuad(self_amd.Lagrange(7, self_amd.GAUSS, 7, self_amd.GAUSS), mesh))
    s = 0.01 * np.random.default_rng(seed).standard_normal(m.shape)
    s[:, 2] += 1.0
    m.SetSolution(s)
    return m, s


def test_full_device_launches_beside_stage_launches():
    dt, rounds, steps = 1e-6, 6, 10
    full, s = model(64, 64, 1)
    large, sl = model(128, 96, 2)
    for m in (full, large):
        for _ in range(rounds * steps):
            for st in range(3):
                m.Stage(st, dt)
        m.want = m.solution
    full.SetSolution(s)
    large.SetSolution(sl)
    for _ in range(rounds):
        call("selfamd_model2d_forward_step", large._h, steps, dt)
        call("selfamd_model2d_forward_step", full._h, steps, dt)
    np.testing.assert_array_equal(full.solution, full.want)
    np.testing.assert_array_equal(large.solution, large.want)
    # and waited for each time
    full.SetSolution(s)
    large.SetSolution(sl)
    for _ in range(rounds):
        call("selfamd_model2d_forward_step", large._h, steps, dt)
        full.ForwardStep(steps, dt)
    np.testing.assert_array_equal(full.solution, full.want)
    np.testing.assert_array_equal(large.solution, large.want)
