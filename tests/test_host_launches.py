"""What the library asks of the HIP runtime, seen by a runtime of two devices without a GPU
(fake_hip.c) that takes the place of libamdhip64 in a child process: the devices that work is
launched on, the sizes of grids."""
import os
import subprocess
import sys
import textwrap

import pytest

HERE = os.path.dirname(os.path.abspath(__file__))

PRELUDE = """
import ctypes, sys
fake = ctypes.CDLL(sys.argv[1], ctypes.RTLD_GLOBAL)  # found by its soname when the library is loaded
fake.fake_log.restype = ctypes.c_char_p
import numpy as np
import self_amd
from self_amd import call
from tests import cases

def log():
    lines = fake.fake_log().decode().splitlines()
    fake.fake_log_clear()
    return lines

def model(kind, N, nx, ny):
    return cases.Case(kind, N, nx, ny, periodic=True, metrics="affine").gpu_model()[0]

log()
"""


@pytest.fixture(scope="module")
def run(tmp_path_factory):
    lib = str(tmp_path_factory.mktemp("hip") / "libamdhip64.so.7")
    subprocess.run(["gcc", "-O1", "-shared", "-fPIC", "-Wall", "-Wl,-soname,libamdhip64.so.7", "-o", lib,
                    os.path.join(HERE, "fake_hip.c")], check=True)

    def child(code):
        out = subprocess.run([sys.executable, "-c", PRELUDE + textwrap.dedent(code), lib], cwd=os.path.dirname(HERE),
                             capture_output=True, text=True, timeout=100)
        assert out.returncode == 0, out.stdout + out.stderr
    return child


def test_batch_works_on_its_own_device_whatever_the_current_one(run):
    run("""
    models = [model("sw", N, 8, 8) for N in (3, 5, 7)]
    batch = self_amd.Batch(models, [1e-4] * 3)
    log()
    fake.hipSetDevice(1)
    batch.ForwardStep(64)   # groups as branches: streams of their own
    batch.scatter()
    lines = log()
    assert any(l.startswith("stream") for l in lines) and any("k_copy_list" in l for l in lines)
    elsewhere = [l for l in lines if not l.endswith("device 0")]
    assert not elsewhere, elsewhere[:3]
    current = ctypes.c_int()
    fake.hipGetDevice(ctypes.byref(current))
    assert current.value == 1
    """)


def test_projection_grids_stay_within_the_runtime_limit(run):
    run("""
    a = self_amd.DeviceArray((8,))
    for nyc, kernel in ((4095, "k_project"), (4096, "k_project_values"), (4097, "k_project_values")):
        call("selfamd_project_l2_structured_2d", a.ptr, a.ptr, 7, 3, 4096, nyc, 1, 3, None)
        lines = log()
        assert len(lines) == 1 and f"{len(kernel)}{kernel}" in lines[0], lines  # as mangled
    """)


def test_projection_of_many_small_elements_goes_by_values(run):
    run("""
    a = self_amd.DeviceArray((8,))
    for Nf, Nc, r, nv, n, kernel in ((1, 1, 1, 3, 512, "k_project_values"), (2, 2, 2, 1, 512, "k_project_values"),
                                     (2, 2, 2, 1, 60, "k_project"), (3, 3, 2, 3, 512, "k_project"),
                                     (1, 1, 4, 3, 512, "k_project_values"), (7, 3, 4, 3, 64, "k_project")):
        call("selfamd_project_l2_structured_2d", a.ptr, a.ptr, Nf, Nc, n, n, r, nv, None)
        lines = log()
        assert len(lines) == 1 and f"{len(kernel)}{kernel}" in lines[0], (Nf, Nc, r, nv, n, lines)
    """)


def test_networks_of_very_many_rows_have_grids(run):
    run("""
    for rows, kernel in ((1 << 26, "k_mlp_rows"), (1 << 27, "k_gemm")):
        net = self_amd.MLP(1, 1, 1, rows)
        a = self_amd.DeviceArray((rows, 1), np.float32)
        b = self_amd.DeviceArray((rows, 1), np.float32)
        log()
        call("selfamd_mlp_loss_grad", net._h, a.ptr, b.ptr, rows, None, None)
        lines = log()
        assert lines and f"{len(kernel)}{kernel}" in lines[0], lines[:3]
    """)


def test_small_models_that_step_together_keep_to_graphs(run):
    run("""
    def routes(models, wait):
        \"\"\"How each model's call of a round is launched.\"\"\"
        out = []
        for m in models:
            log()
            call("selfamd_model2d_forward_step", m._h, 4, 1e-4)
            lines = [l.split()[0] for l in log()]
            out.append("R" if "cooperative" in lines else "G" if "graph" in lines else "?")
            if wait:
                call("selfamd_model2d_synchronize", m._h)
        for m in models:
            call("selfamd_model2d_synchronize", m._h)
        return "".join(out)

    a, b, c = (model("lsw", 3, 9, 9) for _ in range(3))
    assert routes([a, b], False) == "RR" and routes([a, b], False) == "RR"  # two: one after the other
    assert routes([a, b, c], False) == "RRG"                                # a third joins
    assert routes([a, b, c], False) == "GGG" and routes([a, b, c], False) == "GGG"
    assert routes([a, b, c], True) == "GGR"                                 # waited for each time from here on
    assert routes([a, b, c], True) == "RRR"
    assert routes([a], False) == "R"
    big = [model("lsw", 3, 66, 66) for _ in range(3)]                       # 1,089 blocks of a wavefront
    assert routes(big, False) == "RRR" and routes(big, False) == "RRR"
    del b, c
    assert routes([a], False) == "R"
    """)


def test_launches_that_fill_the_device_are_short(run):
    run("""
    for n, steps, launches in ((9, 4096, 1), (9, 4097, 2), (66, 512, 1), (66, 1025, 3)):
        m = model("lsw", 3, n, n)
        log()
        call("selfamd_model2d_forward_step", m._h, steps, 1e-4)
        assert sum(l.startswith("cooperative") for l in log()) == launches, (n, steps)
        call("selfamd_model2d_synchronize", m._h)
    """)


def test_tiles_of_small_meshes_are_tuned_on_stage_launches(run):
    run("""
    from self_amd import autotune
    m = model("sw", 7, 8, 8)
    type(m).solution = property(lambda self: np.ones(self.shape))  # no kernel has stored one
    autotune._model = lambda kind, N, nx: ((lambda: model("sw", 7, 8, 8)), 1e-4)
    m.ForwardStep(4, 1e-4)
    assert any(l.startswith("cooperative") for l in log())
    autotune.tune(7, 8, steps=4, warmup=3, repeats=2)
    assert not any(l.startswith("cooperative") for l in log())
    m.SetStageLaunches()
    m.ForwardStep(4, 1e-4)
    assert not any(l.startswith("cooperative") for l in log())
    m.SetStageLaunches(False)
    m.ForwardStep(4, 1e-4)
    assert any(l.startswith("cooperative") for l in log())
    """)
