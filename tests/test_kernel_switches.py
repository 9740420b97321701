"""The experiment switches of the planner: kernels of the catalogue's lengths outside the catalogue
(RK_HALF, RK_WAVE, RK_PIPE, RK_OCC) come from the run-time compiler."""

import os
import subprocess
import sys
from pathlib import Path

import pytest

ROOT = Path(__file__).resolve().parents[1]

PROGRAM = """
import numpy
from reikna_amd import ArrayMetadata, _lib
from reikna_amd.fft import NativeFftPlan
for shape, axes in (((16, 1024), (1,)), ((64, 2**20), (1,)), ((256, 256, 256), (0, 1, 2)), ((4096, 997), (1,)),
                    ((4096, 12288), (1,)), ((100, 1080), (1,)), ((16, 1080, 1920), (1, 2))):
    for dtype in (numpy.complex64, numpy.complex128):
        meta = ArrayMetadata(shape, dtype)
        plan = NativeFftPlan(meta, meta, axes, _lib.RK_FFT_DRY_RUN)
        print(shape, [(p.L, p.wave, p.pipe, p.occ, p.pair) for p in plan.passes])
"""


@pytest.mark.parametrize("switch", ["RK_HALF=1", "RK_WAVE=1", "RK_PIPE=1", "RK_OCC=64", "RK_OCC=0", "RK_FIXED_MODES=0",
                                    "RK_PAIR=0"])
def test_switches_leave_every_plan_possible(switch):
    name, value = switch.split("=")
    r = subprocess.run([sys.executable, "-c", PROGRAM], cwd=ROOT, env={**os.environ, name: value},
                       capture_output=True, text=True, timeout=120)
    assert r.returncode == 0, r.stderr[-2000:]
    if name == "RK_WAVE":
        assert "True" in r.stdout
