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


CHAINS = """
import numpy
from reikna_amd import ArrayMetadata, _lib
from reikna_amd.fft import NativeFftPlan
for n in (65521, 2**18):
    meta = ArrayMetadata((33, n), numpy.complex128)
    print(max(p.L for p in NativeFftPlan(meta, meta, (1,), _lib.RK_FFT_DRY_RUN).passes))
"""


# 65521 points: M = 2^17, two passes of up to 512 points or three of up to 64
@pytest.mark.parametrize("limit,longest", [(None, [64, 512]), ("512", [512, 512]), ("511", [64, 64]), ("256", [64, 64]),
                                           ("32", [32, 32])])
def test_factor_max_bounds_every_chain(limit, longest):
    """RK_FACTOR_MAX, also where it is one of the planner's own limits."""
    env = {k: v for k, v in os.environ.items() if k != "RK_FACTOR_MAX"}
    r = subprocess.run([sys.executable, "-c", CHAINS], cwd=ROOT, env={**env, **({"RK_FACTOR_MAX": limit} if limit else {})},
                       capture_output=True, text=True, timeout=120)
    assert r.returncode == 0, r.stderr[-2000:]
    assert [int(x) for x in r.stdout.split()] == longest
