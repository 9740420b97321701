"""Short-row tiles (both sides FLAT) leave registers for as many work-groups per CU as their LDS does."""

import os
import re
import shutil
import subprocess
import tempfile
from pathlib import Path

import pytest

from reikna_amd.csrc import build

ROOT = Path(__file__).resolve().parents[1]
HIPCC = os.environ.get("HIPCC", "/opt/rocm/bin/hipcc")


@pytest.mark.skipif(not Path(HIPCC).exists(), reason="hipcc not available")
@pytest.mark.parametrize("length", [24, 48])
def test_registers(length):
    c = build.tile_c_row(length)
    v = build.VAR_PLAIN | build.VAR_MODE_FF
    threads = c * build.threads_per_instance(length)
    assert threads <= 256
    tmp = Path(tempfile.mkdtemp(prefix="rk_flat_"))
    try:
        (tmp / "k.hip").write_text(
            f'#include "fft_device.hpp"\nextern "C" __global__ void __launch_bounds__({threads}) '
            f"k(rk_pass_args a) {{ rkfft::fft_pass_entry<{length}, {c}, {v}>(a); }}\n")
        r = subprocess.run([HIPCC, "-x", "hip", "--offload-arch=gfx950", "--offload-device-only", "-S", *build.COMMON_FLAGS,
                            *build.DEVICE_FLAGS, f"-I{build.HERE}", f"-I{ROOT / 'include'}", str(tmp / "k.hip"), "-o",
                            str(tmp / "k.s")], capture_output=True, text=True, timeout=300)
        assert r.returncode == 0, r.stderr[-4000:]
        text = (tmp / "k.s").read_text()
    finally:
        shutil.rmtree(tmp, ignore_errors=True)
    vgprs, lds = (int(re.search(rf"; {k}:?\s+(\d+)", text).group(1)) for k in ("TotalNumVgprs", "LDSByteSize"))
    # four waves per work-group, one per SIMD of 512 registers, allocated in eights
    work_groups = min(8, 512 // ((vgprs + 7) // 8 * 8))
    assert work_groups >= min(8, 160 * 1024 // lds), (vgprs, lds)
