"""A chirp table ends in the middle of its axis where every radix that reads it is even: no position of a
first stage's lower inputs, or of a last stage's lower outputs, lies beyond."""

import os
import shutil
import subprocess
import tempfile
from pathlib import Path

import pytest

ROOT = Path(__file__).resolve().parents[1]
HIPCC = os.environ.get("HIPCC", "/opt/rocm/bin/hipcc")

PROGRAM = r"""
#include "fft_device.hpp"
#include <cstdio>
using namespace rkfft;
template <int L> int check() {
    using P = Plan<L>;
    constexpr int SL = P::NSTAGE - 1, R0 = P::R0, RL = P::radix(SL);
    int bad = 0;
    for (int t = 0; t < P::T; ++t) {
        if (R0 % 2 == 0)
            for (int r = 0; r < R0 / 2; ++r) bad += 2 * (t + r * P::T) >= L;   // loads, staged stores
        if (RL % 2 == 0)
            for (int q = 0; q < P::q(SL); ++q)
                for (int r = 0; r < RL / 2; ++r)
                    if (stage_valid<L, SL>(t, q)) bad += 2 * stage_out_pos<L, SL>(t, q * RL + r) >= L;
    }
    if (bad) std::printf("L=%d: %d positions\n", L, bad);
    return bad;
}
template <int... L> int all() { return (check<L>() + ...); }
int main() {
    return all<8, 12, 16, 20, 24, 32, 40, 48, 64, 80, 96, 128, 160, 192, 240, 256, 320, 384, 512, 640, 768, 1024, 1280,
               1536, 2048, 2560, 3072, 4096, 5120, 6144, 8192>() != 0;
}
"""


@pytest.mark.skipif(not Path(HIPCC).exists(), reason="hipcc not available")
def test_lower_halves():
    tmp = Path(tempfile.mkdtemp(prefix="rk_chirp_"))
    try:
        (tmp / "check.hip").write_text(PROGRAM)
        r = subprocess.run([HIPCC, "--offload-arch=gfx950", "--offload-host-only", "-O1", "-std=c++17",
                            f"-I{ROOT / 'reikna_amd' / 'csrc'}", str(tmp / "check.hip"), "-o", str(tmp / "check")],
                           capture_output=True, text=True, timeout=300)
        assert r.returncode == 0, r.stderr[-4000:]
        run = subprocess.run([str(tmp / "check")], capture_output=True, text=True, timeout=60)
        assert run.returncode == 0, run.stdout
    finally:
        shutil.rmtree(tmp, ignore_errors=True)
