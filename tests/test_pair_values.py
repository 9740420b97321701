"""The in-register DFTs of pairs of instances: each half is, bit for bit, the DFT of one instance."""

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
#include <cmath>
#include <cstdio>
using namespace rkfft;
template <int R> int check(bool lower) {
    float2 a[R], b[R];
    cpair2 p[R];
    for (int n = 0; n < R; ++n) {
        const bool zero = lower && n >= R / 2;
        a[n] = zero ? make_float2(0, 0) : make_float2(std::cos(3.0 * n + 1), std::sin(5.0 * n * n));
        b[n] = zero ? make_float2(0, 0) : make_float2(std::sin(7.0 * n + 2), std::cos(2.0 * n * n));
        p[n].x = rk_v2<float>{a[n].x, b[n].x};
        p[n].y = rk_v2<float>{a[n].y, b[n].y};
    }
    if (lower) { dft_lower<R>(a); dft_lower<R>(b); dft_lower<R>(p); }
    else { dft<R>(a); dft<R>(b); dft<R>(p); }
    int bad = 0;
    for (int k = 0; k < R; ++k)
        bad += p[k].x.x != a[k].x || p[k].y.x != a[k].y || p[k].x.y != b[k].x || p[k].y.y != b[k].y;
    if (bad) std::printf("radix %d%s: %d of %d values differ\n", R, lower ? " lower" : "", bad, R);
    return bad;
}
template <int... R> int all(bool lower) { return (check<R>(lower) + ...); }
int main() { return all<2, 3, 4, 5, 6, 7, 8, 9, 10, 12, 15, 16>(false) + all<2, 4, 6, 8, 10, 12, 16>(true) != 0; }
"""


@pytest.mark.skipif(not Path(HIPCC).exists(), reason="hipcc not available")
def test_pair_dfts_equal_single_ones():
    tmp = Path(tempfile.mkdtemp(prefix="rk_pair_dft_"))
    try:
        (tmp / "check.hip").write_text(PROGRAM)
        r = subprocess.run([HIPCC, "--offload-arch=gfx950", "--offload-host-only", "-O1", "-std=c++17", "-ffp-contract=off",
                            f"-I{ROOT / 'reikna_amd' / 'csrc'}", str(tmp / "check.hip"), "-o", str(tmp / "check")],
                           capture_output=True, text=True, timeout=300)
        assert r.returncode == 0, r.stderr[-4000:]
        run = subprocess.run([str(tmp / "check")], capture_output=True, text=True, timeout=60)
        assert run.returncode == 0, run.stdout
    finally:
        shutil.rmtree(tmp, ignore_errors=True)
