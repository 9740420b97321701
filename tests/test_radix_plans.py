"""Radix plans: the kernels' and the build's lists agree and keep their limits,
and every in-register DFT matches the definition in double precision."""

import os
import shutil
import subprocess
import tempfile
from pathlib import Path

import numpy
import pytest

import oracle
from reikna_amd.csrc import build

ROOT = Path(__file__).resolve().parents[1]
HIPCC = os.environ.get("HIPCC", "/opt/rocm/bin/hipcc")

PROGRAM = r"""
#include "fft_device.hpp"
#include <cmath>
#include <cstdio>
using namespace rkfft;
template <int R> double error(bool lower) {
    double2 v[R], x[R];
    for (int n = 0; n < R; ++n) x[n] = v[n] = lower && n >= R / 2 ? make_double2(0, 0) : make_double2(std::cos(3.0 * n + 1), std::sin(5.0 * n * n));
    if (lower) dft_lower<R>(v); else dft<R>(v);
    double worst = 0;
    for (int k = 0; k < R; ++k) {
        double re = 0, im = 0;
        for (int n = 0; n < R; ++n) {
            const double a = -2 * M_PI * ((n * k) % R) / R, c = std::cos(a), s = std::sin(a);
            re += x[n].x * c - x[n].y * s;
            im += x[n].x * s + x[n].y * c;
        }
        worst = std::fmax(worst, std::hypot(v[k].x - re, v[k].y - im));
    }
    return worst;
}
int main() {
    double e = 0;
    e = std::fmax(e, error<2>(false)); e = std::fmax(e, error<3>(false)); e = std::fmax(e, error<4>(false));
    e = std::fmax(e, error<5>(false)); e = std::fmax(e, error<6>(false)); e = std::fmax(e, error<7>(false));
    e = std::fmax(e, error<8>(false)); e = std::fmax(e, error<9>(false)); e = std::fmax(e, error<10>(false));
    e = std::fmax(e, error<12>(false)); e = std::fmax(e, error<15>(false)); e = std::fmax(e, error<16>(false));
    e = std::fmax(e, error<2>(true)); e = std::fmax(e, error<4>(true)); e = std::fmax(e, error<6>(true));
    e = std::fmax(e, error<8>(true)); e = std::fmax(e, error<10>(true)); e = std::fmax(e, error<12>(true));
    e = std::fmax(e, error<16>(true));
    std::printf("dft %.17g\n", e);
    for (int L = 1; L <= 16384; ++L) {
        if (!is_supported_length(L)) continue;
        const RadixList r = make_radix_list(L);
        std::printf("%d", L);
        for (int k = 0; k < r.n; ++k) std::printf(" %d", r.r[k]);
        std::printf("\n");
    }
    return 0;
}
"""


@pytest.mark.skipif(not Path(HIPCC).exists(), reason="hipcc not available")
def test_plans_and_dfts():
    tmp = Path(tempfile.mkdtemp(prefix="rk_radix_"))
    try:
        (tmp / "check.hip").write_text(PROGRAM)
        r = subprocess.run([HIPCC, "--offload-arch=gfx950", "--offload-host-only", "-O1", "-std=c++17",
                            f"-I{ROOT / 'reikna_amd' / 'csrc'}", str(tmp / "check.hip"), "-o", str(tmp / "check")],
                           capture_output=True, text=True, timeout=300)
        assert r.returncode == 0, r.stderr[-4000:]
        out = subprocess.run([str(tmp / "check")], capture_output=True, text=True, timeout=60).stdout.splitlines()
    finally:
        shutil.rmtree(tmp, ignore_errors=True)
    assert float(out[0].split()[1]) < 16 * 16 * 2.3e-16   # 16 terms of size one, a few roundings each
    for line in out[1:]:
        length, *radices = map(int, line.split())
        assert numpy.prod(radices) == length
        assert radices == build.radix_list(length)
        t = length // radices[0]
        if radices != build.prime_power_list(length):
            assert t <= 1024 and (length > 4096 or t <= 256)
            assert all(-(-(length // r) // t) * r <= 20 for r in radices)
        if length in build.batch_lengths():
            assert t <= 256


@pytest.mark.gpu
@pytest.mark.parametrize("layout", ["rows", "columns"])
def test_lengths_of_composite_radices(queue, layout):
    """The catalogue's lengths, where their plans have idle threads or composite radices, and mixed ones."""
    from reikna_amd import Array
    from reikna_amd.fft import FFT

    for n in (6, 9, 10, 12, 15, 18, 21, 24, 45, 48, 63, 75, 80, 90, 96, 100, 105, 125, 160, 192, 225, 250, 320, 360, 384, 500,
              640, 720, 729, 768, 960, 1000, 1050, 1080, 1280, 1350, 1440, 1536, 1920, 2000, 2187, 2560, 3072, 4000, 4050):
        shape, axis = ((7, n), 1) if layout == "rows" else ((n, 37), 0)
        rng = numpy.random.default_rng(n)
        data = (rng.standard_normal(shape) + 1j * rng.standard_normal(shape)).astype(numpy.complex64)
        a = Array.from_host(queue, data)
        out = Array.empty_like(queue.device, a)
        fftc = FFT(a, axes=(axis,)).compile(queue.device)
        for inverse, ref in ((0, oracle.fftn), (1, oracle.ifftn)):
            fftc(queue, out, a, inverse)
            assert oracle.rel_l2(out.get(queue), ref(data, (axis,))) <= oracle.tolerance(shape, (axis,)), (n, inverse)
