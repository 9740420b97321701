"""Bluestein transforms use only the lower half of their axis on the chirp
sides, and bound no position of its first quarter: the planner's lengths keep
both true, and the shortest and longest rows of every M agree with the oracle."""

import numpy
import pytest

import oracle
from reikna_amd import Array, ArrayMetadata, _lib
from reikna_amd.fft import FFT, NativeFftPlan


def test_every_length_plans():
    for n in [*range(2, 1100), 2047, 2048, 4095, 4096, 4097, 8191, 8192, 65521, 65536, 98304]:
        meta = ArrayMetadata((3, n), numpy.complex64)
        for flags in (_lib.RK_FFT_FORCE_BLUESTEIN, _lib.RK_FFT_FORCE_BLUESTEIN | _lib.RK_FFT_FORCE_MULTIPASS):
            passes = NativeFftPlan(meta, meta, (1,), flags | _lib.RK_FFT_DRY_RUN).passes
            m = passes[0].axis_len
            assert 2 * n - 1 <= m < 4 * n and (m % 2 or 2 * n <= m)


# rows of N points: N = M/2, M/2 - 1 and the smallest N that takes M
EDGES = [(64, 32), (64, 31), (64, 25), (96, 48), (96, 41), (160, 80), (160, 65), (2048, 1024), (2048, 1023), (2048, 769),
         (8192, 4096), (8192, 3073), (16384, 8191), (20480, 8193), (131072, 65536), (131072, 49153)]


@pytest.mark.gpu
@pytest.mark.parametrize("m,n", EDGES, ids=str)
@pytest.mark.parametrize("layout", ["rows", "columns"])
def test_edges_match_oracle(queue, m, n, layout):
    shape, axis = ((5, n), 1) if layout == "rows" else ((n, 37 if n < 5000 else 18), 0)
    rng = numpy.random.default_rng(n)
    data = (rng.standard_normal(shape) + 1j * rng.standard_normal(shape)).astype(numpy.complex64)
    a = Array.from_host(queue, data)
    out = Array.empty_like(queue.device, a)
    fft = FFT(a, axes=(axis,), flags=_lib.RK_FFT_FORCE_BLUESTEIN)
    fftc = fft.compile(queue.device)
    assert fft.native_plan.passes[0].axis_len == m
    fftc(queue, out, a, 0)
    assert oracle.rel_l2(out.get(queue), oracle.fftn(data, (axis,))) <= oracle.tolerance(shape, (axis,))
    fftc(queue, out, a, 1)
    assert oracle.rel_l2(out.get(queue), oracle.ifftn(data, (axis,))) <= oracle.tolerance(shape, (axis,))
