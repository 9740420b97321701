"""Instances of at most 96 points and 16 threads: the 75-point plan and 32-instance column tiles."""

import numpy
import pytest

import oracle
from reikna_amd import Array, ArrayMetadata, _lib
from reikna_amd.csrc import build
from reikna_amd.fft import FFT, NativeFftPlan


def test_plans():
    assert build.radix_list(75) == [5, 5, 3]
    for n in (49, 63, 70, 75, 81, 90, 98, 100):
        widths = []
        for dtype in (numpy.complex64, numpy.complex128):
            meta = ArrayMetadata((n, 4096), dtype)
            widths.append(NativeFftPlan(meta, meta, (0,), _lib.RK_FFT_DRY_RUN).passes[0].C)
        assert widths == [32 if n in (49, 63, 70, 75, 90) else 16, 32 if n == 49 else 16], n
        assert build.tile_c_col(n) == widths[0]


@pytest.mark.gpu
@pytest.mark.parametrize("n", [63, 70, 75, 90])
def test_matches_oracle(queue, n):
    rng = numpy.random.default_rng(n)
    for shape, axis in [((n, w), 0) for w in (1, 31, 32, 33, 301)] + [((3, n, 47), 1)] + [((c, n), 1) for c in (1, 16, 17, 18, 301)]:
        data = (rng.standard_normal(shape) + 1j * rng.standard_normal(shape)).astype(numpy.complex64)
        a = Array.from_host(queue, data)
        out = Array.empty_like(queue.device, a)
        fftc = FFT(a, axes=(axis,)).compile(queue.device)
        for inverse, ref in ((0, oracle.fftn), (1, oracle.ifftn)):
            fftc(queue, out, a, inverse)
            assert oracle.rel_l2(out.get(queue), ref(data, (axis,))) <= oracle.tolerance(shape, (axis,)), (shape, inverse)
