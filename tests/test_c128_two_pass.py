"""complex128 chains of two passes with 512-point column tiles."""

import numpy
import pytest

from reikna_amd import Array, ArrayMetadata, _lib
from reikna_amd.fft import FFT, NativeFftPlan


def test_complex128_pass_lengths():
    def lengths(n):
        meta = ArrayMetadata((16, n), numpy.complex128)
        return [(p.L, p.C) for p in NativeFftPlan(meta, meta, (1,), _lib.RK_FFT_DRY_RUN).passes]

    assert lengths(2**18) == [(512, 8), (512, 8)]
    assert lengths(2**17) == [(512, 8), (256, 16)]
    assert [x for x, _ in lengths(2**19)] == [64, 128, 64]


@pytest.mark.gpu
@pytest.mark.parametrize("shape,inverse", [
    ((1, 2**17), 0), ((3, 2**18), 1), ((2, 384 * 512), 0), ((5, 500 * 512), 1), ((17, 2**18), 0),
], ids=str)
def test_complex128_two_pass_matches_numpy(queue, shape, inverse):
    rng = numpy.random.default_rng(21)
    data = rng.standard_normal(shape) + 1j * rng.standard_normal(shape)
    a = Array.from_host(queue, data)
    out = Array.empty_like(queue.device, a)
    fft = FFT(a, axes=(1,))
    fftc = fft.compile(queue.device)
    assert [p.L > 256 for p in fft.native_plan.passes].count(True) >= 1 and len(fft.native_plan.passes) == 2
    fftc(queue, out, a, inverse)
    want = (numpy.fft.ifft if inverse else numpy.fft.fft)(data, axis=1)
    got = out.get(queue)
    # rounding errors of log2(n) stages in 53 bits (the bound of the complex128 suite)
    assert numpy.linalg.norm(got - want) <= 5e-16 * numpy.log2(shape[1]) * numpy.linalg.norm(want)
