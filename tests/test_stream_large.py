"""Plans over several axes of arrays larger than the Infinity Cache: every access of a pass streams, except in
column tiles of no whole cache lines."""

import numpy
import pytest

import oracle
from reikna_amd import Array, ArrayMetadata, _lib
from reikna_amd.fft import FFT, NativeFftPlan

NONE, LOAD, BOTH = (False, False), (True, False), (True, True)


@pytest.mark.parametrize("shape,axes,dtype,want", [
    ((8192, 8192), (0, 1), "complex64", [BOTH] * 4),
    ((512, 512, 512), (0, 1, 2), "complex64", [BOTH] * 3),
    ((256, 512, 512), (0, 1, 2), "complex128", [BOTH] * 3),
    ((4096, 8192), (0, 1), "complex64", [LOAD, NONE, NONE]),       # 256 MiB, the cache's size
    ((4096, 4096), (0, 1), "complex128", [LOAD, NONE]),
    ((6000, 6000), (0, 1), "complex64", [BOTH, NONE, BOTH, BOTH]),   # 75 adjacent values in the second pass
    ((512, 512, 504), (0, 1, 2), "complex64", [BOTH, NONE, BOTH]),   # axis 1: rows of 31 lines and a half
    ((3, 2**26), (1,), "complex64", [LOAD, NONE, (False, True)]),   # one axis: the caller's ends, in chunks
], ids=str)
def test_streaming_passes(shape, axes, dtype, want):
    meta = ArrayMetadata(shape, getattr(numpy, dtype))
    plan = NativeFftPlan(meta, meta, axes, _lib.RK_FFT_DRY_RUN)
    assert [(p.nt_load, p.nt_store) for p in plan.passes] == want


@pytest.mark.gpu
@pytest.mark.parametrize("shape", [(6000, 6000), (257, 512, 512)], ids=str)
def test_matches_oracle(queue, shape):
    """A plane wave per axis: one peak, the rest zero to rounding."""
    freq = tuple(n // 3 + k for k, n in enumerate(shape))
    data = numpy.ones(shape, numpy.complex64)
    for k, (n, f) in enumerate(zip(shape, freq)):
        wave = numpy.exp(2j * numpy.pi * f * numpy.arange(n) / n).astype(numpy.complex64)
        data *= wave.reshape([-1 if j == k else 1 for j in range(len(shape))])
    a = Array.from_host(queue, data)
    out = Array.empty_like(queue.device, a)
    fft = FFT(a)
    fftc = fft.compile(queue.device)
    assert any(p.nt_load and p.nt_store for p in fft.native_plan.passes)
    fftc(queue, out, a, 0)
    got = out.get(queue)
    want = numpy.zeros(shape, numpy.complex64)
    want[freq] = data.size
    # the waves themselves carry a rounding error of 32 bits per axis
    assert oracle.rel_l2(got, want) <= oracle.tolerance(shape, tuple(range(len(shape))))
