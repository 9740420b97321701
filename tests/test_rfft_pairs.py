"""The kernels that make the outputs k and N/2 - k in one thread: every N/2 up to
a few, odd and even, against numpy in double precision."""

import numpy
import pytest

import oracle
from reikna_amd import Array
from reikna_amd.fft.rfft import IRFFT, RFFT

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dtype", [numpy.float32, numpy.float64], ids=["f32", "f64"])
@pytest.mark.parametrize("n", [2, 4, 6, 8, 10, 14, 126, 128, 130, 1020, 1022, 1026, 8190])
def test_mirrored_pairs(queue, n, dtype):
    rng = numpy.random.default_rng(n)
    tol = oracle.tolerance((max(n, 4),)) * (1 if dtype == numpy.float32 else 5e-16 / 2e-7)
    ctype = numpy.complex64 if dtype == numpy.float32 else numpy.complex128
    a = rng.normal(size=(3, 2, n)).astype(dtype)
    a_dev = Array.from_host(queue, a)
    ref = numpy.fft.rfft(a.astype(numpy.float64), axis=-1)
    for last in (False, True):
        rf = RFFT(a_dev, dont_store_last=last)
        out = Array.empty_like(queue.device, rf.parameter.output)
        rf.compile(queue.device)(queue, out, a_dev)
        want = ref[..., : n // 2] if last else ref
        assert oracle.rel_l2(out.get(queue), want) <= tol
    fa = (rng.normal(size=(3, 2, n // 2 + 1)) + 1j * rng.normal(size=(3, 2, n // 2 + 1))).astype(ctype)
    fa_dev = Array.from_host(queue, fa)
    irf = IRFFT(fa_dev)
    out = Array.empty_like(queue.device, irf.parameter.output)
    irf.compile(queue.device)(queue, out, fa_dev)
    assert oracle.rel_l2(out.get(queue), numpy.fft.irfft(fa.astype(numpy.complex128), axis=-1)) <= tol
