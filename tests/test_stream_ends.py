"""Which accesses of a plan of several passes carry the nontemporal hint."""

import numpy
import pytest

import oracle
from reikna_amd import Array, ArrayMetadata, _lib
from reikna_amd.fft import FFT, NativeFftPlan


def ends(shape, axes, flags=0, dtype=numpy.complex64):
    meta = ArrayMetadata(shape, dtype)
    return [(p.nt_load, p.nt_store) for p in NativeFftPlan(meta, meta, axes, _lib.RK_FFT_DRY_RUN | flags).passes]


NONE, LOAD, STORE, BOTH = (False, False), (True, False), (False, True), (True, True)


@pytest.mark.parametrize("shape,axes,want", [
    ((5, 2**20), (1,), [NONE, NONE]),            # 40 MiB
    ((6, 2**20), (1,), [LOAD, STORE]),           # 48 MiB
    ((32, 2**20), (1,), [LOAD, STORE]),          # 256 MiB, one chunk
    ((1, 2**24), (1,), [LOAD, NONE, STORE]),
    ((128, 128, 128), (0, 1, 2), [NONE] * 3),
    ((256, 256, 256), (0, 1, 2), [LOAD, NONE, STORE]),
    ((16, 1080, 1920), (1, 2), [LOAD, NONE]),    # 253 MiB over two axes: its stores stay cached
    ((64, 1024, 1024), (1, 2), [LOAD, STORE]),   # chunked
    ((4096, 4096), (1,), [NONE]),                # one pass of 256 MiB in and out together
    ((8192, 4096), (1,), [BOTH]),
    ((16, 4096, 601), (1,), [NONE]),             # 32-byte column segments never stream
], ids=str)
def test_streaming_ends(shape, axes, want):
    assert ends(shape, axes) == want


def test_generated_ends_keep_streaming_throughout():
    assert ends((32, 2**20), (1,), _lib.RK_FFT_FUSED_ENDS) == [BOTH, BOTH]
    assert ends((8, 2**20), (1,), _lib.RK_FFT_FUSED_ENDS) == [LOAD, STORE]


@pytest.mark.gpu
@pytest.mark.parametrize("shape,axes,dtype", [
    ((6, 2**20), (1,), "complex64"),
    ((17, 3 * 2**17), (1,), "complex64"),
    ((257, 255, 256), (0, 1, 2), "complex64"),
    ((9, 1080, 1350), (1, 2), "complex64"),
    ((3, 2**20), (1,), "complex128"),
], ids=str)
def test_streaming_ends_match_oracle(queue, shape, axes, dtype):
    rng = numpy.random.default_rng(11)
    data = (rng.standard_normal(shape) + 1j * rng.standard_normal(shape)).astype(dtype)
    a = Array.from_host(queue, data)
    out = Array.empty_like(queue.device, a)
    fft = FFT(a, axes=axes)
    fftc = fft.compile(queue.device)
    assert any(p.nt_load or p.nt_store for p in fft.native_plan.passes)
    fftc(queue, out, a, 0)
    bound = oracle.tolerance(shape, axes) * (1 if dtype == "complex64" else 2.5e-9)
    assert oracle.rel_l2(out.get(queue), oracle.fftn(data, axes)) <= bound
