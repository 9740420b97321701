"""Nontemporal hints of column passes by whether their rows of instances are whole cache lines."""

import numpy
import pytest

import oracle
from reikna_amd import Array, ArrayMetadata, _lib
from reikna_amd.fft import FFT, NativeFftPlan

NONE, LOAD, STORE, BOTH = (False, False), (True, False), (False, True), (True, True)


def hints(shape, axes, dtype="complex64", strides=None, out_strides=None):
    dt = getattr(numpy, dtype)
    plan = NativeFftPlan(ArrayMetadata(shape, dt, strides=strides), ArrayMetadata(shape, dt, strides=out_strides), axes,
                         _lib.RK_FFT_DRY_RUN)
    return [(p.nt_load, p.nt_store) for p in plan.passes]


@pytest.mark.parametrize("shape,axes,dtype,want", [
    ((32, 1000, 1000), (1,), "complex64", [NONE]),      # rows of 62 lines and a half
    ((32, 1000, 1008), (1,), "complex64", [BOTH]),
    ((100, 256, 2001), (1,), "complex64", [NONE]),
    ((100, 256, 2000), (1,), "complex64", [BOTH]),
    ((524, 64, 1000), (1,), "complex64", [BOTH]),       # tiles of 512 bytes: whole half lines do
    ((524, 64, 1001), (1,), "complex64", [NONE]),
    ((131, 256, 1000), (1,), "complex64", [NONE]),      # tiles of 128 bytes
    ((100, 250, 1003), (1,), "complex128", [NONE]),
    ((100, 250, 1004), (1,), "complex128", [BOTH]),
    ((100, 250, 1000), (1,), "complex128", [BOTH]),
    ((2048, 65536), (0,), "complex64", [BOTH]),         # 64-byte tiles of whole rows
    ((300, 1000, 1000), (1, 2), "complex64", [LOAD, NONE]),       # chunked, in place
    ((64, 2048, 2048), (1, 2), "complex64", [LOAD, STORE]),
    # a chain's ends together, by units of 64 bytes: 1000 * 8 and 900 * 8 bytes
    ((100, 1000 * 1000), (1,), "complex64", [LOAD, STORE]),
    ((40, 900 * 1000), (1,), "complex64", [NONE, NONE]),
    ((2000, 150 * 200), (1,), "complex64", [NONE, NONE]),
    ((64, 2**20), (1,), "complex64", [LOAD, STORE]),
    ((60, 500 * 500), (1,), "complex128", [LOAD, STORE]),
], ids=str)
def test_rows_of_whole_lines(shape, axes, dtype, want):
    assert hints(shape, axes, dtype) == want


def test_strided_rows():
    """Rows whose distance is no multiple of a line begin inside one; elements apart share every line."""
    shape = (1000, 65536)
    dense, padded = (8 * 65536, 8), (8 * 65544, 8)
    assert hints(shape, (0,), strides=dense, out_strides=dense) == [BOTH]
    assert hints(shape, (0,), strides=padded, out_strides=dense) == [STORE]
    assert hints(shape, (0,), strides=dense, out_strides=padded) == [LOAD]
    assert hints(shape, (0,), strides=(16 * 65536, 16), out_strides=dense) == [STORE]


@pytest.mark.gpu
@pytest.mark.parametrize("shape,axes", [((17, 256, 8001), (1,)), ((70, 512, 1002), (1,)), ((60, 750 * 900), (1,)),
                                        ((34, 1000, 1000), (1, 2))], ids=str)
def test_matches_oracle(queue, shape, axes):
    rng = numpy.random.default_rng(17)
    data = (rng.standard_normal(shape, numpy.float32) + 1j * rng.standard_normal(shape, numpy.float32)).astype(numpy.complex64)
    a = Array.from_host(queue, data)
    out = Array.empty_like(queue.device, a)
    FFT(a, axes=axes).compile(queue.device)(queue, out, a, 0)
    got = out.get(queue)
    pick = numpy.unique([0, 1, shape[0] // 2, shape[0] - 1])
    data, got = data[pick], got[pick]
    assert oracle.rel_l2(got, oracle.fftn(data, axes)) <= oracle.tolerance(shape, axes)
