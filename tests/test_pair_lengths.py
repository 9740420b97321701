"""Pair tiles of the lengths whose kernels the run-time compiler makes, and the plans that stay with single ones.

CPU: a dry run reports them as the plan runs them.  GPU: every such length against the FP64 oracle.
"""

import numpy
import pytest

import oracle
from reikna_amd import Array, ArrayMetadata, _lib
from reikna_amd.fft import FFT, NativeFftPlan

# every length from 512 to 1200 with a pair kernel that the catalogue lacks
LENGTHS = [540, 576, 600, 648, 675, 686, 720, 729, 810, 864, 900, 1008, 1080, 1125, 1152]


def columns(n):
    """A width at which columns of n points run as pairs: these three only in streaming passes."""
    return 32800 if n in (540, 675, 720) else 8208


def dry_run(shape, axes, flags=0):
    meta = ArrayMetadata(shape, numpy.complex64)
    return NativeFftPlan(meta, meta, axes, _lib.RK_FFT_DRY_RUN | flags)


def data_of(shape, seed):
    rng = numpy.random.default_rng(seed)
    return (rng.standard_normal(shape, numpy.float32) + 1j * rng.standard_normal(shape, numpy.float32)).astype(numpy.complex64)


@pytest.mark.parametrize("n", LENGTHS)
def test_dry_run_reports_pairs(n):
    assert [p.pair for p in dry_run((n, columns(n)), (0,)).passes] == [16]
    assert [p.pair for p in dry_run((n, columns(n) - 8), (0,)).passes] == [0]     # rows of no whole lines
    # without run-time compilation the catalogue's passes of this axis, if any, stay single
    try:
        assert not any(p.pair for p in dry_run((n, columns(n)), (0,), _lib.RK_FFT_NO_JIT).passes)
    except _lib.RkError as e:
        assert "run-time compilation is off" in str(e)


@pytest.mark.parametrize("shape,axes,want", [
    ((16, 1080, 1920), (1, 2), [0, 16]),
    ((32, 729, 800), (1,), [16]),
    ((120, 720 * 720), (1,), [16, 16]),
    ((67, 1000 * 1000), (1,), [0, 0]),      # tiles of 16 would cross the rows of a chunk
    ((60, 800 * 800), (1,), [0, 0]),        # many idle lanes
], ids=str)
def test_dry_run_plans(shape, axes, want):
    assert [p.pair for p in dry_run(shape, axes).passes] == want


def test_chunks_hold_whole_tiles_of_run_time_compiled_lengths():
    """A chunk's workspace is rebased, so no launched tile may reach past its chunk."""
    paired = 0
    for a in LENGTHS:
        for b in (*LENGTHS, 512, 768, 1000, 1024):
            for rows in (67, 127, 301):
                plan = dry_run((rows, a * b), (1,))
                for p in plan.passes:
                    paired += bool(p.pair)
                    if plan.chunk_rows:
                        assert (p.n_inst // rows) % (p.pair or p.C) == 0, (a, b, rows, p)
    assert paired


def check(queue, shape, axes, inverse, pairs):
    data = data_of(shape, shape[axes[0]])
    a = Array.from_host(queue, data)
    out = Array.empty_like(queue.device, a)
    fft = FFT(a, axes=axes)
    fftc = fft.compile(queue.device)
    assert any(p.pair for p in fft.native_plan.passes) == pairs
    assert bool(fft.native_plan.chunk_rows) == (len(shape) == 2 and axes == (1,))
    fftc(queue, out, a, inverse)
    got = out.get(queue)
    # instances spread over the array, the first, the last and their neighbours among them
    def spread(n):
        return numpy.unique(numpy.clip([0, 1, 15, 16, 17, n // 3, n // 2, n - 17, n - 16, n - 2, n - 1], 0, n - 1))
    for k in range(len(shape)):
        if k not in axes:
            data, got = data.take(spread(shape[k]), axis=k), got.take(spread(shape[k]), axis=k)
    ref = oracle.ifftn(data, axes) if inverse else oracle.fftn(data, axes)
    assert oracle.rel_l2(got, ref) <= oracle.tolerance(shape, axes)


@pytest.mark.gpu
@pytest.mark.parametrize("n", LENGTHS)
def test_lengths_match_oracle(queue, n):
    for inverse in (0, 1):
        check(queue, (n, columns(n)), (0,), inverse, True)


@pytest.mark.gpu
@pytest.mark.parametrize("shape,axes,pairs", [
    ((2, 1080, 4112), (1,), True),          # two outer indices of 257 tiles
    ((1024, 8206), (0,), True),             # a ragged last tile
    ((67, 720 * 720), (1,), True),          # a chain of run-time compiled pairs, a short last chunk
    ((60, 800 * 800), (1,), False),         # chunks of single tiles
], ids=str)
def test_shapes_match_oracle(queue, shape, axes, pairs):
    check(queue, shape, axes, 0, pairs)
