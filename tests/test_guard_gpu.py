"""A transform writes its output array and nothing else: every element around
it, and between its padded rows, keeps its value."""

import numpy
import pytest

import oracle
from reikna_amd import Array, ArrayMetadata
from reikna_amd.fft import BatchFFT, BatchItem, NativeFftPlan
from reikna_amd.runtime import Buffer

pytestmark = pytest.mark.gpu

GUARD = 1 << 16   # elements on either side: more than any ragged tile spans
MARK = numpy.complex64(7 - 3j)


def guarded(shape, pad=0):
    """Metadata of an array of rows `pad` elements apart inside the guards."""
    strides, step = [], 8
    for k in range(len(shape) - 1, -1, -1):
        strides.insert(0, step)
        step *= shape[k] + (pad if k == len(shape) - 1 else 0)
    span = sum((n - 1) * s for n, s in zip(shape, strides)) // 8 + 1
    return ArrayMetadata(shape, numpy.complex64, strides=strides, first_element_offset=8 * GUARD,
                         buffer_size=8 * (span + 2 * GUARD))


def marked(queue, meta):
    n = meta.buffer_size // 8
    flat = ArrayMetadata((n,), numpy.complex64)
    buf = Buffer(queue.device, meta.buffer_size)
    Array(queue.device, flat, buf).set(queue, numpy.full(n, MARK))
    return buf, flat


SHAPES = [((count, n), (1,)) for n in (2, 3, 4, 5, 6, 7, 8, 12, 15, 16, 20, 32, 48, 60, 64, 96, 100, 128, 160, 256, 320)
          for count in (1, 3, 301)]
SHAPES += [((5, n), (1,)) for n in (17, 97, 251, 509, 997, 1000, 1024, 1536, 2003, 2048, 4096, 5003, 8192, 12288, 65521, 65536)]
SHAPES += [((n, width), (0,)) for n in (2, 8, 17, 96, 100, 256, 509, 997, 1024, 1080, 5003) for width in (1, 7, 18, 33)]
SHAPES += [((3, 10, 12), (0, 1, 2)), ((17, 64, 9), (0, 1)), ((2, 100, 30), (1, 2))]


@pytest.mark.parametrize("pad", [0, 3])
def test_nothing_else_is_written(queue, pad):
    rng = numpy.random.default_rng(2)
    for shape, axes in SHAPES:
        if pad and shape[-1] == 1:
            continue
        meta = guarded(shape, pad)
        buf, flat = marked(queue, meta)
        data = (rng.standard_normal(shape) + 1j * rng.standard_normal(shape)).astype(numpy.complex64)
        src = Array.from_host(queue, data)
        plan = NativeFftPlan(src.metadata, meta, axes)
        ws = Buffer(queue.device, plan.workspace_bytes) if plan.workspace_bytes else None
        plan.execute(buf.ptr, src.ptr, 0, ws.ptr if ws else None, queue.stream)
        whole = Array(queue.device, flat, buf).get(queue)
        inner = numpy.lib.stride_tricks.as_strided(whole[GUARD:], shape, meta.strides)
        got = inner.copy()
        inner[...] = MARK
        assert (whole == MARK).all(), (shape, axes, numpy.nonzero(whole != MARK)[0][:4] - GUARD)
        assert oracle.rel_l2(got, oracle.fftn(data, axes)) <= oracle.tolerance(shape, axes), (shape, axes)


@pytest.mark.parametrize("lengths", [(2, 3, 7, 13, 16, 1), (8, 997), (64, 96, 5003, 5, 12), (32, 4096, 10)], ids=str)
def test_batch_items_write_their_own_range(queue, lengths):
    rng = numpy.random.default_rng(3)
    items, at = [], GUARD
    for n in lengths:
        items.append(BatchItem(n, 3, at, at, n + 1, n + 1))
        at += 3 * (n + 1)
    meta = ArrayMetadata((at + GUARD,), numpy.complex64)
    data = (rng.standard_normal(meta.shape) + 1j * rng.standard_normal(meta.shape)).astype(numpy.complex64)
    src = Array.from_host(queue, data)
    buf, flat = marked(queue, meta)
    out = Array(queue.device, flat, buf)
    BatchFFT(queue.device, items)(queue, out, src, 0)
    whole = out.get(queue)
    for it in items:
        for j in range(it.count):
            s = slice(it.out_offset + j * it.out_dist, it.out_offset + j * it.out_dist + it.length)
            want = oracle.fftn(data[s], (0,))
            assert oracle.rel_l2(whole[s], want) <= max(oracle.tolerance((it.length,)), 1e-12), it
            whole[s] = MARK
    assert (whole == MARK).all(), numpy.nonzero(whole != MARK)[0][:4] - GUARD
