"""Transposes at the edges of the 64 x 64 tile, with all loads in flight and with a
branch per load (arrays that exceed the cache)."""

import numpy
import pytest

from reikna_amd import Array
from reikna_amd.algorithms import Transpose

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dtype", [numpy.int8, numpy.int32, numpy.complex64, numpy.complex128], ids=lambda d: d.__name__)
@pytest.mark.parametrize("shape", [(1, 1), (1, 129), (129, 1), (63, 65), (64, 64), (65, 63), (128, 130), (3, 67, 100),
                                   (4100, 4099)], ids=str)
def test_edges(queue, shape, dtype):
    n = int(numpy.prod(shape))
    data = (numpy.arange(n) % 113).astype(dtype).reshape(shape)
    axes = (*range(len(shape) - 2), len(shape) - 1, len(shape) - 2)
    a = Array.from_host(queue, data)
    tr = Transpose(a, axes=axes)
    out = Array.empty_like(queue.device, tr.parameter.output)
    tr.compile(queue.device)(queue, out, a)
    assert numpy.array_equal(out.get(queue), data.transpose(axes))
