"""Arguments of a compiled computation: positional, keyword and defaulted
calls give the same values to its steps, and every layout is checked."""

import numpy
import pytest

from reikna_amd import Annotation, ArrayMetadata, Parameter
from reikna_amd.core.computation import ComputationCallable
from reikna_amd.runtime import Array, VirtualDevice, _ForeignBuffer


class Recorder:
    argnames = ["output", "input", "inverse"]

    def __init__(self):
        self.seen = []

    def __call__(self, queue, values):
        self.seen.append((values["output"], values["input"], values["inverse"], type(values["inverse"])))


META = ArrayMetadata((4, 8), numpy.complex64)


def array(meta=META, size=None):
    return Array(VirtualDevice(), meta, _ForeignBuffer(VirtualDevice(), 0, meta.buffer_size if size is None else size, None))


def make():
    rec = Recorder()
    params = [Parameter("output", Annotation(META, "o")), Parameter("input", Annotation(META, "i")),
              Parameter("inverse", Annotation(numpy.int32), default=0)]
    return rec, ComputationCallable(VirtualDevice(), params, [rec], {}, [])


@pytest.mark.parametrize("inverse", [0, 1, True, numpy.int64(1)])
def test_positional_keyword_and_default(inverse):
    rec, call = make()
    a, b = array(), array()
    call(None, a, b, inverse)
    call(None, a, b, inverse=inverse)
    call(None, input=b, output=a, inverse=inverse)
    assert all(s == (a, b, int(inverse), numpy.int32) for s in rec.seen)
    call(None, a, b)
    assert rec.seen[-1] == (a, b, 0, numpy.int32)


@pytest.mark.parametrize("bad", [
    array(ArrayMetadata((8, 4), numpy.complex64)),
    array(ArrayMetadata((4, 8), numpy.complex128)),
    array(ArrayMetadata((4, 8), numpy.complex64, strides=(128, 16))),
    array(ArrayMetadata((4, 8), numpy.complex64, first_element_offset=8)),
    array(META, 255),
], ids=["shape", "dtype", "strides", "offset", "size"])
def test_wrong_layouts_are_refused(bad):
    _, call = make()
    for args, kwds in (((bad, array(), 0), {}), ((array(), bad, 0), {}), ((array(), bad), {"inverse": 1})):
        with pytest.raises(ValueError):
            call(None, *args, **kwds)


def test_wrong_calls_are_refused():
    _, call = make()
    for args, kwds in (((array(),), {}), ((array(), array(), 0, 0), {}), ((array(), array()), {"nothing": 1}),
                       ((array(), numpy.zeros((4, 8), numpy.complex64), 0), {})):
        with pytest.raises(TypeError):
            call(None, *args, **kwds)
