"""NativeFftPlan.execute takes any number as its direction."""

import numpy
import pytest

from reikna_amd import ArrayMetadata, _lib
from reikna_amd.fft import NativeFftPlan


@pytest.mark.parametrize("inverse", [0, True, 1.0, numpy.float32(1), numpy.int32(1), numpy.bool_(True)], ids=repr)
def test_directions(inverse):
    meta = ArrayMetadata((4, 16), numpy.complex64)
    plan = NativeFftPlan(meta, meta, (1,), _lib.RK_FFT_DRY_RUN)
    with pytest.raises(ValueError, match="dry-run"):   # reaches the library, which refuses a dry run's plan
        plan.execute(256, 256, inverse, None, None)
