"""Column tiles that compute two adjacent instances per thread (PairIO).

CPU: which passes run as pairs, over the layouts the planner accepts, and the
LDS form of the pair tile's FLAT store against the plain padded position.
GPU: the smallest and ragged sizes of every form against the FP64 oracle.
"""

import os
import shutil
import subprocess
import tempfile
from pathlib import Path

import numpy
import pytest

import oracle
from reikna_amd import Array, ArrayMetadata, _lib
from reikna_amd.fft import FFT, NativeFftPlan, PlanTuning

ROOT = Path(__file__).resolve().parents[1]
CSRC = ROOT / "reikna_amd" / "csrc"
HIPCC = os.environ.get("HIPCC", "/opt/rocm/bin/hipcc")


def pairs(shape, axes, strides=None, out_strides=None, tuning=None, dtype=numpy.complex64):
    meta = ArrayMetadata(shape, dtype, strides=strides)
    out = ArrayMetadata(shape, dtype, strides=out_strides)
    return [p.pair for p in NativeFftPlan(meta, out, axes, _lib.RK_FFT_DRY_RUN, tuning).passes]


PLANNED = [
    # streaming chains: the first pass's H and the last pass's NS are even
    ((64, 2**20), (1,), [16, 16]),
    ((256, 2**18), (1,), [16, 16]),
    ((512, 2**17), (1,), [16, 0]),      # 512 * 256: passes of 256 points never
    ((4, 2**20), (1,), [0, 0]),         # not streaming
    ((128, 1000 * 1000), (1,), [0, 0]),   # tiles would cross the rows of a chunk
    ((96, 1000 * 1024), (1,), [16, 16]),
    ((200, 800 * 800), (1,), [0, 0]),
    ((256, 640 * 640), (1,), [0, 0]),   # 20 values per thread
    ((1000, 8192), (0,), [16]),
    ((1000, 8194), (0,), [0]),
    ((1000, 4096), (0,), [0]),
    # a strided axis of 1024 points: at least 512 tiles of 16 and an even inner extent
    ((1024, 8192), (0,), [16]),
    ((1024, 8193), (0,), [0]),
    ((1024, 8000), (0,), [0]),
    ((8, 1024, 1024), (1,), [16]),
    ((8, 1024, 1023), (1,), [0]),
    ((512, 8192), (0,), [0]),
]


@pytest.mark.parametrize("shape,axes,want", PLANNED, ids=lambda v: str(v))
def test_passes_that_run_as_pairs(shape, axes, want):
    assert pairs(shape, axes) == want
    # complex128 passes and a forced column tile width never do
    assert not any(pairs(shape, axes, dtype=numpy.complex128))
    assert not any(pairs(shape, axes, tuning=PlanTuning(col_tile=16)))
    assert not any(pairs(shape, axes, tuning=PlanTuning(fixed_modes=0)))


def test_chunks_hold_whole_tiles():
    """A chunk's workspace is rebased, so no launched tile may reach past its chunk."""
    for n in (1000 * 1000, 1000 * 1024, 1000 * 768, 1000 * 512, 640 * 1000, 500 * 1000, 2**20, 2**17, 12288, 65521, 3 * 2**17):
        for rows in (67, 70, 127, 200, 2001, 9001):
            meta = ArrayMetadata((rows, n), numpy.complex64)
            plan = NativeFftPlan(meta, meta, (1,), _lib.RK_FFT_DRY_RUN)
            for p in plan.passes:
                if plan.chunk_rows:
                    assert (p.n_inst // rows) % (p.pair or p.C) == 0, (n, rows, p)


def test_pairs_need_unit_strides():
    n, m = 1024, 8192
    dense = (8 * m, 8)
    assert pairs((n, m), (0,), dense, dense) == [16]
    assert pairs((n, m), (0,), (16 * m, 16), dense) == [0]
    assert pairs((n, m), (0,), dense, (16 * m, 16)) == [0]
    assert pairs((n, m), (0,), (8 * m + 8, 8), (8 * m + 24, 8)) == [16]   # padded rows, odd row strides


PROGRAM = r"""
#include "fft_device.hpp"
#include <cstdio>
using namespace rkfft;
template <int L, int C> int check() {
    constexpr int T = Plan<L>::T, NT = (C / 2) * T, LP = lds_pitch_pair(L, C, T), R0 = Plan<L>::R0;
    int bad = 0;
    bool* seen = new bool[(C / 2) * L]();
    for (int tid = 0; tid < NT; ++tid)
        for (int i = 0; i < R0; ++i) {
            const int e = 2 * (tid + (i / 2) * NT) + i % 2, ce = e / L, p = e - ce * L;
            bad += flat_pair_lds<L, NT, LP>(tid, i / 2, i % 2) != ce * LP + lds_pad(p);
            bad += e >= (C / 2) * L || seen[e];
            if (e < (C / 2) * L) seen[e] = true;
        }
    for (int e = 0; e < (C / 2) * L; ++e) bad += !seen[e];
    bad += LP < lds_pad(L - 1) + 1 || pair_lds_bytes(L, C, T) != (C / 2) * LP * 8;
    if (bad) std::printf("L=%d C=%d: %d mismatches\n", L, C, bad);
    delete[] seen;
    return bad;
}
int main() {
    int bad = 0;
@CALLS@
    return bad != 0;
}
"""


@pytest.mark.skipif(not Path(HIPCC).exists(), reason="hipcc not available")
def test_flat_store_positions():
    calls = "\n".join(f"    bad += check<{n}, {c}>();" for n in (16, 48, 64, 80, 96, 256, 320, 512, 768, 1000, 1024)
                      for c in (16, 32, 48))
    tmp = Path(tempfile.mkdtemp(prefix="rk_pair_"))
    try:
        (tmp / "check.hip").write_text(PROGRAM.replace("@CALLS@", calls))
        build = subprocess.run(
            [HIPCC, "--offload-arch=gfx950", "--offload-host-only", "-O1", "-std=c++17", f"-I{CSRC}",
             f"-I{ROOT / 'include'}", str(tmp / "check.hip"), "-o", str(tmp / "check")],
            capture_output=True, text=True, timeout=300)
        assert build.returncode == 0, build.stderr[-4000:]
        run = subprocess.run([str(tmp / "check")], capture_output=True, text=True, timeout=60)
        assert run.returncode == 0, run.stdout[-4000:]
    finally:
        shutil.rmtree(tmp, ignore_errors=True)


def data_of(shape, seed):
    rng = numpy.random.default_rng(seed)
    return (rng.standard_normal(shape) + 1j * rng.standard_normal(shape)).astype(numpy.complex64)


@pytest.mark.gpu
@pytest.mark.parametrize("shape,axes,inverse", [
    ((1024, 8192), (0,), 0),            # the fewest tiles that run as pairs
    ((1024, 8194 + 14), (0,), 1),       # a ragged last tile
    ((3, 1024, 2734), (1,), 0),         # tiles across the outer index
    ((66, 2**19), (1,), 1),             # 1024 * 512, a short last chunk
    ((257, 2**17), (1,), 0),            # 512 * 256
    pytest.param((67, 1000 * 1000), (1,), 0, marks=pytest.mark.skip(
        reason="pair tiles that cross the rows of a chunk read outside its workspace: such tiles are no longer launched")),
    ((1000, 8208), (0,), 1),
    ((2, 1000, 4512), (1,), 0),
], ids=str)
def test_pair_tiles_match_oracle(queue, shape, axes, inverse):
    data = data_of(shape, 3)
    a = Array.from_host(queue, data)
    out = Array.empty_like(queue.device, a)
    fft = FFT(a, axes=axes)
    fftc = fft.compile(queue.device)
    assert any(p.pair for p in fft.native_plan.passes)
    fftc(queue, out, a, inverse)
    got = out.get(queue)
    # rows / columns spread over the array, the first and the last among them
    n = [k for k in range(len(shape)) if k not in axes]
    pick = tuple(slice(None) if k in axes else numpy.unique(numpy.linspace(0, shape[k] - 1, 24).astype(int))
                 for k in range(len(shape)))
    sub = data[pick] if len(n) == 1 else data[pick[0]][:, :, pick[2]]
    res = got[pick] if len(n) == 1 else got[pick[0]][:, :, pick[2]]
    ref = oracle.ifftn(sub, axes) if inverse else oracle.fftn(sub, axes)
    assert oracle.rel_l2(res, ref) <= oracle.tolerance(shape, axes)
    # in place: the same passes on the same buffer
    fftc(queue, a, a, inverse)
    assert numpy.array_equal(a.get(queue), got)


@pytest.mark.gpu
def test_pair_tiles_strided_view(queue):
    """Padded rows and an element offset that leaves the pairs at 8-byte addresses."""
    shape = (1024, 8192)
    data = data_of(shape, 5)
    a = Array.empty(queue.device, shape, numpy.complex64, strides=(8 * 8195, 8), first_element_offset=24)
    out = Array.empty(queue.device, shape, numpy.complex64, strides=(8 * 8193, 8), first_element_offset=8)
    a.set(queue, data)
    plan = NativeFftPlan(a.metadata, out.metadata, (0,))
    assert [p.pair for p in plan.passes] == [16]
    plan.execute(out.ptr, a.ptr, 0, None, queue.stream)
    got = out.get(queue)
    assert oracle.rel_l2(got, oracle.fftn(data, (0,))) <= oracle.tolerance(shape, (0,))
