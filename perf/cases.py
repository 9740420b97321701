"""The work that users of this framework run, one dict per case: transforms of
rows, long rows, images and volumes, of smooth, odd and prime lengths, in
complex64 and complex128, forward and inverse, real transforms, a spectrogram
and a batch of uneven lengths.

Every case goes through the public entry points (``reikna_amd.fft``): a
computation is planned and compiled once for the shape (``prepare``), and a
pass (``run``) is the calls a program makes on it.  Inputs are normally
distributed, made on the GPU from the seed alone; outputs are torch tensors
that the framework writes through ``Array.from_torch``.
"""

import functools
import math

import numpy
import torch

from reikna_amd import Array, ArrayMetadata, Device, Queue
from reikna_amd.fft import FFT, BatchFFT
from reikna_amd.fft.batch import packed_items, sample_lengths
from reikna_amd.fft.rfft import IRFFT, RFFT
from reikna_amd.fft.spectrogram import Spectrogram, hann_window

# Most elements of a drawn complex64 transform; half as many in complex128 and
# for prime lengths (each costs about twice the work).  The largest listed
# case has twice as many.
DRAWN_MAX = 2**25
DRAWN_MIN = 2**14


def _fft(name, shape, axes, dtype="complex64", direction="forward"):
    case = {"kind": "fft", "shape": ",".join(map(str, shape)), "axes": ",".join(map(str, axes)),
            "dtype": dtype, "direction": direction}
    return {"name": name, **case} if name else case


def listed():
    return [
        # a handful of short rows, there and back: the smallest calls, a user's inner loop
        _fft("rows_16x1024", (16, 1024), (1,), direction="both"),
        # many short rows of a length that is no power of two (FIR filtering, OFDM symbols)
        _fft("rows_4096x1000", (4096, 1000), (1,)),
        # rows of a prime length nobody chose for speed (recorded frames)
        _fft("rows_4096x997", (4096, 997), (1,)),
        # rows of middling length 3 * 2^12 (range lines, sweeps)
        _fft("rows_4096x12288", (4096, 12288), (1,)),
        # a few long rows of a prime length, back to the time domain
        _fft("rows_33x65521", (33, 65521), (1,), direction="inverse"),
        # a large batch of long rows: the headline transform
        _fft("rows_64x1048576", (64, 2**20), (1,)),
        # one volume, all three axes
        _fft("volume_256", (256, 256, 256), (0, 1, 2)),
        # a stack of HD images, both image axes, back from the frequency domain
        _fft("images_16x1080x1920", (16, 1080, 1920), (1, 2), direction="inverse"),
        # long rows in double precision
        _fft("rows_32x262144_c128", (32, 2**18), (1,), dtype="complex128"),
        # long real rows to their spectra and back
        {"name": "real_64x1048576", "kind": "real", "rows": 64, "length": 2**20},
        # a few minutes of a recording as a spectrogram
        {"name": "spectrogram_16777216", "kind": "spectrogram", "samples": 2**24, "frame": 256, "overlap": 128},
        # transforms of many different lengths in one launch (64 .. 65536; 2^k, 3 * 2^k, 5 * 2^k, primes)
        {"name": "batch_512", "kind": "batch", "count": 512, "lo": 64, "hi": 65536, "lengths_seed": 5},
    ]


# -- drawn cases -----------------------------------------------------------
def _log_uniform(rng, lo, hi):
    return math.exp(rng.uniform(math.log(lo), math.log(hi)))


def _smooth_near(rng, x):
    """A length 2^a 3^b 5^c 7^d near x, its odd part one of the common ones."""
    odd = rng.choice((1, 1, 1, 3, 5, 7, 9, 15, 21, 25, 27, 45, 75, 125))
    return max(2, odd * 2 ** max(0, round(math.log2(x / odd))))


def _prime_near(x):
    n = max(5, int(x)) | 1
    while any(n % f == 0 for f in range(3, math.isqrt(n) + 1, 2)):
        n += 2
    return n


def draw(rng):
    kind = rng.choice(("rows", "rows", "rows", "primes", "images", "volume", "real", "spectrogram", "batch"))
    double = kind in ("rows", "images") and rng.random() < 0.25
    dtype = "complex128" if double else "complex64"
    direction = rng.choice(("forward", "forward", "inverse", "both"))
    most = DRAWN_MAX // (2 if double or kind == "primes" or direction == "both" else 1)
    total = _log_uniform(rng, DRAWN_MIN, most / 2)
    if kind == "rows":
        n = _smooth_near(rng, _log_uniform(rng, 16, min(2**21, total)))
        return _fft("", (max(1, int(total / n)), n), (1,), dtype, direction)
    if kind == "primes":
        n = _prime_near(_log_uniform(rng, 17, min(2**17, total)))
        return _fft("", (max(1, int(total / n)), n), (1,), dtype, direction)
    if kind == "images":
        side = math.sqrt(min(total, 2**23))
        h = _smooth_near(rng, side * rng.uniform(0.3, 1.0) / 2)
        w = _smooth_near(rng, side * rng.uniform(0.3, 1.0))
        return _fft("", (max(1, int(total / (h * w))), h, w), (1, 2), dtype, direction)
    if kind == "volume":
        side = total ** (1 / 3)
        a, b, c = (_smooth_near(rng, side * rng.uniform(0.6, 1.2)) for _ in range(3))
        return _fft("", (a, b, c), (0, 1, 2), dtype, direction)
    if kind == "real":
        n = 2 * _smooth_near(rng, _log_uniform(rng, 64, min(2**20, total)) / 2)
        return {"kind": "real", "rows": max(1, int(total / n)), "length": n}
    if kind == "spectrogram":
        frame = 2 ** rng.randint(7, 11)
        return {"kind": "spectrogram", "samples": max(8 * frame, int(total / 2)), "frame": frame,
                "overlap": rng.choice((frame // 2, 3 * frame // 4, frame // 3))}
    return {"kind": "batch", "count": rng.randint(4, 512), "lo": 64, "hi": 65536, "lengths_seed": rng.randint(0, 10**6)}


# -- what a program has in hand ---------------------------------------------
@functools.cache
def _queue():
    """The program's one queue."""
    return Queue(Device(0))


def _ints(text):
    return tuple(int(x) for x in str(text).split(","))


def _random(shape, dtype, seed):
    gen = torch.Generator(device="cuda")
    gen.manual_seed(int(seed))
    return torch.randn(shape, dtype=dtype, device="cuda", generator=gen)


def _batch_lengths(case):
    return sample_lengths(case["count"], case["lo"], case["hi"], case["lengths_seed"])


def _input(case, seed):
    if case["kind"] == "fft":
        return _random(_ints(case["shape"]), getattr(torch, case["dtype"]), seed)
    if case["kind"] == "real":
        return _random((case["rows"], case["length"]), torch.float32, seed)
    if case["kind"] == "spectrogram":
        return _random((case["samples"],), torch.float32, seed)
    return _random((sum(_batch_lengths(case)),), torch.complex64, seed)


def prepare(case, seed):
    dev = Device(0)
    state = {"case": case, "queue": _queue(), "x": _input(case, seed)}
    state["xa"] = Array.from_torch(state["x"])

    def output(name, like):
        meta = like.annotation.array_metadata if hasattr(like, "annotation") else like
        state[name] = torch.empty(meta.shape, dtype=getattr(torch, meta.dtype.name), device="cuda")
        state[name + "a"] = Array.from_torch(state[name])

    if case["kind"] == "fft":
        state["fft"] = FFT(state["xa"], axes=_ints(case["axes"])).compile(dev)
        output("y", state["xa"].metadata)
        if case["direction"] == "both":
            output("z", state["xa"].metadata)
    elif case["kind"] == "real":
        shape = (case["rows"], case["length"] // 2 + 1)
        state["rfft"] = RFFT(state["xa"]).compile(dev)
        state["irfft"] = IRFFT(ArrayMetadata(shape, numpy.complex64)).compile(dev)
        output("y", ArrayMetadata(shape, numpy.complex64))
        output("z", state["xa"].metadata)
    elif case["kind"] == "spectrogram":
        spec = Spectrogram(state["xa"], case["frame"], case["overlap"])
        state["spectrogram"] = spec.compile(dev)
        step = case["frame"] - case["overlap"]
        frames = (case["samples"] - case["overlap"]) // step
        output("y", ArrayMetadata((case["frame"] // 2 + 1, frames), numpy.float32))
    else:
        state["batch"] = BatchFFT(dev, packed_items(_batch_lengths(case)))
        output("y", state["xa"].metadata)
    torch.cuda.synchronize()
    return state


# -- one pass -----------------------------------------------------------------
def run(state):
    case, queue = state["case"], state["queue"]
    if case["kind"] == "fft":
        if case["direction"] == "both":
            state["fft"](queue, state["ya"], state["xa"], 0)
            state["fft"](queue, state["za"], state["ya"], 1)
            return state["y"], state["z"]
        state["fft"](queue, state["ya"], state["xa"], int(case["direction"] == "inverse"))
        return state["y"]
    if case["kind"] == "real":
        state["rfft"](queue, state["ya"], state["xa"])
        state["irfft"](queue, state["za"], state["ya"])
        return state["y"], state["z"]
    if case["kind"] == "spectrogram":
        state["spectrogram"](queue, state["ya"], state["xa"])
        return state["y"]
    state["batch"](queue, state["ya"], state["xa"])
    return state["y"]


def work(case):
    """Each array of the caller's read or written once; 5 N log2 N operations per complex transform."""
    if case["kind"] == "fft":
        shape, axes = _ints(case["shape"]), _ints(case["axes"])
        size = math.prod(shape)
        calls = 2 if case["direction"] == "both" else 1
        flops = 5 * size * sum(math.log2(shape[a]) for a in axes)
        return {"bytes": calls * 2 * size * numpy.dtype(case["dtype"]).itemsize, "flops": calls * flops}
    if case["kind"] == "real":
        size, spectrum = case["rows"] * case["length"], case["rows"] * (case["length"] // 2 + 1)
        return {"bytes": 2 * (4 * size + 8 * spectrum), "flops": 2 * 2.5 * size * math.log2(case["length"])}
    if case["kind"] == "spectrogram":
        frames = (case["samples"] - case["overlap"]) // (case["frame"] - case["overlap"])
        return {"bytes": 4 * case["samples"] + 4 * frames * (case["frame"] // 2 + 1),
                "flops": 2.5 * frames * case["frame"] * math.log2(case["frame"])}
    lengths = _batch_lengths(case)
    return {"bytes": 16 * sum(lengths), "flops": sum(5 * n * math.log2(n) for n in lengths)}


# -- the same in 64 bits ------------------------------------------------------
def exact(case, seed):
    x = _input(case, seed).cpu()
    if case["kind"] == "fft":
        x, axes = x.to(torch.complex128), _ints(case["axes"])
        if case["direction"] == "both":
            return torch.fft.fftn(x, dim=axes), x
        return torch.fft.ifftn(x, dim=axes) if case["direction"] == "inverse" else torch.fft.fftn(x, dim=axes)
    if case["kind"] == "real":
        x = x.double()
        return torch.fft.rfft(x), x
    if case["kind"] == "spectrogram":
        frames = x.double().unfold(0, case["frame"], case["frame"] - case["overlap"])
        # the window as the framework holds it, in 32 bits
        window = torch.from_numpy(hann_window(case["frame"]).astype(numpy.float32)).double()
        return torch.fft.rfft(frames * window).abs().T.contiguous()
    lengths = _batch_lengths(case)
    return torch.cat([torch.fft.fft(p) for p in x.to(torch.complex128).split(lengths)])
