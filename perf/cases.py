"""Performance cases of the FFT library: transforms a program runs on device-resident buffers through `Plan.execute_tensors`.

A program makes a plan for its lengths once, keeps it with its buffers, and calls it for every new input; so `prepare` makes the inputs, the
plans and the output buffers, and `run` executes the plans. The five "kind"s:

  c2c    one complex transform (1-D to 3-D; forward, or inverse with normalization; f32, f64, or f16 storage with f32 compute)
  real   R2C and then C2R of its spectrum, normalized (filtering: 1-D signals, 2-D images, 3-D grids; f32, f64)
  r2r    a DCT or DST and its normalized inverse (spectral solvers, coding; types I to IV; f32, f64)
  conv   circular convolution with one kernel spectrum per plan (1-D, 2-D; f32, f64)
"""
import math
import os
import sys

import numpy as np
import torch

sys.path.insert(0, os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "vkfft-rs_amd"))
import vkfft_amd as vk  # noqa: E402

_context = None


def _ctx():
    global _context
    if _context is None:
        torch.cuda.init()  # torch's HIP runtime is the one the library binds to
        _context = vk.HipExecutionContext(0)
    return _context


def _case(name, kind, dims, batch, precision="f32", inverse=False, r2r=""):
    return {"name": name, "kind": kind, "dims": "x".join(str(d) for d in dims), "batch": batch, "precision": precision, "inverse": inverse, "r2r": r2r}


def listed():
    return [
        # one small field per call, as in an iterative solver or a control loop: launches and latency
        _case("c2c_64x64_f32_b1", "c2c", [64, 64], 1),
        # the benchmark's batched rows (radar, channelizers): one pass over memory
        _case("c2c_1024_f32_b8192", "c2c", [1024], 8192),
        # an odd length without powers of two, double precision, back from the spectrum
        _case("c2c_1001_f64_inverse_b8192", "c2c", [1001], 8192, "f64", True),
        # the benchmark's long real signals, there and back (fast convolution, spectral filters)
        _case("real_1048576_f32_b256", "real", [1 << 20], 256),
        # the benchmark's large images
        _case("c2c_4096x4096_f32_b16", "c2c", [4096, 4096], 16),
        # the benchmark's simulation volume in double precision
        _case("c2c_512x512x512_f64_b1", "c2c", [512, 512, 512], 1, "f64"),
        # the benchmark's prime lengths: a transform length given by the data
        _case("c2c_4099_f32_b4096", "c2c", [4099], 4096),
        _case("c2c_65537_f32_b4096", "c2c", [65537], 4096),
        # video frames or camera images, filtered in the frequency domain
        _case("real_1080x1920_f32_b16", "real", [1080, 1920], 16),
        # a cosine-basis solver or image coder on frames
        _case("dct2_720x1280_f32_b16", "r2r", [720, 1280], 16, r2r="dct2"),
        # images convolved with one point-spread function
        _case("conv_1024x1024_f32_b8", "conv", [1024, 1024], 8),
        # half-precision storage of large fields (memory-bound pipelines)
        _case("c2c_2048x2048_f16_b8", "c2c", [2048, 2048], 8, "f16"),
    ]


def _smooth(rng, low, high, primes):
    """A length in [low, high] with only these prime factors, near a draw that is uniform over the logarithm."""
    at = int(round(math.exp(rng.uniform(math.log(low), math.log(high)))))
    for step in range(high):
        for n in (at + step, at - step):
            if low <= n <= high:
                m = n
                for p in primes:
                    while m % p == 0:
                        m //= p
                if m == 1:
                    return n
    return low


def _length(rng, low, high):
    """Lengths as programs choose them: powers of two, round numbers, other factors the radices cover, and whatever the data has."""
    which = rng.random()
    if which < 0.2:
        return _smooth(rng, low, high, (2,))
    if which < 0.55:
        return _smooth(rng, low, high, (2, 3, 5))
    if which < 0.8:
        return _smooth(rng, low, high, (2, 3, 5, 7, 11, 13))
    return int(round(math.exp(rng.uniform(math.log(low), math.log(high)))))


def draw(rng):
    kind = rng.choice(["c2c", "c2c", "c2c", "real", "real", "r2r", "conv"])
    rank = rng.choice([1, 2] if kind == "conv" else [1, 1, 2, 2, 3] if kind != "r2r" else [1, 2])
    top = {"c2c": {1: 1 << 20, 2: 4096, 3: 400}, "real": {1: 1 << 20, 2: 4096, 3: 400}, "r2r": {1: 8192, 2: 2048}, "conv": {1: 1 << 18, 2: 2048}}[kind][rank]
    dims = [_length(rng, 16, top) for _ in range(rank)]
    if kind == "real" and rng.random() < 0.8:
        dims[-1] += dims[-1] % 2  # real axes are mostly even
    precision = rng.choice(["f32", "f32", "f32", "f64", "f16"] if kind == "c2c" else ["f32", "f32", "f64"])
    points = math.prod(dims)
    most = 1 << (23 if precision == "f64" else 24)
    total = math.exp(rng.uniform(math.log(1 << 12), math.log(most)))
    batch = max(1, min(1 << 16, int(total / points)))
    if points > 2 * most:
        dims, batch = dims[:1], 1
    inverse = kind == "c2c" and rng.random() < 0.4
    r2r = rng.choice(["dct2", "dct2", "dct2", "dct3", "dct4", "dct1", "dst2", "dst1"]) if kind == "r2r" else ""
    c = _case("", kind, dims, batch, precision, inverse, r2r)
    del c["name"]
    return c


def _dims(case):
    return [int(d) for d in case["dims"].split("x")]


def _spectrum_dims(case):
    d = _dims(case)
    return d[:-1] + [d[-1] // 2 + 1]


def _inputs(case, seed):
    """Samples in [-1, 1); a convolution's kernel is a normalized positive window of up to 15 samples per axis at the origin."""
    g = torch.Generator(device="cuda").manual_seed(seed)
    f = torch.float64 if case["precision"] == "f64" else torch.float32
    shape = [case["batch"]] + _dims(case) + ([2] if case["kind"] in ("c2c", "conv") else [])
    x = torch.rand(shape, generator=g, device="cuda", dtype=f).mul_(2).sub_(1)
    if case["precision"] == "f16":
        return x.half(), None
    if case["kind"] not in ("c2c", "conv"):
        return x, None
    x = torch.view_as_complex(x)
    if case["kind"] == "c2c":
        return x, None
    h = np.zeros(_dims(case))
    w = [min(15, d) for d in h.shape]
    h[tuple(slice(0, k) for k in w)] = np.random.default_rng(seed).uniform(0, 1, w)
    return x, np.fft.fftn(h / h.sum()).astype(np.complex128 if case["precision"] == "f64" else np.complex64)


_PRECISION = {"f32": vk.Precision.F32, "f64": vk.Precision.F64, "f16": vk.Precision.F16StorageF32Compute}


def _plan(case, transform, direction):
    c = vk.FftConfig.new(_dims(case)).with_batch_count(case["batch"]).with_precision(_PRECISION[case["precision"]]).with_transform(transform)
    c.with_inverse_normalization(direction == vk.Direction.Inverse)
    return vk.Plan(_ctx(), vk.TransformIr.build(c, direction))


def prepare(case, seed):
    x, spectrum = _inputs(case, seed)
    kinds, ways = vk.TransformKind, vk.Direction
    if case["kind"] == "c2c":
        plans = [_plan(case, kinds.ComplexToComplex, ways.Inverse if case["inverse"] else ways.Forward)]
        outs = [torch.empty_like(x)]
    elif case["kind"] == "real":
        plans = [_plan(case, kinds.RealToComplex, ways.Forward), _plan(case, kinds.ComplexToReal, ways.Inverse)]
        complex_type = torch.complex128 if case["precision"] == "f64" else torch.complex64
        outs = [torch.empty([case["batch"]] + _spectrum_dims(case), device="cuda", dtype=complex_type), torch.empty_like(x)]
    elif case["kind"] == "r2r":
        t = (kinds.dct if case["r2r"][:3] == "dct" else kinds.dst)(int(case["r2r"][3:]))
        plans = [_plan(case, t, ways.Forward), _plan(case, t, ways.Inverse)]
        outs = [torch.empty_like(x), torch.empty_like(x)]
    else:
        c = vk.FftConfig.new(_dims(case)).with_batch_count(case["batch"]).with_precision(_PRECISION[case["precision"]])
        ir = vk.ConvolutionIr.build(c, spectrum)
        plans = [vk.Plan(_ctx(), ir.ir, desc=ir.desc())]
        outs = [torch.empty_like(x)]
    return {"x": x, "plans": plans, "outs": outs}


def run(state):
    x = state["x"]
    for plan, y in zip(state["plans"], state["outs"]):
        plan.execute_tensors(x, y)
        x = y
    return state["outs"]


def work(case):
    """Each transform reads its input once and writes its output once; 5 N log2 N operations for a complex transform, half for a real one."""
    d, b = _dims(case), case["batch"]
    n = math.prod(d)
    size = {"f32": 4, "f64": 8, "f16": 2}[case["precision"]]
    ops = 5.0 * n * math.log2(n) * b
    if case["kind"] == "c2c":
        return {"bytes": 4 * size * n * b, "flops": ops}
    if case["kind"] == "real":
        return {"bytes": 2 * size * b * (n + 2 * math.prod(_spectrum_dims(case))), "flops": ops}
    if case["kind"] == "r2r":
        return {"bytes": 4 * size * n * b, "flops": ops}
    return {"bytes": 4 * size * n * b + 2 * size * n, "flops": 2 * ops + 6.0 * n * b}


def tolerance(case):
    """About four times the largest error against 64 bits that the family shows."""
    if case["precision"] == "f16":
        return {"rel": 1e-3}  # results rounded to binary16: 2.1e-4 seen
    return {"rel": 4e-6 if case["precision"] == "f32" else 4e-6 * 2.0 ** -29}  # up to 7e-7 and 1.5e-15 seen


def _r2r_matrix(kind, n):
    """FFTW's REDFT / RODFT sums as a matrix, angles reduced as whole numbers before they are rounded."""
    k, j = np.arange(n)[:, None], np.arange(n)[None, :]
    t = int(kind[3:])
    if kind[:3] == "dct":
        if t == 1:
            m = 2 * np.cos(np.pi * ((j * k) % (2 * (n - 1))) / (n - 1))
            m[:, 0] /= 2
            m[:, -1] /= 2
        elif t == 2:
            m = 2 * np.cos(np.pi * (((2 * j + 1) * k) % (4 * n)) / (2 * n))
        elif t == 3:
            m = 2 * np.cos(np.pi * (((2 * k + 1) * j) % (4 * n)) / (2 * n))
            m[:, 0] /= 2
        else:
            m = 2 * np.cos(np.pi * (((2 * j + 1) * (2 * k + 1)) % (8 * n)) / (4 * n))
    elif t == 1:
        m = 2 * np.sin(np.pi * (((j + 1) * (k + 1)) % (2 * (n + 1))) / (n + 1))
    else:
        m = 2 * np.sin(np.pi * (((2 * j + 1) * (k + 1)) % (4 * n)) / (2 * n))
    return torch.from_numpy(m).cuda()


def exact(case, seed):
    x, spectrum = _inputs(case, seed)
    axes = tuple(range(1, 1 + len(_dims(case))))
    if case["kind"] == "c2c":
        z = torch.view_as_complex(x.double()) if case["precision"] == "f16" else x.to(torch.complex128)
        z = torch.fft.ifftn(z, dim=axes) if case["inverse"] else torch.fft.fftn(z, dim=axes)
        return [torch.view_as_real(z) if case["precision"] == "f16" else z]
    if case["kind"] == "real":
        return [torch.fft.rfftn(x.double(), dim=axes), x.double()]
    if case["kind"] == "r2r":
        y = x.double()
        for axis in axes:
            y = torch.movedim(torch.movedim(y, axis, -1) @ _r2r_matrix(case["r2r"], y.shape[axis]).T, -1, axis)
        return [y.contiguous(), x.double()]
    k = torch.from_numpy(spectrum.astype(np.complex128)).cuda()
    return [torch.fft.ifftn(torch.fft.fftn(x.to(torch.complex128), dim=axes) * k, dim=axes)]
