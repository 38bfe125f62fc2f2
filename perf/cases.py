"""Performance cases of the transform library, over the range it is used in.

Three kinds of program:
  call   one transform per call through the fft.h classes, as a program ported
         from the CPU library makes it (the call returns when the result is
         there): FP32 / FP64, split / interleaved, each of the four kinds,
         2^6 .. 2^22 points;
  batch  a batched plan, forward and then inverse (filtering, convolution,
         solvers): short rows, long signals, 2-D and 3-D grids, complex and
         real, FP32 and FP64, interleaved and split, any batch size;
  queue  thousands of 1-D FP32 transforms of uneven sizes in one launch.

Lengths are powers of two (the library takes no others); batch sizes and
aspect ratios are arbitrary.
"""
import math

import torch

from fft_amd import afft

_CLASSES = {"c": afft.complex_transform, "ci": afft.inverse_complex_transform,
            "r": afft.real_transform, "ri": afft.inverse_real_transform}


def _call(name, kind, lg, fmt, dtype="f32"):
    return {"name": name, "use": "call", "kind": kind, "dims": str(1 << lg), "batch": 1, "fmt": fmt, "dtype": dtype}


def _batch(name, kind, dims, batch, fmt="il", dtype="f32"):
    return {"name": name, "use": "batch", "kind": kind, "dims": "x".join(str(d) for d in dims), "batch": batch,
            "fmt": fmt, "dtype": dtype}


def listed():
    return [
        # one short transform per call: launch and wait dominate
        _call("call_4096", "c", 12, "split"),
        # one long real signal per call: a single transform has to fill the GPU
        _call("call_real_4m", "r", 22, "il"),
        # radar / channelizer rows, an odd batch
        _batch("rows_1024", "c", (1024,), 30011),
        # spectrogram frames of real samples, split output, an odd batch
        _batch("frames_2048", "r", (2048,), 20001, "split"),
        # the library's headline: 64 signals of 2^20 points
        _batch("signals_1m", "c", (1 << 20,), 64),
        # long real recordings
        _batch("real_4m", "r", (1 << 22,), 16),
        # very long signals, which need a third pass
        _batch("signals_16m", "c", (1 << 24,), 2),
        # double precision signals
        _batch("double_1m", "c", (1 << 20,), 16, "il", "f64"),
        # a periodic 3-D field of a solver
        _batch("field_256", "c", (256, 256, 256), 1),
        # one large real image
        _batch("image_8192", "r", (8192, 8192), 1),
        # a stack of small real images
        _batch("images_256", "r", (256, 256), 99),
        # requests of uneven sizes, 70 % complex, both directions
        {"name": "queue_10000", "use": "queue", "jobs": 10000, "lo": 6, "hi": 16, "mix": 5},
    ]


def _log_uniform(rng, lo, hi):
    return 2.0 ** rng.uniform(lo, hi)


def draw(rng):
    what = rng.choice(["call", "rows", "rows", "signals", "signals", "grid", "grid", "queue"])
    dtype = "f64" if rng.random() < 0.2 else "f32"
    fmt = "split" if rng.random() < 0.3 else "il"
    if what == "call":
        c = _call("", rng.choice(["c", "ci", "r", "ri"]), rng.randint(6, 22), fmt, dtype)
    elif what == "queue":
        lo = rng.randint(0, 10)
        c = {"use": "queue", "jobs": int(_log_uniform(rng, 6, 13.2)), "lo": lo, "hi": rng.randint(lo, 16),
             "mix": rng.randint(1, 1 << 20)}
    else:
        # elements of all transforms: no case costs more than signals_1m
        top = 24.5 if what == "grid" else 26.0
        if what == "rows":
            dims = [1 << rng.randint(2, 14)]
        elif what == "signals":
            dims = [1 << rng.randint(15, 24)]
            top = 25.0 if dims[0] > 1 << 22 else top
        else:
            dims = [1 << 30]
            while math.prod(dims) > 1 << 24:
                dims = [1 << rng.randint(3, 9) for _ in range(3)] if rng.random() < 0.5 else \
                    [1 << rng.randint(4, 13) for _ in range(2)]
        if dtype == "f64":
            top -= 1.5
        batch = max(1, int(_log_uniform(rng, 18.0, top) / math.prod(dims)))
        c = _batch("", rng.choice(["c", "r"]), dims, batch, fmt, dtype)
    c.pop("name", None)
    return c


def _shape(case):
    dims = [int(d) for d in case["dims"].split("x")]
    # the complex side of a real transform has its first axis halved
    half = [dims[0] // 2 + 1] + dims[1:]
    return dims, half


def _real_dtype(case):
    return torch.float64 if case["dtype"] == "f64" else torch.float32


def _signal(case, seed, dims, real):
    """Noise samples in [-1, 1), the transform's time-domain input."""
    g = torch.Generator(device="cuda").manual_seed(int(seed))
    shape = [case["batch"]] + dims + ([] if real else [2])
    x = torch.rand(shape, generator=g, device="cuda", dtype=_real_dtype(case)).mul_(2).sub_(1)
    return x if real else torch.view_as_complex(x)


def _spectrum(case, seed, dims):
    """The half spectrum of a 1-D real signal."""
    n = dims[0]
    g = torch.Generator(device="cuda").manual_seed(int(seed))
    z = torch.randn([case["batch"], n // 2 + 1, 2], generator=g, device="cuda", dtype=_real_dtype(case))
    z[:, 0, 1] = 0
    z[:, n // 2, 1] = 0
    return torch.view_as_complex(z)


def _parts(z, fmt):
    """The buffers the library reads for the complex tensor z."""
    if fmt == "il":
        return [torch.view_as_real(z).contiguous(), None]
    return [z.real.contiguous(), z.imag.contiguous()]


def _space(case, shape, real):
    """Output buffers: a real tensor, or the (re, im) pair of a complex one."""
    full = [case["batch"]] + shape
    make = lambda s: torch.empty(s, device="cuda", dtype=_real_dtype(case))  # noqa: E731
    if real:
        return [make(full)]
    return [make(full + [2]), None] if case["fmt"] == "il" else [make(full), make(full)]


def _input(case, seed):
    dims, _ = _shape(case)
    if case["kind"] == "ri":
        return _spectrum(case, seed, dims)
    return _signal(case, seed, dims, case["kind"] == "r")


_BINS = {0: lambda n: (2 * n, 2 * n), 1: lambda n: (2 * n, 2 * n),
         2: lambda n: (n, 2 * (n // 2 + 1)), 3: lambda n: (2 * (n // 2 + 1), n)}


def _requests(case):
    """(kind, log2 n, offset of the input, offset of the output) of every job,
    and the floats of the input and output buffers."""
    g = torch.Generator().manual_seed(case["mix"])
    u = torch.rand([case["jobs"], 3], generator=g, dtype=torch.float64).tolist()
    jobs, src, dst = [], 0, 0
    for a, b, c in u:
        lg = case["lo"] + min(int(a * (case["hi"] - case["lo"] + 1)), case["hi"] - case["lo"])
        kind = (2 if c < 0.5 else 3) if b < 0.3 and lg > 0 else (0 if c < 0.5 else 1)
        n_in, n_out = _BINS[kind](1 << lg)
        jobs.append((kind, lg, src, dst))
        src += (n_in + 63) // 64 * 64
        dst += (n_out + 63) // 64 * 64
    return jobs, src, dst


def _request_data(jobs, floats, seed):
    g = torch.Generator(device="cuda").manual_seed(int(seed))
    x = torch.rand(floats, generator=g, device="cuda").mul_(2).sub_(1)
    # bins 0 and n/2 of a real signal's spectrum are real
    ends = [o + 1 + k * (1 << lg) for kind, lg, o, _ in jobs if kind == 3 for k in (0, 1)]
    if ends:
        x[torch.tensor(ends, device="cuda")] = 0
    return x


def prepare(case, seed):
    if case["use"] == "queue":
        jobs, n_in, n_out = _requests(case)
        x = _request_data(jobs, n_in, seed)
        y = torch.zeros(n_out, device="cuda")
        a, b = x.data_ptr(), y.data_ptr()
        q = afft.Queue(case["jobs"], 16)
        q.prepare(afft.Queue.jobs([(kind, lg, a + 4 * i, b + 4 * o) for kind, lg, i, o in jobs]))
        return {"use": "queue", "queue": q, "x": x, "y": y}
    dims, half = _shape(case)
    fmt = afft.afft_interleaved if case["fmt"] == "il" else afft.afft_split
    dt = "float64" if case["dtype"] == "f64" else "float32"
    z, kind = _input(case, seed), case["kind"]
    src = [z] if kind == "r" else _parts(z, case["fmt"])
    del z
    if case["use"] == "call":
        dst = _space(case, half if kind == "r" else dims, kind == "ri")
        return {"use": "call", "plan": _CLASSES[kind](dims, dt, fmt), "args": src + dst, "out": dst}
    spec = _space(case, half if kind == "r" else dims, False)
    back = _space(case, dims, kind == "r")
    there = afft.Plan(kind, dims, case["batch"], dt, fmt)
    again = afft.Plan("ri" if kind == "r" else "ci", dims, case["batch"], dt, fmt)
    if kind == "r":
        # Plan takes (src, -, dst_re, dst_im) and (src_re, src_im, dst, -)
        return {"use": "batch", "there": there, "again": again, "a": [src[0], None] + spec,
                "b": spec + [back[0], None], "spec": spec, "back": back}
    return {"use": "batch", "there": there, "again": again, "a": src + spec, "b": spec + back, "spec": spec,
            "back": back}


def run(state):
    if state["use"] == "queue":
        state["queue"].launch()
        return state["y"]
    if state["use"] == "call":
        state["plan"](*state["args"])
        return state["out"]
    state["there"](*state["a"])
    state["again"](*state["b"])
    return {"spectrum": state["spec"], "back": state["back"]}


def _sides(case):
    """(bytes of the real or complex time side, bytes of the spectrum, real
    flops of one transform) of the whole batch."""
    dims, half = _shape(case)
    n, m = math.prod(dims), math.prod(half)
    size = 8 if case["dtype"] == "f64" else 4
    real = case["kind"] in ("r", "ri")
    flops = (2.5 if real else 5.0) * n * math.log2(n)
    return size * n * (1 if real else 2) * case["batch"], 2 * size * (m if real else n) * case["batch"], \
        flops * case["batch"]


def work(case):
    if case["use"] == "queue":
        jobs, _, _ = _requests(case)
        size = sum(sum(_BINS[kind](1 << lg)) for kind, lg, _, _ in jobs)
        return {"bytes": 4.0 * size, "flops": sum((5.0 if kind < 2 else 2.5) * (1 << lg) * lg for kind, lg, _, _ in jobs)}
    a, b, flops = _sides(case)
    if case["use"] == "call":
        return {"bytes": a + b, "flops": flops}
    return {"bytes": 2 * (a + b), "flops": 2 * flops}


def _as_parts(z, fmt):
    return [torch.view_as_real(z), None] if fmt == "il" else [z.real, z.imag]


def exact(case, seed):
    """The same outputs from torch.fft on the CPU in 64 bits."""
    if case["use"] == "queue":
        jobs, n_in, n_out = _requests(case)
        x = _request_data(jobs, n_in, seed).cpu().double()
        y = torch.zeros(n_out, dtype=torch.float64)
        for kind, lg, i, o in jobs:
            n = 1 << lg
            a, b = _BINS[kind](n)
            v = x[i:i + a]
            if kind != 2:
                v = torch.view_as_complex(v.view(-1, 2))
            if kind == 0:
                w = torch.fft.fft(v)
            elif kind == 1:
                w = torch.fft.ifft(v, norm="forward")
            elif kind == 2:
                w = torch.fft.rfft(v)
            else:
                w = torch.fft.irfft(v, n, norm="forward")
            y[o:o + b] = w if kind == 3 else torch.view_as_real(w).reshape(-1)
        return y
    dims, _ = _shape(case)
    kind = case["kind"]
    x = _input(case, seed).cpu()
    x = x.to(torch.complex128 if x.is_complex() else torch.float64)
    # the halved axis (the first) goes last, as torch wants it
    axes = list(range(2, len(dims) + 1)) + [1]
    if kind == "c":
        z = torch.fft.fftn(x, dim=axes)
        back = x
    elif kind == "ci":
        z = torch.fft.ifftn(x, dim=axes, norm="forward")
    elif kind == "r":
        z = torch.fft.rfftn(x, dim=axes)
        back = x
    else:
        return [torch.fft.irfft(x, dims[0], norm="forward")]
    if case["use"] == "call":
        return _as_parts(z, case["fmt"])
    # the inverse is unnormalised: it gives the input times the length
    back = back * math.prod(dims)
    return {"spectrum": _as_parts(z, case["fmt"]),
            "back": [back] if kind == "r" else _as_parts(back, case["fmt"])}
