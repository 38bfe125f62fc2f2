"""GPU tests of transforms whose arrays reach 4 GiB: 32-bit buffer offsets end
there, and the tiles take their general addressing (64-bit addresses, the format
looked up at each access).  Row kernels against the same batch in two parts
(below the limit) and against the oracle on rows around the limit; column kernels
against the outer product that the transform of an outer product is."""
import numpy as np
import pytest

from oracle import oracle as O
from test_gpu_rows import bound

pytestmark = pytest.mark.gpu

IL, SP = 1, 0
GIB4 = 1 << 30  # floats of 4 GiB


def _say(*a):
    print("[gpu-case]", *a, flush=True)


@pytest.fixture(autouse=True)
def _give_back():
    yield
    import torch
    torch.cuda.empty_cache()


def _sides(t, m, batch, fmt, real):
    """The argument pair of one side of `batch` transforms of m elements."""
    if real:
        return (t[:m * batch], None)
    if fmt == IL:
        return (t[:2 * m * batch], None)
    return (t[:m * batch], t[m * batch:2 * m * batch])


def _part(side, first, count, m, fmt, real):
    f = 2 * m if fmt == IL and not real else m
    return tuple(None if a is None else a[first * f:(first + count) * f] for a in side)


def _host(side, i, m, fmt, real):
    p = [None if a is None else a.cpu().numpy().astype(np.float64) for a in _part(side, i, 1, m, fmt, real)]
    if real:
        return p[0]
    return p[0][0::2] + 1j * p[0][1::2] if fmt == IL else p[0] + 1j * p[1]


# kind, points, format: rows of 64 (eight a group), 4096, the radix-32 and the
# half-LDS rows, r2c and c2r rows
ROWS = [("c", 64, SP), ("ci", 4096, SP), ("c", 16384, SP), ("ci", 32768, SP), ("c", 2048, IL), ("r", 16384, SP),
        ("ri", 16384, SP), ("ri", 32768, SP), ("r", 1024, IL)]


@pytest.mark.parametrize("kind,n,fmt", ROWS)
def test_rows(kind, n, fmt):
    import torch
    from fft_amd.afft import Plan
    m = n // 2 + 1
    real_in, real_out = kind == "r", kind == "ri"
    mi, mo = (m if kind == "ri" else n), (m if kind == "r" else n)
    # the array of the complex side reaches 4 GiB (interleaved: of points)
    batch = (GIB4 if fmt == SP else GIB4 // 2) // (m if kind in ("r", "ri") else n) + 3
    _say("large rows", kind, n, fmt, batch)
    g = torch.Generator(device="cuda").manual_seed(n)
    fi, fo = mi * batch * (1 if real_in else 2), mo * batch * (1 if real_out else 2)
    x = torch.rand(fi, generator=g, device="cuda").mul_(2).sub_(1)
    y, z = torch.full((fo,), 9.0, device="cuda"), torch.full((fo,), 8.0, device="cuda")
    src = _sides(x, mi, batch, fmt, real_in)
    if kind == "ri":  # bins 0 and n/2 are real
        im = (src[0].view(batch, m, 2)[..., 1] if fmt == IL else src[1].view(batch, m))
        im[:, 0] = 0
        im[:, n // 2] = 0
    dst, ref = _sides(y, mo, batch, fmt, real_out), _sides(z, mo, batch, fmt, real_out)
    p = Plan(kind, (n,), batch, format=fmt)
    assert len(p.describe()) == 1
    p(*src, *dst)
    torch.cuda.synchronize()
    p.close()
    half = batch // 2
    for first, count in ((0, half), (half, batch - half)):
        q = Plan(kind, (n,), count, format=fmt)
        q(*_part(src, first, count, mi, fmt, real_in), *_part(ref, first, count, mo, fmt, real_out))
        torch.cuda.synchronize()
        q.close()
    step = 1 << 27
    num = den = 0.0
    for i in range(0, fo, step):
        a, b = y[i:i + step].double(), z[i:i + step].double()
        num += float((a - b).pow(2).sum())
        den += float(b.pow(2).sum())
    assert (num / den) ** 0.5 <= 2 * bound(n, np.float32)
    for i in (0, 1, half, batch - 4, batch - 2, batch - 1):
        row = _host(src, i, mi, fmt, real_in)
        want = {"c": lambda: O.fft(row), "ci": lambda: O.fft(row, inverse=True), "r": lambda: O.rfft(row),
                "ri": lambda: O.irfft(row, (n,))}[kind]()
        got = _host(dst, i, mo, fmt, real_out)
        assert np.linalg.norm(got - want) <= bound(n, np.float32) * np.linalg.norm(want), (kind, n, i)


# kind, shape, format: one column pass (1024 points), its two-pass form (8192),
# the real column pass and the real pass between columns
COLUMNS = [("c", (1024, 1 << 20), SP), ("ci", (8192, 1 << 17), SP), ("r", (1024, 1 << 20), SP), ("r", (1024, 1 << 20), IL),
           ("r", (8192, 1 << 17), SP)]


@pytest.mark.parametrize("kind,shape,fmt", COLUMNS)
def test_columns(kind, shape, fmt):
    import torch
    from fft_amd.afft import Plan
    rows, cols = shape
    _say("large columns", kind, shape, fmt)
    rng = np.random.default_rng(rows)
    a, b = rng.uniform(-1, 1, rows), rng.uniform(-1, 1, cols)
    if kind != "r":
        a, b = a + 1j * rng.uniform(-1, 1, rows), b + 1j * rng.uniform(-1, 1, cols)
    h = rows // 2 + 1 if kind == "r" else rows
    fa = np.fft.rfft(a) if kind == "r" else np.fft.fft(a) if kind == "c" else np.fft.ifft(a) * rows
    fb = np.fft.fft(b) if kind != "ci" else np.fft.ifft(b) * cols
    da, db, dfa, dfb = (torch.from_numpy(v).cuda() for v in (a, b, fa, fb))
    x = torch.empty(rows * cols * (1 if kind == "r" else 2), device="cuda")
    y = torch.full((2 * h * cols,), 9.0, device="cuda")
    src, dst = _sides(x, rows * cols, 1, fmt, kind == "r"), _sides(y, h * cols, 1, fmt, False)
    for r in range(rows):
        v = da[r] * db
        if kind == "r":
            src[0][r * cols:(r + 1) * cols] = v
        elif fmt == IL:
            src[0][2 * r * cols:2 * (r + 1) * cols] = torch.view_as_real(v).reshape(-1)
        else:
            src[0][r * cols:(r + 1) * cols] = v.real
            src[1][r * cols:(r + 1) * cols] = v.imag
    p = Plan(kind, shape, 1, format=fmt)
    p(*src, *dst)
    torch.cuda.synchronize()
    p.close()
    num = den = 0.0
    for r in range(h):
        want = dfa[r] * dfb
        if fmt == IL:
            got = torch.view_as_complex(dst[0][2 * r * cols:2 * (r + 1) * cols].double().view(cols, 2))
        else:
            got = torch.complex(dst[0][r * cols:(r + 1) * cols].double(), dst[1][r * cols:(r + 1) * cols].double())
        num += float((got - want).abs().pow(2).sum())
        den += float(want.abs().pow(2).sum())
    # the input is rounded to FP32 as well: one more rounding
    n = rows * cols
    assert (num / den) ** 0.5 <= bound(n, np.float32) + 2.0 ** -24
